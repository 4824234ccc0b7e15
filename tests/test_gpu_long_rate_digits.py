"""The long-horizon rate network as modules at checkpoint_size=45, whose hidden
currents run on the int8 digits: its gradients against the float64 truth of
its own raster, at the bars of test_gpu_long_rate (whose modules run under the
memory policy, on the bf16 planes).  Not against the oracle's own: an fp32
evaluation of this network lies up to 1.6e-5 from the truth, so two that are
equally near it, as the digits and the planes are, may lie 3e-5 apart (2.8e-5
measured at the modules' init, where the digits are the nearer: gx 1.3e-5, the
oracle and the planes 1.5e-5)."""

from __future__ import annotations

import pytest
import torch

import myelin_amd as myelin
from myelin_amd import linear as L
from tests import test_gpu_long_rate as R
from tests.helpers import norm_rel_err

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _step(x, labels, wh, bh, wo, bo):
    leaves = [t.to(DEV).requires_grad_() for t in (x, wh, bh, wo, bo)]
    _, hidden = myelin.linear_surrogate_lif_forward(*leaves[:3], R.P, surrogate="superspike", surrogate_slope=10.0,
                                                    checkpoint_size=45)
    _, rates = myelin.linear_surrogate_lif_rate_forward(hidden, *leaves[3:], R.P, surrogate="superspike",
                                                        surrogate_slope=10.0, checkpoint_size=45, reduction="none")
    loss = torch.nn.functional.cross_entropy(rates * R.T, labels.to(DEV), reduction="sum") / R.B
    grads = torch.autograd.grad(loss, leaves)
    return hidden.detach(), rates.detach(), dict(zip(("gx", "gwh", "gbh", "gwo", "gbo"), grads))


def _check(init, got, hidden, rates, ref, truth, what):
    same = R._check_raster(hidden, ref, truth)
    x, labels, wh, bh, wo, bo = R._case(init)
    mine = truth if same else R._truth(x, labels, wh, bh, wo, bo, hidden, rates)
    for k, g in got.items():
        e, bar = norm_rel_err(g, mine[k]), max(1e-5, 1.1 * ref["to_truth"][k])
        print(f"{what} {k}: HIP to truth {e:.2e}, oracle to truth {ref['to_truth'][k]:.2e} (bar {bar:.2e})", flush=True)
        assert e <= bar, k


@pytest.mark.parametrize("init", ["default", "kaiming"])
def test_gradients_against_the_truth(monkeypatch, init):
    routes, operands = [], L._Split.operands
    monkeypatch.setattr(L._Split, "operands", lambda split: routes.append(operands(split)) or routes[-1])
    ref, truth = R._oracle_rows(init)
    x, labels, wh, bh, wo, bo = R._case(init)
    print(f"case: long_rate_digits full batch, init={init}", flush=True)
    hidden, rates, full = _step(x, labels, wh, bh, wo, bo)
    assert [isinstance(wt, L._Digits) for _, wt, _ in routes] == [True]
    _check(init, {"gx": full["gx"][:, :R.ROWS].cpu()}, hidden[:, :R.ROWS].cpu(), rates[:R.ROWS].cpu(), ref, truth,
           "full batch rows")
    print(f"case: long_rate_digits {R.ROWS} rows, init={init}", flush=True)
    part_hidden, part_rates, part = _step(x[:, :R.ROWS].contiguous(), labels[:R.ROWS], wh, bh, wo, bo)
    assert torch.equal(part_hidden, hidden[:, :R.ROWS])  # a current does not depend on the rows computed with it
    _check(init, {k: v.cpu() for k, v in part.items()}, part_hidden.cpu(), part_rates.cpu(), ref, truth,
           f"{R.ROWS} rows")
