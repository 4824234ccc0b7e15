"""Infinite inputs of an fp32 layer: infinity times a weight's zero plane is no
number, so they never run on the split products."""

from __future__ import annotations

import pytest
import torch

import myelin_amd as myelin
from myelin_amd import linear as L
from tests.helpers import seeded

pytestmark = pytest.mark.gpu
DEV = "cuda"


# the chunked and the fused shapes
@pytest.mark.parametrize("T,B,F,N", [(11, 5, 136, 72), (9, 128, 72, 4096)])
@pytest.mark.parametrize("value", [float("inf"), float("-inf")])
def test_currents_are_those_of_the_fp32_engine(monkeypatch, T, B, F, N, value):
    print("case: infinite_input", T, B, F, N, value, flush=True)
    g = seeded(T)
    x = (torch.rand(T, B, F, generator=g) < 0.2).float()
    x[3, 1, 5] = value
    w = ((torch.rand(F, N, generator=g) - 0.4) * 0.5).mul(256).round().div(256)  # exact in bf16: two planes are zero
    w[w == 0.0] = 1.0
    outs = []
    monkeypatch.setattr(L, "_DIGITS_MIN_F_FUSED", 0)
    for macs in (0, 1 << 62):
        monkeypatch.setattr(L, "_SPLIT_MIN_MACS", macs)
        st, s = myelin.linear_surrogate_lif_forward(x.to(DEV), w.to(DEV), None, myelin.LIFParams(reset=-0.2),
                                                    surrogate="atan", surrogate_slope=4.0)
        outs.append((st.membrane, s))
    assert not bool(torch.isnan(outs[1][0]).any())
    for a, c in zip(*outs):
        assert torch.equal(a, c)
