"""Layers over spikes on the int8 digits: several chunks, recomputed spans,
gradients with sums that are exact, and inputs that turn out not to be spikes."""

from __future__ import annotations

import pytest
import torch

import myelin_amd as myelin
from myelin_amd import _lib
from myelin_amd import linear as L
from tests.helpers import assert_norm_close, assert_same_bits, seeded

pytestmark = pytest.mark.gpu
DEV = "cuda"
P = myelin.LIFParams(tau_mem=9.0, threshold=0.7, reset=-0.2)


def _print_case(**kw):
    print("case:", " ".join(f"{k}={v}" for k, v in kw.items()), flush=True)


@pytest.fixture
def calls(monkeypatch):
    """The library's calls, by name; the split at any size."""

    names, real = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: names.append(name) or real(name, *a))
    monkeypatch.setattr(L, "_SPLIT_MIN_MACS", 0)
    monkeypatch.setattr(L, "_DIGITS_MIN_F_FUSED", 0)
    monkeypatch.setattr(L, "_DIGITS_MIN_MACS_DX", 0)
    return names


def _gemms(names):
    return sum(n.startswith("myelin_gemm_spikes") for n in names)


def _case(T, B, F, N, seed):
    g = seeded(seed)
    x = (torch.rand(T, B, F, generator=g) < 0.2).float()
    w = (2.0 * torch.rand(F, N, generator=g) - 0.9) * (6.0 / F) ** 0.5
    b = torch.rand(N, generator=g) * 0.1
    return x, w, b, torch.randn(T, B, N, generator=g)


def _run(x, w, b, gs, ck):
    leaves = [t.to(DEV).requires_grad_() for t in (x, w, b)]
    st, s = myelin.linear_surrogate_lif_forward(*leaves, P, surrogate="atan", surrogate_slope=4.0, checkpoint_size=ck)
    return [st.membrane.detach(), s.detach(), *torch.autograd.grad(s, leaves, gs.to(DEV))]


# budgets of four steps' currents: chunks of four steps, spans of one
# checkpoint chunk; one that is a multiple of neither; a fused shape
@pytest.mark.parametrize("T,B,F,N,ck", [(23, 5, 136, 72, 3), (23, 5, 136, 72, 4), (9, 128, 72, 4096, 2)])
def test_chunks_and_recomputed_spans(monkeypatch, calls, T, B, F, N, ck):
    _print_case(test="digit_chunks", T=T, B=B, F=F, N=N, ck=ck)
    case = _case(T, B, F, N, T + ck)
    whole = _run(*case, None)
    assert _gemms(calls) == 1
    del calls[:]
    monkeypatch.setattr(L, "_CURRENT_CHUNK_ELEMS", 4 * B * N)
    chunked = _run(*case, None)
    assert _gemms(calls) == -(-T // 4)
    for a, c, what in zip(whole, chunked, ("membrane", "spikes", "gx", "gw", "gb")):
        assert_same_bits(a, c, what)
    del calls[:]
    recomputed = _run(*case, ck)
    assert _gemms(calls) > -(-T // 4)  # the forward's and the backward's
    for i, what in enumerate(("membrane", "spikes")):
        assert_same_bits(whole[i], recomputed[i], what)
    # the adjoint is the same bits; its products sum in other groups (dX by
    # the K split of fewer rows, dW and db by span): the fp32 gradients' bar
    for i, what in ((2, "gx"), (3, "gw"), (4, "gb")):
        assert_norm_close(recomputed[i].cpu(), whole[i].cpu(), 1e-5, what)


@pytest.mark.parametrize("t0,t1", [(0, 16), (16, 48), (33, 64)])
def test_recompute_reproduces_the_forward_trace(calls, t0, t1):
    """A span's recompute from its checkpoint, on a slice of the words, is the
    forward's trace bit for bit."""

    _print_case(test="digit_recompute", t0=t0, t1=t1)
    T, B, F, N = 64, 6, 200, 136
    x, w, b, _ = (t.to(DEV) for t in _case(T, B, F, N, 3))
    stream = _lib.stream(x.device)
    xs, wt, _ = L._Split(x, w, stream).operands()
    assert isinstance(wt, L._Digits)
    args = (0.9, 0.7, -0.2, 4.0, _lib.RULE_THRESHOLD, _lib.PREC["fp32"], stream)
    pre, ckpt = torch.empty(T, B, N, device=DEV), torch.empty(T, B, N, device=DEV)
    L._lif_fwd(xs, w, b, None, 0, T, *args, pre=pre, ckpt=ckpt, wt=wt, exact=True)
    part = torch.empty(t1 - t0, B, N, device=DEV)
    L._lif_fwd(xs, w, b, ckpt[t0], t0, t1, *args, pre=part, wt=wt, exact=True, budget=5 * B * N)
    assert_same_bits(part, pre[t0:t1], "trace")


@pytest.mark.parametrize("T,B,F,N,ck", [(23, 5, 136, 72, None), (23, 5, 136, 72, 4), (9, 128, 72, 4096, 4)])
def test_gradients_where_the_sums_are_exact(monkeypatch, calls, T, B, F, N, ck):
    """Weights and biases of multiples of 2^-8 make every current exact on
    either engine: the same raster, so every gradient is compared."""

    _print_case(test="digit_exact_sums", T=T, B=B, F=F, N=N, ck=ck)
    x, w, b, gs = _case(T, B, F, N, 8)
    w, b = (t.mul(256).round().div(256) for t in (w, b))
    digits = _run(x, w, b, gs, ck)
    assert _gemms(calls)
    monkeypatch.setattr(L, "_SPLIT_MIN_MACS", 1 << 62)
    fp32 = _run(x, w, b, gs, ck)
    assert torch.equal(digits[1], fp32[1])
    for a, c, what in zip(digits, fp32, ("membrane", "spikes", "gx", "gw", "gb")):
        assert float((a - c).abs().max()) <= 1e-5 * float(c.abs().max()), what


# an input whose sample shows spikes, with one other value in a place that
# the sample leaves out; the second changes the engine after the first chunk's
# currents were computed as if it were spikes
@pytest.mark.parametrize("value", [0.3, 0.5, 2.0, float("inf")])
@pytest.mark.parametrize("shape", [(23, 5, 136, 72), (9, 128, 72, 4096)])
@pytest.mark.parametrize("ck", [None, 4])
def test_one_value_that_is_no_spike(monkeypatch, calls, value, shape, ck):
    _print_case(test="digit_one_value", value=value, shape=shape, ck=ck)
    T, B, F, N = shape
    x, w, b, gs = _case(T, B, F, N, 9)
    w, b = (t.mul(256).round().div(256) for t in (w, b))
    step = x.numel() // 64
    assert step > 65
    x.view(-1)[2 * step + 65] = value
    got = _run(x, w, b, gs, ck)
    monkeypatch.setattr(L, "_SPLIT_MIN_MACS", 1 << 62)
    want = _run(x, w, b, gs, ck)
    for a, c, what in zip(got, want, ("membrane", "spikes", "gx", "gw", "gb")):
        if value in (0.5, 2.0):  # the bf16 planes: exact currents, gradients in another order
            assert float((a - c).abs().max()) <= 1e-5 * float(c.abs().max()), what
        else:
            assert torch.equal(torch.nan_to_num(a, 7.0), torch.nan_to_num(c, 7.0)), what


@pytest.mark.parametrize("wants_dx,macs,digits", [(True, 1, True), (True, 1 << 62, False), (False, 1 << 62, True)])
def test_the_engine_of_a_layer_whose_input_wants_its_gradient(monkeypatch, calls, wants_dx, macs, digits):
    _print_case(test="digit_dx", wants_dx=wants_dx, macs=macs)
    monkeypatch.setattr(L, "_DIGITS_MIN_MACS_DX", macs)
    x, w, b, gs = _case(23, 5, 136, 72, 12)
    leaves = [x.to(DEV).requires_grad_(wants_dx), *(t.to(DEV).requires_grad_() for t in (w, b))]
    _, s = myelin.linear_surrogate_lif_forward(*leaves, P, surrogate="atan", checkpoint_size=4)
    assert (_gemms(calls) > 0) == digits and ("myelin_gemm_parts" in calls) == (not digits)
    s.backward(gs.to(DEV))
    assert all((t.grad is not None) == t.requires_grad for t in leaves)


@pytest.mark.parametrize("kind", ["spikes", "real", "late", "empty"])
def test_packed_inference(monkeypatch, calls, kind):
    _print_case(test="digit_packed", kind=kind)
    T, B, F, N = 23, 5, 136, 72
    x, w, b, _ = _case(T, B, F, N, 10)
    w, b = (t.mul(256).round().div(256) for t in (w, b))
    if kind == "real":
        x = torch.randn(T, B, F, generator=seeded(2)).mul(64).round().div(64) * 1.25
    elif kind == "late":
        x[T - 1, B - 1, F - 2] = 0.5
    elif kind == "empty":
        x.zero_()
    monkeypatch.setattr(L, "_CURRENT_CHUNK_ELEMS", 4 * B * N)
    layer = myelin.LinearSurrogateLIFPacked(F, N, P).to(DEV)
    with torch.no_grad():
        layer.synapse.weight.copy_(w)
        layer.synapse.bias.copy_(b)
        got = layer(x.to(DEV))
        if kind == "spikes":
            assert _gemms(calls) == -(-T // 4)
        monkeypatch.setattr(L, "_SPLIT_MIN_MACS", 1 << 62)
        want = layer(x.to(DEV))
    assert torch.equal(got.data, want.data)
