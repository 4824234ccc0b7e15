"""Exact synapse currents of spikes on the int8 MFMA (myelin_cast_spikes,
myelin_weight_digits, myelin_gemm_spikes) against float64, at the edges of
its tiles and stages and of the digits' range."""

from __future__ import annotations

import pytest
import torch

import myelin_amd as myelin
from myelin_amd import _lib
from myelin_amd import linear as L
from tests.helpers import seeded

DEV = "cuda"


def _print_case(**kw):
    print("case:", " ".join(f"{k}={v}" for k, v in kw.items()), flush=True)


def _operands(x, w):
    """(words, xb, digits, scale, flags) of x [M, F] and w [F, N] on the GPU."""

    (M, F), N = x.shape, w.shape[1]
    stages = -(-F // 128)
    kp = 128 * stages
    stream = _lib.stream(x.device)
    words = torch.full((stages, M, 4), 77, dtype=torch.int32, device=DEV)
    xb = torch.empty((M, F), dtype=torch.bfloat16, device=DEV)
    flags = torch.zeros(2, dtype=torch.int32, device=DEV)
    q = torch.full((-(-N // 32), 128, kp), 77, dtype=torch.int8, device=DEV)
    scale = torch.empty(N, device=DEV)
    _lib.call("myelin_cast_spikes", x.data_ptr(), words.data_ptr(), xb.data_ptr(), M, F, 4 * stages, flags.data_ptr(),
              stream)
    _lib.call("myelin_weight_digits", w.data_ptr(), q.data_ptr(), scale.data_ptr(), F, N, kp, flags.data_ptr(), stream)
    return words, xb, q, scale, flags


def _product(words, q, scale, bias, N):
    out = torch.full((words.shape[1], N), float("nan"), device=DEV)
    _lib.call("myelin_gemm_spikes", words.data_ptr(), words.stride(0) // 4, q.data_ptr(), scale.data_ptr(),
              _lib.ptr(bias), out.data_ptr(), words.shape[1], N, q.shape[2], N, _lib.stream(out.device))
    return out


# tiles of 128 rows x 32 neurons, and of 256 rows from 512 of them on (the
# last two); one stage of 128 inputs, remainders of each
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,F", [(1, 33, 1), (127, 64, 127), (128, 65, 128), (129, 96, 129), (300, 31, 1000),
                                   (20011, 300, 72), (65600, 40, 257)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_digit_products_match_float64(M, N, F, with_bias):
    _print_case(test="digits", M=M, N=N, F=F, with_bias=with_bias)
    g = seeded(M + N + F)
    x = (torch.rand(M, F, generator=g) < (0.1 if with_bias else 0.9)).float()
    # columns of very different size, small weights beside large ones (a
    # column of many more binades is turned away: test_gpu_digit_range)
    w = torch.randn(F, N, generator=g) * torch.exp2(torch.randint(-40, 40, (N,), generator=g).float())
    w = w * torch.exp2(-torch.randint(0, 4, (F, N), generator=g).float())
    w[:, N // 2] = 0.0
    bias = torch.randn(N, generator=g) if with_bias else None
    xd, wd, bd = x.to(DEV), w.to(DEV), None if bias is None else bias.to(DEV)
    words, xb, q, scale, flags = _operands(xd, wd)
    assert flags.tolist() == [0, 0]
    packed = myelin.pack_spikes(xd).data
    rows = words.permute(1, 0, 2).reshape(M, -1)
    assert torch.equal(xb.float(), xd) and torch.equal(rows[:, :packed.shape[1]], packed)
    assert not bool(rows[:, packed.shape[1]:].any())
    got = _product(words, q, scale, bd, N)
    ref = xd.double() @ wd.double()
    # weights: rounded to multiples of 2^(e - 30), 2^(e - 1) <= column max <
    # 2^e, so each within 2^(e - 31) <= 2^-30 column max; the sum is rounded
    # at most twice to fp32 (2^-24 each), then the bias sum
    colmax = wd.double().abs().max(0).values
    tol = ref.abs() * 2.0**-23 + xd.double().sum(1, keepdim=True) * colmax * 2.0**-30
    if bd is not None:
        ref = ref + bd.double()
        tol = tol + ref.abs() * 2.0**-24
    off = (got.double() - ref).abs()
    assert bool((off <= tol).all()), f"largest error {float((off / tol.clamp_min(1e-300)).max()):.2f} of the bound"
    # a row does not depend on the rows computed with it
    r0 = M // 3
    assert torch.equal(_product(words[:, r0:r0 + 130], q, scale, bd, N), got[r0:r0 + 130])


@pytest.mark.gpu
@pytest.mark.parametrize("case,expect", [("spikes", [0, 0]), ("two", [0, 1]), ("minus", [0, 1]), ("half", [0, 1]), ("real", [1, 1]),
                                         ("nan", [1, 1]), ("w_inf", [0, 1]), ("w_nan", [0, 1]), ("w_tiny", [0, 1])])
def test_flags_say_what_the_digits_cannot_hold(case, expect):
    _print_case(test="digit_flags", case=case)
    g = seeded(5)
    x = (torch.rand(70, 300, generator=g) < 0.1).float()
    w = torch.randn(300, 40, generator=g)
    x[69, 299] = {"two": 2.0, "minus": -1.0, "half": 0.5, "real": 0.3, "nan": float("nan")}.get(case, 1.0)
    if case == "w_tiny":
        w[:, 39] = 1e-35
    elif case.startswith("w_"):
        w[299, 39] = float(case[2:])
    assert _operands(x.to(DEV), w.to(DEV))[4].tolist() == expect


@pytest.mark.gpu
@pytest.mark.parametrize("value", ["spikes", "half", "real"])
def test_fused_shape_layer_takes_the_engine_its_input_allows(monkeypatch, value):
    """A layer wide enough for the fused kernel: spikes run on the digits,
    multiples of 1/2 on the bf16 planes, real values on the fp32 engine (bit
    for bit the layer without a split)."""

    _print_case(test="digit_layer", value=value)
    T, B, F, N = 9, 128, 72, 4096
    assert L._fused(B, N)
    g = seeded(6)
    x = (torch.rand(T, B, F, generator=g) < 0.3).float() * {"spikes": 1.0, "half": 0.5, "real": 0.3}[value]
    w = (torch.rand(F, N, generator=g) - 0.4) * 0.5
    b = torch.rand(N, generator=g) * 0.1
    gs = torch.randn(T, B, N, generator=g).to(DEV)
    p = myelin.LIFParams(tau_mem=9.0, threshold=0.7, reset=-0.2)
    res, routes, operands = [], [], L._Split.operands
    monkeypatch.setattr(L._Split, "operands", lambda split: routes.append(operands(split)) or routes[-1])
    monkeypatch.setattr(L, "_DIGITS_MIN_F_FUSED", 0)
    for macs in (0, 1 << 62):
        monkeypatch.setattr(L, "_SPLIT_MIN_MACS", macs)
        leaves = [t.to(DEV).requires_grad_() for t in (x, w, b)]
        _, s = myelin.linear_surrogate_lif_forward(*leaves, p, surrogate="atan", surrogate_slope=4.0, checkpoint_size=4)
        res.append([s.detach(), *torch.autograd.grad(s, leaves, gs)])
        if macs == 0:
            (_, wt, _), = routes
            assert isinstance(wt, L._Digits) == (value == "spikes") and (wt is None) == (value == "real")
    if value == "real":
        for a, c in zip(*res):
            assert torch.equal(a, c)
    else:
        assert float((res[0][0] != res[1][0]).float().mean()) <= 1e-4
        if torch.equal(res[0][0], res[1][0]):
            for a, c in zip(res[0][1:], res[1][1:]):
                assert float((a - c).abs().max() / c.abs().max()) <= 1e-5


def test_host_validation():
    with pytest.raises(ValueError, match="row pitch"):
        _lib.call("myelin_cast_spikes", 16, 16, None, 4, 200, 6, 16, None)
    with pytest.raises(ValueError, match="null pointer"):
        _lib.call("myelin_cast_spikes", 16, 16, None, 4, 200, 8, None, None)
    with pytest.raises(ValueError, match="aligned"):
        _lib.call("myelin_weight_digits", 16, 8, 16, 200, 4, 256, 16, None)
    with pytest.raises(ValueError, match="row pitch"):
        _lib.call("myelin_weight_digits", 16, 16, 16, 70000, 4, 70016, 16, None)
    with pytest.raises(ValueError, match="ldc"):
        _lib.call("myelin_gemm_spikes", 16, 4, 16, 16, None, 16, 4, 64, 128, 32, None)
    with pytest.raises(ValueError, match="row pitch"):
        _lib.call("myelin_gemm_spikes", 16, 4, 16, 16, None, 16, 4, 64, 64, 64, None)
    with pytest.raises(ValueError, match="x_rows"):
        _lib.call("myelin_gemm_spikes", 16, 3, 16, 16, None, 16, 4, 64, 128, 64, None)
