"""The int8 digits of an fp32 weight hold 31 bits of each column's largest:
where they would lose what an fp32 product keeps, the layer takes another
engine, whichever inputs spike; and the digits' sums are joined without loss."""

from __future__ import annotations

import pytest
import torch

from myelin_amd import _lib
from myelin_amd import linear as L
from tests.helpers import seeded

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _print_case(**kw):
    print("case:", " ".join(f"{k}={v}" for k, v in kw.items()), flush=True)


def _kaiming(g, F, N):
    return (2.0 * torch.rand(F, N, generator=g) - 1.0) * (6.0 / F) ** 0.5


def _operands(x, w):
    stream = _lib.stream(torch.device(DEV, 0))
    return L._Split(x.to(DEV), w.to(DEV), stream).operands()


def _digits_flag(w):
    """flags[1] as the digits of ``w`` leave it."""

    F, N = w.shape
    kp = -(-F // 128) * 128
    wd = w.to(DEV).contiguous()
    flags = torch.zeros(2, dtype=torch.int32, device=DEV)
    q = torch.empty((-(-N // 32), 128, kp), dtype=torch.int8, device=DEV)
    scale = torch.empty(N, device=DEV)
    _lib.call("myelin_weight_digits", wd.data_ptr(), q.data_ptr(), scale.data_ptr(), F, N, kp, flags.data_ptr(),
              _lib.stream(wd.device))
    return int(flags[1])


# one weight of each column `ratio` times the layer's bound, on an input that
# never spikes: it must cost the others nothing.  (Without the range check the
# currents were 1.0e-4 of their 2-norm off at 1e4, 6e-3 at 1e6, 0.9 at 1e8.)
@pytest.mark.parametrize("ratio", [1.0, 4.0, 1e2, 1e4, 1e6, 1e8, 1e10])
def test_a_large_weight_on_a_silent_input(ratio):
    _print_case(test="digit_outlier", ratio=ratio)
    g = seeded(11)
    T, B, F, N = 4, 32, 1024, 64
    x = (torch.rand(T, B, F, generator=g) < 0.1).float()
    x[..., 0] = 0.0
    w = _kaiming(g, F, N)
    w[0] = ratio * (6.0 / F) ** 0.5
    xs, wt, _ = _operands(x, w)
    assert isinstance(wt, L._Digits) == (ratio < 100)
    pre = torch.empty(T, B, N, device=DEV)  # decay 0: the currents
    L._lif_fwd(xs, w.to(DEV), None, None, 0, T, 0.0, float("inf"), 0.0, 1.0, _lib.RULE_THRESHOLD, _lib.PREC["fp32"],
               _lib.stream(pre.device), pre=pre, wt=wt)
    ref = (x.double().reshape(-1, F) @ w.double()).reshape(T, B, N)
    # an fp32 sum of n terms rounds n times; sqrt(F) times 2^-24 of the sum of
    # the magnitudes that spike is four standard deviations and more of that
    tol = (x.double().reshape(-1, F) @ w.double().abs()).reshape(T, B, N) * F**0.5 * 2.0**-24
    off = (pre.cpu().double() - ref).abs()
    assert bool((off <= tol).all()), f"{float((off / tol).max()):.2f} of the bound"
    assert float((pre.cpu().double() - ref).norm() / ref.norm()) <= 4e-7


# the digits take what layers are made of, and weights they hold exactly
# whatever the range; they turn away a column with a group of inputs (one
# chunk of 128 here) far smaller than the rest, and one small weight too many
@pytest.mark.parametrize("F,N", [(128, 33), (784, 256), (1000, 40), (4096, 64)])
@pytest.mark.parametrize("kind,flag", [("uniform", 0), ("normal", 0), ("laplace", 0), ("pruned", 0), ("dyadic", 0),
                                       ("group", 1), ("one_column", 1)])
def test_which_weights_take_the_digits(F, N, kind, flag):
    _print_case(test="digit_weights", F=F, N=N, kind=kind)
    g = seeded(F + N)
    w = torch.randn(F, N, generator=g)
    if kind == "uniform":
        w = _kaiming(g, F, N)
    elif kind == "laplace":
        w = torch.empty(F, N).exponential_(generator=g) * torch.where(torch.rand(F, N, generator=g) < 0.5, -1.0, 1.0)
    elif kind == "pruned":
        w = w * (torch.rand(F, N, generator=g) < 0.1)
    elif kind == "dyadic":  # 2^-30 of the column's largest and up: held exactly
        w = torch.exp2(-torch.randint(0, 29, (F, N), generator=g).float())
        w[0] = 1.0
    elif kind == "group":
        w[:128] *= 2.0**-12
        w[127] = 8.0
    elif kind == "one_column":
        w[:, N - 1] *= 2.0**-12
        w[F - 1, N - 1] = 8.0
    assert _digits_flag(w) == flag


def test_share_of_small_weights():
    """The lines themselves: of 512 weights in one chunk a quarter and six may
    be rounded, a 16th and six below 2^-10, a 256th and six below 2^-14 of the
    power of two above the column's largest."""

    for share, value in ((4, 2.0**-8), (16, 2.0**-11), (256, 2.0**-15)):
        for extra, flag in ((0, 0), (1, 1)):
            w = torch.full((512, 20000), 0.75)  # 625 groups of 32: one chunk of 512 each
            n = 512 // share + 6 + extra
            w[:n, 19999] = value * 0.7  # 0.75 < 1 = 2^e; 0.7 has 24 bits: rounded
            assert _digits_flag(w) == flag, (share, extra)


@pytest.mark.parametrize("K", [2003, 65024])
def test_large_sums_that_cancel(K):
    """Half of the inputs add 32767 units, which lies in the two low digits,
    the others take 65536 units off in the two high ones: the low sum alone
    passes 2^24, the whole stays below it and is returned exactly."""

    _print_case(test="digit_cancel", K=K)
    n = K // 3
    w = torch.zeros(K, 32)
    unit = 2.0**-30
    w[:2 * n] = 32767 * unit
    w[2 * n:3 * n] = -65536 * unit
    w[K - 1] = 0.75  # the column's largest: sets the unit; silent
    x = torch.ones(1, 4, K)
    x[..., K - 1] = 0.0
    x[0, 1, 0] = x[0, 2, 2 * n] = x[0, 3, 1] = x[0, 3, 2 * n + 1] = 0.0
    xs, wt, _ = _operands(x, w)
    assert isinstance(wt, L._Digits)
    pre = torch.empty(1, 4, 32, device=DEV)
    L._lif_fwd(xs, w.to(DEV), None, None, 0, 1, 0.0, float("inf"), 0.0, 1.0, _lib.RULE_THRESHOLD, _lib.PREC["fp32"],
               _lib.stream(pre.device), pre=pre, wt=wt)
    ref = (x.double().reshape(4, K) @ w.double()).reshape(1, 4, 32)
    assert bool((ref.abs() < 2.0**24 * unit).all())
    assert torch.equal(pre.cpu().double(), ref)
