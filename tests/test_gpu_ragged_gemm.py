"""fp32 GEMMs of any width on the 128 x 128 tiles (rows and bases at any
4-byte address), against float64."""

from __future__ import annotations

import pytest
import torch

from myelin_amd import _lib
from myelin_amd import linear as L
from tests.helpers import seeded

DEV = "cuda"


def _operand(g, rows, cols, off):
    """(view [rows, cols], its values in float64) `off` floats into a buffer
    of NaN, as is what follows it: no output may see them."""

    buf = torch.full((off + rows * cols + 8,), float("nan"))
    view = buf[off:off + rows * cols].view(rows, cols)
    view.copy_(torch.randn(rows, cols, generator=g))
    ref = view.double()
    return buf.to(DEV)[off:off + rows * cols].view(rows, cols), ref


# one tile and its remainders of 4 to 127, of 1 to 3 (the 64 x 64 tiles where
# the operand is contiguous along them); partial stages of 32 k; outputs that
# fill the chip on either engine, with and without a K split
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(128, 128, 33), (133, 255, 64), (131, 129, 95), (130, 259, 1001),
                                   (2051, 963, 70), (5000, 1030, 33), (261, 389, 4099)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("off", [0, 3])
def test_ragged_products_match_float64(M, N, K, ta, tb, off):
    print("case: ragged_gemm", M, N, K, ta, tb, off, flush=True)
    g = seeded(M + N + K)
    a, ar = _operand(g, *((K, M) if ta else (M, K)), off)
    b, br = _operand(g, *((N, K) if tb else (K, N)), off)
    bias = torch.randn(N, generator=g)
    ar, br = ar.t() if ta else ar, br.t() if tb else br
    ref = (ar.to(DEV) @ br.to(DEV).contiguous() + bias.double().to(DEV))
    # each of the K products and the sums of any order round once: K + 1
    # times 2^-24 of the sum of magnitudes
    tol = (ar.abs().to(DEV) @ br.abs().to(DEV).contiguous() + bias.double().abs().to(DEV)) * (K + 1) * 2.0**-24
    for split in (False, True):
        out = torch.full((M, N), float("nan"), device=DEV)
        L._gemm(a, b, out, M, N, K, M if ta else K, K if tb else N, N, ta, tb, False, _lib.PREC["fp32"],
                _lib.stream(out.device), bias=bias.to(DEV), split=split)
        assert bool(((out.double() - ref).abs() <= tol).all()), (split, float((out.double() - ref).abs().max()))
        if not split:
            # rows do not depend on how many are computed, nor on the tiles
            r = min(M, 70)
            if not ta:
                few = torch.empty((r, N), device=DEV)
                L._gemm(a, b, few, r, N, K, K, K if tb else N, N, ta, tb, False, _lib.PREC["fp32"],
                        _lib.stream(out.device), bias=bias.to(DEV), split=False)
                assert torch.equal(few, out[:r])
