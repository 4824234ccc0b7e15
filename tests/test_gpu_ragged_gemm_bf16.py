"""bf16-precision GEMMs over fp32 operands of any width on 128 x 128 or 64 x 64
tiles, against float64 of the rounded operands."""

from __future__ import annotations

import pytest
import torch

from myelin_amd import _lib
from myelin_amd import linear as L
from tests.helpers import seeded

DEV = "cuda"


# few tiles (64 x 64), tiles past a round of the chip (128 x 128), last tiles
# of one to three and of more columns, short and long K
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(150, 150, 150), (640, 201, 333), (5120, 201, 333), (999, 999, 129), (1280, 513, 785),
                                   (300, 301, 2001), (4097, 333, 65)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_ragged_products_match_float64(M, N, K, ta, tb):
    print("case: ragged_gemm_bf16", M, N, K, ta, tb, flush=True)
    g = seeded(M + N + K)
    a, b = torch.randn(*((K, M) if ta else (M, K)), generator=g), torch.randn(*((N, K) if tb else (K, N)), generator=g)
    ar, br = (t.bfloat16().double().to(DEV) for t in (a.t() if ta else a, b.t() if tb else b))
    ref = ar.contiguous() @ br.contiguous()
    # products of bf16 values are exact in fp32; K sums of any order round once each
    tol = (ar.abs().contiguous() @ br.abs().contiguous()) * K * 2.0**-24
    for split in (False, True):
        out = torch.full((M, N), float("nan"), device=DEV)
        L._gemm(a.to(DEV), b.to(DEV), out, M, N, K, M if ta else K, K if tb else N, N, ta, tb, False,
                _lib.PREC["bf16"], _lib.stream(out.device), split=split)
        assert bool(((out.double() - ref).abs() <= tol).all()), (split, float((out.double() - ref).abs().max()))
        if not split and not ta:
            # rows do not depend on how many are computed, nor on the tiles
            few = torch.empty((70, N), device=DEV)
            L._gemm(a.to(DEV), b.to(DEV), few, 70, N, K, K, K if tb else N, N, ta, tb, False, _lib.PREC["bf16"],
                    _lib.stream(out.device), split=False)
            assert torch.equal(few, out[:70])
