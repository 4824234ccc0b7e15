"""Which layers try the split of their fp32 synapse: a host rule."""

import pytest

from myelin_amd import _lib
from myelin_amd import linear as L

FP32 = _lib.PREC["fp32"]


# shapes that the fused kernel takes keep it where it is the faster: narrow
# inputs, whose products cost less than a pass over the currents
@pytest.mark.parametrize("F,dense,packed", [(64, False, False), (120, False, False), (128, False, True),
                                            (184, False, True), (192, True, True), (1024, True, True)])
def test_fused_shapes_by_their_inputs(monkeypatch, F, dense, packed):
    monkeypatch.setattr(L.torch.cuda, "is_current_stream_capturing", lambda: False)
    T, B, N = 1 << 17, 256, 4096
    assert L._fused(B, N)
    assert L._split_eligible(FP32, T, B, F, N) == dense
    assert L._split_eligible(FP32, T, B, F, N, packed=True) == packed
    assert not L._split_eligible(FP32, T, B, F, N, ints=False)


def test_other_shapes(monkeypatch):
    monkeypatch.setattr(L.torch.cuda, "is_current_stream_capturing", lambda: False)
    T, B, F, N = 2000, 32, 64, 1024
    assert not L._fused(B, N)
    for ints in (True, False):
        assert not L._split_eligible(FP32, 10, B, F, N, ints=ints)  # too little work
        assert not L._split_eligible(FP32, T, B, F + 4, N, ints=ints)
        assert not L._split_eligible(_lib.PREC["bf16"], T, B, F, N, ints=ints)
        assert L._split_eligible(FP32, 2 * T, B, F, N, ints=ints)
    monkeypatch.setattr(L.torch.cuda, "is_current_stream_capturing", lambda: True)
    assert not L._split_eligible(FP32, 2 * T, B, F, N)
