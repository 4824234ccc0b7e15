"""State carried in place (m_final is m0) through the recurrences whose lanes
own packed words: workgroups hold eight words, so a raster whose word count
is no multiple of eight has half-waves past its last row, which must not read
state that the rows' own lanes, in other workgroups, have replaced."""

from __future__ import annotations

import pytest
import torch

from myelin_amd import _lib
from tests.helpers import assert_same_bits, seeded

pytestmark = pytest.mark.gpu
DEV = "cuda"

# words in all: 1, 9 (a second workgroup with seven half-waves too many), an
# odd and an even count over many rows
SHAPES = [(1, 5), (3, 70), (63, 1000), (1, 2850), (301, 2050)]


def _case(B, N, T, seed):
    print("case: in_place_state", B, N, T, flush=True)
    g = seeded(seed)
    x = 0.25 + 0.6 * torch.randn(T, B, N, generator=g)
    return x.to(DEV), (0.9 * torch.rand(B, N, generator=g)).to(DEV)


@pytest.mark.parametrize("B,N", SHAPES)
@pytest.mark.parametrize("T", [1, 17])
def test_packed_forward(B, N, T):
    x, m0 = _case(B, N, T, B + N)
    outs = []
    for in_place in (False, True):
        m = m0.clone()
        m_final = m if in_place else torch.empty_like(m0)
        words = torch.empty((T, B, -(-N // 32)), dtype=torch.int32, device=DEV)
        ckpt = torch.empty((-(-T // 16), B, N), device=DEV)
        _lib.call("myelin_lif_fwd_f32", x.data_ptr(), m.data_ptr(), m_final.data_ptr(), None, words.data_ptr(),
                  ckpt.data_ptr(), T, B, N, 0.9, 1.0, -0.1, 10.0, _lib.RULE_THRESHOLD, 16, _lib.stream(x.device))
        outs.append((words, m_final, ckpt))
    assert torch.equal(outs[0][0], outs[1][0])
    assert_same_bits(outs[0][1], outs[1][1], "final membrane")
    assert_same_bits(outs[0][2], outs[1][2], "checkpoints")
    assert_same_bits(outs[1][2][0], m0, "first checkpoint")


@pytest.mark.parametrize("B,N", SHAPES)
@pytest.mark.parametrize("T", [1, 17])
def test_currents_recurrence(B, N, T):
    x, m0 = _case(B, N, T, B + N + 1)
    outs = []
    for in_place in (False, True):
        m = m0.clone()
        out = {"m_final": m if in_place else torch.empty_like(m0), "spikes": torch.empty_like(x),
               "pre": torch.empty_like(x), "words": torch.empty((T, B, -(-N // 32)), dtype=torch.int32, device=DEV),
               "counts": torch.zeros_like(m0), "ckpt": torch.empty((-(-T // 4), B, N), device=DEV)}
        _lib.call("myelin_lif_currents_fwd", x.data_ptr(), m.data_ptr(), out["m_final"].data_ptr(),
                  out["spikes"].data_ptr(), out["pre"].data_ptr(), out["words"].data_ptr(), None,
                  out["counts"].data_ptr(), out["ckpt"].data_ptr(), T, B, N, 0, T, 0, 0, 4, 0.9, 1.0, -0.1, 10.0,
                  _lib.RULE_THRESHOLD, _lib.stream(x.device))
        outs.append(out)
    for name, want in outs[0].items():
        assert torch.equal(want, outs[1][name]), name
    assert_same_bits(outs[1]["ckpt"][0], m0, "first checkpoint")
