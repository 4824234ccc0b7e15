"""Packed counts and rates onto few outputs: exact, and split over workgroups
where one would walk many rows alone."""

from __future__ import annotations

import pytest
import torch

import myelin_amd as myelin
from tests.helpers import seeded

pytestmark = pytest.mark.gpu
DEV = "cuda"


# rows of one to three words; up to 320 rows an output (one workgroup sums
# them), a row more, and tens of thousands
@pytest.mark.parametrize("shape", [(320, 3, 10), (321, 3, 10), (64, 5, 70), (65, 5, 33), (1000, 32, 10), (200, 128, 32)])
@pytest.mark.parametrize("dim", [None, (0, -1), (1, -1), (0, 1)])
def test_counts_and_rates(shape, dim):
    print("case: count_split", shape, dim, flush=True)
    x = (torch.rand(shape, generator=seeded(shape[0])) < 0.3).to(torch.uint8)
    packed = myelin.pack_spikes(x.to(DEV))
    want = x.long().sum() if dim is None else x.long().sum(dim)
    size = x.numel() // want.numel()
    assert torch.equal(myelin.packed_spike_count(packed, dim=dim).cpu(), want)
    assert torch.equal(myelin.packed_spike_rate(packed, dim=dim).cpu(), want.float() / size)
    assert torch.equal(myelin.packed_spike_rate(packed, dim=dim, dtype=torch.float64).cpu(), want.double() / size)


def test_one_output_of_many_short_rows_is_split():
    """25,600 rows of one word: by one workgroup 620 us, by many 11; a count
    of every row, which reads the same words, takes 9."""

    packed = myelin.pack_spikes((torch.rand(200, 128, 10, generator=seeded(1)) < 0.3).to(DEV))

    def us(dim):
        best = float("inf")
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        for _ in range(5):
            start.record()
            for _ in range(10):
                myelin.packed_spike_count(packed, dim=dim)
            end.record()
            torch.cuda.synchronize()
            best = min(best, start.elapsed_time(end) * 100)
        return best

    us(None)
    assert us(None) < 8 * us(-1)
