"""Bitpacking at ragged row lengths, element sizes and base alignments, and
the counts and rates at the edges of their launch shapes: bit-exact against
the oracle."""

from __future__ import annotations

import pytest
import torch

import myelin_amd as myelin
from myelin_amd import _lib
from oracle import torch_ref as R
from tests.helpers import seeded

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _print_case(**kw):
    print("case:", " ".join(f"{k}={v}" for k, v in kw.items()), flush=True)


# rows of one word and less, rows starting on 16, 8, 4, 2 and 1 bytes, rows
# ending in each part of a word; rows narrower than an unpacking lane's 16
# elements
@pytest.mark.parametrize("n", [1, 3, 15, 16, 17, 24, 31, 32, 33, 40, 63, 64, 100, 1000, 2311, 2312])
@pytest.mark.parametrize("dtype", [torch.uint8, torch.bool, torch.bfloat16, torch.float32, torch.int64, torch.float64])
def test_ragged_rows_round_trip(n, dtype):
    rows = 67 if n < 1000 else 9
    for offset in (0, 1, 3):  # elements the tensor starts past its storage
        _print_case(test="ragged", n=n, dtype=dtype, offset=offset)
        g = seeded(n + offset)
        s = (torch.rand(rows * n + offset, generator=g) < 0.4).to(dtype)
        x = s.to(DEV)[offset:].view(rows, n)
        words, shape = R.pack_spikes(s[offset:].view(rows, n))
        pk = myelin.pack_spikes(x)
        assert torch.equal(pk.data.cpu(), words)
        assert torch.equal(myelin.unpack_spikes(pk, dtype=dtype), x)
        # an output that starts off 16 bytes
        out = torch.zeros(rows * n + offset, dtype=dtype, device=DEV)
        _lib.call("myelin_unpack", pk.data.data_ptr(), out[offset:].data_ptr(), _lib.DT[dtype], rows, n,
                  _lib.stream(out.device))
        assert torch.equal(out[offset:].view(rows, n), x) and not bool(out[:offset].any())


def test_values_other_than_one_and_signed_zeros():
    _print_case(test="ragged_values")
    half = torch.tensor([0x0000, 0x8000, 0x0001, 0x8001, 0x7C00, 0x7FFF, 0xFFFF, 0x3F80] * 5, dtype=torch.int32)
    for dtype in (torch.float16, torch.bfloat16):
        x = half.to(torch.int16).view(dtype)[:37]
        assert torch.equal(myelin.pack_spikes(x.to(DEV)).data.cpu(), R.pack_spikes(x)[0])
    x = torch.arange(256, dtype=torch.int32).to(torch.uint8)[:251]
    for y in (x, x.view(torch.int8)):
        assert torch.equal(myelin.pack_spikes(y.to(DEV)).data.cpu(), R.pack_spikes(y)[0])


# one workgroup an output, several adding to one (more than 32768 words an
# output), few rows an output (scattered), every leading dim kept; lane and
# wave rows
@pytest.mark.parametrize("shape,dim", [((300, 5, 2312), (0, -1)), ((600, 3, 8192), (0, -1)), ((40, 3, 70), None),
                                       ((5, 7, 700), (0, -1)), ((5, 7, 100), (0, -1)), ((6, 9, 700), -1),
                                       ((6, 9, 100), -1), ((3, 20, 4, 100), (1, -1))])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_rates_equal_the_oracle(shape, dim, dtype):
    _print_case(test="rates", shape=shape, dim=dim, dtype=dtype)
    s = (torch.rand(shape, generator=seeded(sum(shape))) < 0.3).float()
    words, _ = R.pack_spikes(s)
    pk = myelin.pack_spikes(s.to(DEV))
    assert torch.equal(myelin.packed_spike_rate(pk, dim=dim, dtype=dtype).cpu(),
                       R.packed_spike_rate(words, shape, dim, dtype))
    assert torch.equal(myelin.packed_spike_count(pk, dim=dim).cpu(), R.packed_spike_count(words, shape, dim))


# one block of rows and several (over 2040), columns that end inside a block
@pytest.mark.parametrize("R_,K,n", [(1, 1, 33), (255, 3, 700), (2040, 2, 65), (2041, 1, 100), (5000, 1, 2080)])
def test_counts_per_neuron_equal_the_dense_sum(R_, K, n):
    _print_case(test="keep_last", R=R_, K=K, n=n)
    s = torch.rand((R_, K, n), generator=seeded(R_ + n)) < 0.9
    assert torch.equal(myelin.packed_spike_count(myelin.pack_spikes(s.to(DEV)), dim=0).cpu(), s.long().sum(0))
