"""The recurrences choose one or two neurons per lane by the grid, and two
also where a row has an odd length.  Neurons are independent, so any grid's
neurons equal the same neurons run alone (a small grid, one per lane, which
test_gpu_recurrence holds against the oracle), bit for bit."""

from __future__ import annotations

import pytest
import torch

import myelin_amd as myelin
from tests.helpers import assert_same_bits

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _print_case(**kw):
    print("case:", " ".join(f"{k}={v}" for k, v in kw.items()), flush=True)


# around one, two and three waves per SIMD, odd and even; T with full blocks
# of 8, 16 and 32 steps, remainders and checkpoints every 16
@pytest.mark.parametrize("B,N", [(1, 65535), (1, 65537), (3, 30001), (2, 65536), (1, 131073), (5, 39321), (3, 87383)])
@pytest.mark.parametrize("T", [16, 31, 49])
@pytest.mark.parametrize("kind", ["lif", "alif", "plain"])
def test_neurons_do_not_depend_on_the_grid(B, N, T, kind):
    _print_case(test="grids", B=B, N=N, T=T, kind=kind)
    g = torch.Generator(device=DEV).manual_seed(B * N + T)
    x = 0.25 + 0.6 * torch.randn((T, B, N), generator=g, device=DEV)
    gs = torch.randn((T, B, N), generator=g, device=DEV)
    m0 = 0.5 * torch.rand((B, N), generator=g, device=DEV)
    a0 = 0.2 * torch.rand((B, N), generator=g, device=DEV)
    pick = torch.tensor([0, 1, 2, 63, 64, 127, 128, N // 2, N - 130, N - 65, N - 64, N - 2, N - 1], device=DEV)

    def run(x, gs, m0, a0):
        if kind == "plain":
            st, s = myelin.lif_forward(x, myelin.LIFState(m0), myelin.LIFParams())
            return [st.membrane, s]
        x = x.clone().requires_grad_()
        if kind == "lif":
            st, s = myelin.surrogate_lif_forward(x, myelin.LIFState(m0), myelin.LIFParams(reset=-0.1))
            outs = [st.membrane]
        else:
            st, s = myelin.surrogate_alif_forward(x, myelin.ALIFState(m0, a0), myelin.ALIFParams(reset=-0.1),
                                                  surrogate="fast_sigmoid")
            outs = [st.membrane, st.adaptation]
        return [*outs, s.detach(), *torch.autograd.grad([s, st.membrane], [x], [gs, m0])]

    full = run(x, gs, m0, a0)
    part = run(*(t[..., pick].contiguous() for t in (x, gs, m0, a0)))
    for i, (f, p) in enumerate(zip(full, part)):
        assert_same_bits(f[..., pick].contiguous(), p, f"output {i}")


# blocks of 32 and 16 steps (a small and a large grid), word pairs and single
# words, remainders of T and of the last word
@pytest.mark.parametrize("T,B,N", [(1, 1, 1), (32, 3, 33), (33, 2, 95), (70, 4, 1000), (17, 3, 97), (40, 70, 4097),
                                   (31, 33, 9000)])
def test_packed_forward_equals_dense_then_pack(T, B, N):
    _print_case(test="packed", T=T, B=B, N=N)
    g = torch.Generator(device=DEV).manual_seed(T + B + N)
    x = 0.25 + 0.6 * torch.randn((T, B, N), generator=g, device=DEV)
    m0 = 0.5 * torch.rand((B, N), generator=g, device=DEV)
    p = myelin.LIFParams(reset=-0.1)
    st, s = myelin.lif_forward(x, myelin.LIFState(m0), p)
    sp, pk = myelin.lif_forward_packed_spikes(x, myelin.LIFState(m0), p)
    assert torch.equal(pk.data, myelin.pack_spikes(s).data)
    assert_same_bits(sp.membrane, st.membrane, "membrane")
