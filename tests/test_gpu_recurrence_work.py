"""One or two neurons per lane, and the loads kept in flight, follow the grid
and how much arithmetic a step of the surrogate is: whatever is chosen, a
neuron's results are those of the same neuron run in a small grid, bit for
bit."""

from __future__ import annotations

import pytest
import torch

import myelin_amd as myelin
from tests.helpers import assert_same_bits

pytestmark = pytest.mark.gpu
DEV = "cuda"


# one wave per SIMD and its edges (with the extra waves that do not count), and
# the lines of two, three and seven; rows of whole lines and odd ones
@pytest.mark.parametrize("N", [65536, 65537, 67585, 73760, 98304, 131073, 135169, 196608, 196609, 458753])
@pytest.mark.parametrize("surrogate", ["fast_sigmoid", "sigmoid", "atan", "multi_gaussian"])
@pytest.mark.parametrize("hard", [True, False])
@pytest.mark.parametrize("alif", [False, True])
def test_neurons_do_not_depend_on_the_grid(N, surrogate, hard, alif):
    print("case: recurrence_work", N, surrogate, hard, alif, flush=True)
    T = 33
    g = torch.Generator(device=DEV).manual_seed(N)
    x = 0.25 + 0.6 * torch.randn((T, 1, N), generator=g, device=DEV)
    gs = torch.randn((T, 1, N), generator=g, device=DEV)
    m0 = 0.5 * torch.rand((1, N), generator=g, device=DEV)
    a0 = 0.2 * torch.rand((1, N), generator=g, device=DEV)
    pick = torch.tensor([0, 1, 63, 64, 127, 128, N // 2, N - 130, N - 65, N - 64, N - 2, N - 1], device=DEV)

    def run(x, gs, m0, a0):
        x = x.clone().requires_grad_()
        if alif:
            st, s = myelin.surrogate_alif_forward(x, myelin.ALIFState(m0, a0), myelin.ALIFParams(), surrogate=surrogate,
                                                  hard_forward=hard)
        else:
            st, s = myelin.surrogate_lif_forward(x, myelin.LIFState(m0), myelin.LIFParams(), surrogate=surrogate,
                                                 hard_forward=hard, backend="torch")
        return [st.membrane.detach(), s.detach(), *torch.autograd.grad([s, st.membrane], [x], [gs, m0])]

    full = run(x, gs, m0, a0)
    part = run(*(t[..., pick].contiguous() for t in (x, gs, m0, a0)))
    for f, p, what in zip(full, part, ("membrane", "spikes", "gx")):
        assert_same_bits(f[..., pick].contiguous(), p, what)
