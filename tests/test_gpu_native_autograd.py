"""The C++ autograd Functions of the recurrences against the Python ones:
the same entry points, so outputs and gradients are equal bit for bit."""

import threading

import pytest
import torch

from myelin_amd import _lib, autograd

pytestmark = pytest.mark.gpu

PLAIN = (_lib.RULE_THRESHOLD, _lib.SG_NONE)
SURROGATE = (_lib.RULE_SURROGATE, 1)


def _inputs(shape, req):
    gen = torch.Generator().manual_seed(3)
    x = torch.randn(shape, generator=gen)
    m, a = torch.rand(shape[1:], generator=gen), torch.rand(shape[1:], generator=gen)
    return [t.cuda().requires_grad_(bool(req >> i & 1)) for i, t in enumerate((x, m, a))]


@pytest.mark.parametrize("shape", [(1, 1, 1), (17, 3, 33), (40, 5, 64)])
@pytest.mark.parametrize("codes", [PLAIN, SURROGATE])
@pytest.mark.parametrize("req", range(8))
def test_matches_python_functions(shape, codes, req):
    for outs in range(1, 8):
        got = []
        for lif, alif in ((autograd.lif, autograd.alif), (autograd.HipLIFFunction.apply, autograd.HipALIFFunction.apply)):
            x, m, a = ins = _inputs(shape, req)
            out = [*lif(x, m, 0.9, 1.0, 0.0, 10.0, *codes), *alif(x, m, a, 0.9, 0.95, 1.0, 0.2, 0.0, 10.0, *codes)]
            terms = [(t * torch.linspace(0.1, 1, t.numel(), device="cuda").view_as(t)).sum()
                     for i, t in enumerate(out) if outs >> (i % 3) & 1 and t.requires_grad]
            if terms:
                sum(terms).backward()
            got.append(([t.requires_grad for t in out], [t.detach() for t in out], [t.grad for t in ins]))
        (r0, o0, g0), (r1, o1, g1) = got
        assert r0 == r1
        for p, q in zip(o0 + g0, o1 + g1):
            assert (p is None) == (q is None)
            assert p is None or torch.equal(p, q)


def test_errors_and_saved_tensors():
    x, m, _ = _inputs((20, 2, 4), 1)
    with pytest.raises(ValueError, match="spike rule 99"):
        autograd.lif(x, m, 0.9, 1.0, 0.0, 10.0, 99, 1)
    out = autograd.lif(x, m, 0.9, 1.0, 0.0, 10.0, _lib.RULE_SURROGATE, 77)
    with pytest.raises(ValueError, match="surrogate code 77"):  # raised on the engine's thread
        out[1].sum().backward()

    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.cuda()):
        out = autograd.lif(x, m, 0.9, 1.0, 0.0, 10.0, *SURROGATE)
    assert packed == [x.shape, (2, 2, 4)]
    out[1].sum().backward()
    with pytest.raises(RuntimeError, match="second time"):
        out[1].sum().backward()
    out = autograd.lif(x, m, 0.9, 1.0, 0.0, 10.0, *SURROGATE)
    with torch.no_grad():
        x.add_(1)
    with pytest.raises(RuntimeError, match="inplace"):
        out[1].sum().backward()


def test_what_stays_with_the_python_functions():
    x, m, _ = _inputs((4, 2, 8), 1)

    class Sub(torch.Tensor):
        pass

    assert autograd.plain(x, m) and autograd.plain(x, torch.nn.Parameter(m))
    assert not autograd.plain(x.detach().as_subclass(Sub), m)
    seen = []
    torch.func.grad(lambda t: seen.append(autograd.plain(t, m)) or t.sum())(x.detach())
    with torch.autograd.forward_ad.dual_level():
        seen.append(autograd.plain(x, m))
    torch.jit.trace(lambda t: seen.append(autograd.plain(t, m)) or t * 2, x.detach(), check_trace=False)
    assert seen == [False, False, False]


def test_streams_and_threads():
    want = {}

    def run(i, results):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(side):
            x, m, _ = _inputs((33, 4, 32 + i), 3)
            for _ in range(8):
                out = autograd.lif(x, m, 0.9, 1.0, 0.0, 10.0, *SURROGATE)
                gx, gm = torch.autograd.grad((out[0].sum() + out[1].sum()), (x, m))
            results[i] = (gx.cpu(), gm.cpu())

    for i in range(4):
        run(i, want)
    got = {}
    threads = [threading.Thread(target=run, args=(i, got)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(4):
        assert all(torch.equal(p, q) for p, q in zip(want[i], got[i]))
