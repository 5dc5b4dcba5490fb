"""The layer Functions called directly, with and without their optional arguments: the same outputs and gradients, bit for
bit (a layer names every argument)."""
import pytest
import torch

from _util import gen

pytestmark = pytest.mark.gpu
B, T, M = 2, 37, 19


def leaf(*shape, seed, lo=0.0, hi=1.0):
    return (torch.rand(shape, generator=gen(seed)) * (hi - lo) + lo).cuda().requires_grad_(True)


def grads(out, leaves):
    out.square().sum().backward()
    got = [z.grad for z in leaves]
    for z in leaves:
        z.grad = None
    return got


def same(p, q):
    return all((x is None and y is None) or torch.equal(x, y) for x, y in zip(p, q))


@pytest.mark.parametrize("syn", [False, True])
@pytest.mark.parametrize("learn", [False, True])
def test_spiking(syn, learn):
    from sinabs.exodus._compat import SingleExponential
    from sinabs.exodus.layer_function import SpikingLayerFunction as F
    x, a = leaf(B, T, M, seed=1, hi=3.0), leaf(B * M, seed=2, lo=0.6, hi=0.95).requires_grad_(learn)
    a_syn = leaf(B * M, seed=3, lo=0.3, hi=0.9).requires_grad_(learn) if syn else None
    zero, one = torch.zeros(B * M, device="cuda"), torch.ones(B * M, device="cuda")
    args = (x, a, a_syn, zero, zero if syn else None, one, one, None, SingleExponential(), 2, True, True)
    leaves = [z for z in (x, a, a_syn) if z is not None]
    want = None
    for more in ((None, False, True, None, None), (None, False, True), (None, False), (None,), ()):
        out = F.apply(*args, *more)
        got = [out[0], out[1], out[3]] + grads(out[0], leaves)
        assert (got[4] is not None) == learn
        want = want or got
        assert same(got, want)


@pytest.mark.parametrize("learn", [False, True])
def test_leaky(learn):
    from sinabs.exodus.layer_function import LeakyLayerFunction as F
    x, a = leaf(B, T, M, seed=1, lo=-1.0), leaf(B * M, seed=2, lo=0.6, hi=0.95).requires_grad_(learn)
    args = (x, a, torch.zeros(B * M, device="cuda"), True, True)
    want = None
    for more in ((None, None), (None,), ()):
        out = F.apply(*args, *more)
        got = list(out) + grads(out[0], (x, a))
        assert (got[4] is not None) == learn
        want = want or got
        assert same(got, want)


def test_time_constants_in_the_place_of_factors():
    """A time constant that takes no gradient, and one that does."""
    from sinabs.exodus.layer_function import LeakyLayerFunction as F
    x, v0 = leaf(B, T, M, seed=1, lo=-1.0), torch.zeros(B * M, device="cuda")
    for learn in (False, True):
        tau = leaf(M, seed=2, lo=5.0, hi=20.0).requires_grad_(learn)
        got = grads(F.apply(x, None, v0, True, False, None, tau)[0], (x, tau))
        alpha = torch.exp(-1.0 / tau.detach()).expand(B, M).flatten()
        assert torch.equal(got[0], grads(F.apply(x, alpha, v0, True, False)[0], (x,))[0])
        assert (got[1] is not None) == learn
