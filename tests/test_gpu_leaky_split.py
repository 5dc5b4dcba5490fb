"""The leaky layer's backward pass of small layers (a lane per neuron and chunk of 32 steps) against the same recurrence in float64:
ends of chunks, groups and blocks, every form of the call, factors and gradients that do not survive a fold."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def reference(go, gvl, out, x, v0, a, early, norm):
    """In float64 on the kernel's forward values: grad_x, the gradient of alpha, that of the initial state."""
    go, out, x, a, v0 = (z.double() for z in (go, out, x, a, v0))
    h = gvl.double() if gvl is not None else torch.zeros_like(a)
    gx, ga = torch.empty_like(go), torch.zeros_like(a)
    for t in range(go.shape[1] - 1, -1, -1):
        g = h + go[:, t]
        h = g * a
        r = h if early else g
        ga += g * (out[:, t - 1] if t else v0)
        if early:
            ga += g * ((1 - a) * x[:, t] if norm else x[:, t])
        if norm:
            ga -= r * x[:, t]
            r = r * (1 - a)
        gx[:, t] = r
    return gx, ga, h


def run(b, t, m, early, norm, gvl, uniform, alpha, split, poke=None):
    from sinabs.exodus import _hip as hip
    g = torch.Generator(device="cuda").manual_seed(t * 100 + m)
    R = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, v0, gl = R(b, t, m), R(b, m), R(b, m) if gvl else None
    a = alpha(torch.rand(b, m, generator=g, device="cuda"))
    go = torch.full((b, t, m), 0.7, device="cuda") if uniform else R(b, t, m)
    if poke is not None:
        poke(go)
    before = hip.backwardTimeSplit(3 if split else 0)
    try:
        return calls(hip, b, t, m, early, norm, x, v0, gl, a, go, uniform)
    finally:
        hip.backwardTimeSplit(before)


def calls(hip, b, t, m, early, norm, x, v0, gl, a, go, uniform):
    out = hip.layerLeakyForward(x, v0.flatten(), a.flatten(), early, norm)[0]
    one = torch.full((1,), 0.7, device="cuda")
    gx, ga, gv = hip.layerLeakyBackward(one if uniform else go, None if gl is None else gl.flatten(), out, x, v0.flatten(), a.flatten(),
                                        early, norm, True, shape=(b, t, m) if uniform else None)
    plain = hip.layerLeakyBackward(one if uniform else go, None if gl is None else gl.flatten(), None, None, None, a.flatten(), early,
                                   norm, False, shape=(b, t, m) if uniform else None)
    assert torch.equal(torch.nan_to_num(plain[0]), torch.nan_to_num(gx)) and plain[1] is None
    return (gx, ga.view(b, m), gv.view(b, m)), (go, gl, out, x, v0, a, early, norm)


@pytest.mark.parametrize("t", [33, 63, 64, 65, 96, 257, 300, 512, 513, 1024, 1025, 1100])
@pytest.mark.parametrize("b,m", [(1, 1), (2, 15), (2, 16), (1, 17), (2, 65), (4, 300), (1, 16384)])
def test_against_float64(t, b, m):
    for case, (early, norm) in enumerate(((False, False), (True, False), (False, True), (True, True))):
        gvl, uniform = (t + case) % 2 == 0, (t + m + case) % 3 == 0
        got, given = run(b, t, m, early, norm, gvl, uniform, lambda r: 0.6 + 0.399 * r, True)
        gx, ga, gv = reference(*given)
        x, a, out = given[3].double(), given[5].double(), given[2].double()
        # a step rounds twice, and what it loses fades with the factor: 2 / (1 - a) roundings of the largest adjoint, and a few for
        # the results themselves; the sum over the steps has them with each of its terms
        u, g_most = 2.0 ** -24, gx.abs().amax(1) / torch.minimum((a if early else 1.0 + 0 * a), 1 - a if norm else 1.0 + 0 * a)
        per_step = u * (2 / (1 - a) + 8) * g_most.maximum(gv.abs() / a)
        terms = out.abs().sum(1) + given[4].double().abs() + 2 * x.abs().sum(1)
        for p, q, most in zip(got, (gx, ga, gv), (per_step[:, None], per_step * terms, per_step)):
            assert bool(((p.double() - q).abs() <= most).all())


@pytest.mark.parametrize("kind", ["above one", "negative", "zero", "infinite gradient", "no number"])
def test_what_a_fold_would_spoil(kind):
    alpha = {"above one": lambda r: 1.0 + r, "negative": lambda r: -0.9 * r, "zero": lambda r: 0.0 * r}.get(kind, lambda r: 0.5 * r)

    def poke(go):
        if kind == "above one":
            go[:, 8:] = 0                                      # factors whose powers leave the floats' range meet nothing but zeros
        if kind == "infinite gradient":
            go[:, 290] = float("inf")
        if kind == "no number":
            go[0, 250, 3] = float("nan")
    got, _ = run(2, 300, 40, False, False, False, False, alpha, True, poke)
    want, _ = run(2, 300, 40, False, False, False, False, alpha, False, poke)
    for p, q in zip(got, want):
        some = q[torch.isfinite(q)].abs()
        assert torch.allclose(p, q, rtol=1e-5, atol=1e-5 * float(some.max()) if some.numel() else 0.0, equal_nan=True)


@pytest.mark.parametrize("early,norm", [(False, False), (True, True)])
def test_the_switch_of_the_spiking_layers_is_theirs_too(early, norm):
    """Mode 0 gives the kernel with one lane per neuron, which a batch beyond the limit of 16 384 neurons has in mode 1."""
    from sinabs.exodus import _hip as hip
    b, t, m = 41, 300, 400                                     # 16 400 neurons
    g = torch.Generator(device="cuda").manual_seed(1)
    x, go = (torch.randn(b, t, m, generator=g, device="cuda") for _ in range(2))
    a, v0 = 0.6 + 0.399 * torch.rand(b, m, generator=g, device="cuda"), torch.randn(b, m, generator=g, device="cuda")

    def backward(mode, some):
        before = hip.backwardTimeSplit(mode)
        try:
            out = hip.layerLeakyForward(x[some], v0[some].flatten(), a[some].flatten(), early, norm)[0]
            return hip.layerLeakyBackward(go[some], None, out, x[some], v0[some].flatten(), a[some].flatten(), early, norm, True)[0]
        finally:
            hip.backwardTimeSplit(before)
    whole, some = slice(0, b), slice(0, 40)
    one_lane = backward(1, whole)[some]
    assert torch.equal(backward(0, some), one_lane) and torch.equal(backward(0, whole)[some], one_lane)
    assert not torch.equal(backward(1, some), one_lane)
    assert torch.equal(backward(3, some), backward(1, some)) and not torch.equal(backward(3, whole)[some], one_lane)
