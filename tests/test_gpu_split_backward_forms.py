"""The backward kernel with one lane per neuron and 32 steps, over every form of the call that reaches it (synapse,
surrogate from a tensor, gradients on state records, one gradient value, any number of chunks): against the adjoint
recurrences in float64 on the forward pass's own values, with the one-lane kernel held against the same; the two differ in
some bit, which shows that both ran.

Bound: a gradient is a chain of products and sums with three roundings per step and factors of at most one in magnitude,
so 2^-24 times a few times the chain's effective length (the decay forgets after 1 / (1 - a_mem) < 30 steps): 2e-6 in the
2-norm; the sums over a neuron's steps add fp32 partial sums of 8 terms (32 in the one-lane kernel): 2e-5 where the terms
partly cancel."""
import pytest
import torch

from _util import gen

pytestmark = pytest.mark.gpu


@pytest.fixture()
def hip():
    from sinabs.exodus import _hip
    before = _hip.backwardTimeSplit(-1)
    yield _hip
    _hip.backwardTimeSplit(before)


def adjoint64(x, go, sg, v, i, vpost, v0, i0, gv, gi, qv, qi, am, a_syn, c, lo, early, norm):
    d = lambda z: None if z is None else z.double()
    go, sg, v, i, vpost, am, c = (d(z) for z in (go, sg, v, i, vpost, am, c))
    b, t, m = go.shape
    shape = lambda z: z.view(b, m)
    am, c = shape(am), shape(c)
    syn = a_syn is not None
    a_s = shape(d(a_syn)) if syn else None
    k = 1.0 - am if norm else torch.ones_like(am)
    h, hm = shape(d(gv)).clone(), shape(d(gi)).clone() if syn else None
    gx, g_am, g_as = torch.empty_like(go), torch.zeros_like(am), torch.zeros_like(am)
    for s in range(t - 1, -1, -1):
        below = h if qv is None else h + d(qv)[:, s]
        lam = sg[:, s] * go[:, s] + (1.0 - c * sg[:, s]) * below
        if lo is not None:
            lam = torch.where(v[:, s] > shape(d(lo)), lam, torch.zeros_like(lam))
        g_am += lam * (vpost[:, s - 1] if s else shape(d(v0)))
        if norm:
            g_am -= lam * i[:, s]
        h = am * lam
        if syn:
            mu = hm + k * lam + (0.0 if qi is None else d(qi)[:, s])
            g_as += mu * (i[:, s] / a_s if early else (i[:, s - 1] if s else shape(d(i0))))
            hm = a_s * mu
            gx[:, s] = mu * a_s if early else mu
        else:
            gx[:, s] = k * lam
    return gx, g_am.flatten(), g_as.flatten(), h.flatten(), hm.flatten() if syn else None


FORMS = [dict(), dict(syn=True), dict(syn=True, early=False, norm=False, cap=-1), dict(clamp=True, cap=1),
         dict(syn=True, clamp=True, cap=2, uniform=True), dict(uniform=True, norm=False, cap=-1), dict(tensor=True),
         dict(tensor=True, syn=True, clamp=True), dict(rec=True), dict(rec=True, syn=True, clamp=True),
         dict(rec=True, tensor=True, syn=True), dict(kind=2, syn=True), dict(kind=3, syn=True, cap=2)]


@pytest.mark.parametrize("form", FORMS, ids=lambda f: "-".join(f"{k}{v}" for k, v in f.items()) or "plain")
@pytest.mark.parametrize("b,t,m", [(2, 33, 70), (1, 64, 1), (3, 257, 17), (2, 520, 33), (1, 1024, 65), (1, 1100, 20),
                                   (2, 95, 64)])
def test_against_float64(hip, form, b, t, m):
    f = dict(syn=False, early=True, norm=True, cap=2, clamp=False, uniform=False, tensor=False, rec=False, kind=1)
    f.update(form)
    n = b * m
    u = lambda s, lo, hi: (torch.rand(n, generator=gen(s)) * (hi - lo) + lo).cuda()
    r = lambda s, scale: (torch.randn(b, t, m, generator=gen(s)) * scale).cuda()
    x = r(1, 3.0 if f["norm"] else 0.8) + 0.4
    am, c, th = u(2, 0.6, 0.96), u(3, 0.4, 1.0), u(4, 0.6, 1.3)
    a_syn = u(5, 0.3, 0.9) if f["syn"] else None
    v0, gv = u(6, -0.3, 0.5), u(7, -1.0, 1.0)
    i0, gi = (u(8, -0.3, 0.5), u(9, -1.0, 1.0)) if f["syn"] else (None, None)
    lo = u(10, -0.8, -0.1) if f["clamp"] else None
    go = torch.full((1,), 0.7, device="cuda") if f["uniform"] else r(11, 1.0)
    qv, qi = (r(12, 0.3), r(13, 0.3) if f["syn"] else None) if f["rec"] else (None, None)
    fwd = lambda **kw: hip.layerLifForward(x, v0, i0, am, a_syn, c, th, lo, f["clamp"], f["cap"], f["early"], f["norm"], **kw)
    post = fwd(wantRecords=True)
    v = fwd(wantPreReset=True)["v_rec"]
    i = post["i_rec"] if f["syn"] else x
    p0, kind = {1: 0.5, 2: 0.6, 3: 0.7}[f["kind"]], 0 if f["tensor"] else f["kind"]
    th3 = th.view(b, 1, m)
    if f["kind"] == 1:
        sg = torch.exp(-(v - th3).abs().double() / (th3.double() * p0)) / (th3.double() * p0)
    elif f["kind"] == 2:
        w = v - 0.5 * th3
        w = torch.where(v >= th3, w.remainder(th3), w)
        sg = torch.exp(-(w - 0.5 * th3).abs().double() / p0) / th3.double()
    else:
        sg = (v >= th3 - p0).double() / th3.double()
    surr = sg.float() if f["tensor"] else None
    full = go.expand(b, t, m) if f["uniform"] else go
    want = adjoint64(x, full, surr if f["tensor"] else sg, v, i, post["v_rec"], v0, i0, gv, gi, qv, qi, am, a_syn, c, lo,
                     f["early"], f["norm"])

    def run(mode):
        hip.backwardTimeSplit(mode)
        return hip.layerLifBackward(go, gv, gi, x, post["ckpt_v"], post["ckpt_i"], v0, i0, am, a_syn, c, th, lo, f["clamp"],
                                    f["cap"], f["early"], f["norm"], kind, p0, 1.0, surr=surr, gradVRec=qv, gradIRec=qi,
                                    gradUniform=f["uniform"])
    split, again, one = run(1), run(3), run(0)
    for name, bound, s, a, o, w in zip(("x", "alpha_mem", "alpha_syn", "v_init", "i_init"), (2e-6, 2e-5, 2e-5, 1e-5, 1e-5),
                                       split, again, one, want):
        if w is None or s is None:
            assert s is None
            continue
        assert torch.equal(s, a)                       # small layers take this kernel by default
        err = lambda z: float((z.double() - w).norm() / w.norm().clamp_min(1e-30))
        print(f"float64 error {name}: split {err(s):.2e} one lane {err(o):.2e}")
        assert err(s) <= bound and err(o) <= bound, (name, err(s), err(o))
    # what enters a chunk is folded in one kernel and walked in the other: some value of some neuron differs
    assert n < 16 or not torch.equal(split[0], one[0]), "the kernel with one lane per neuron and 32 steps did not run"


@pytest.mark.parametrize("form", [dict(), dict(syn=True, clamp=True, cap=2, uniform=True), dict(rec=True, tensor=True, syn=True)],
                         ids=["plain", "syn", "records"])
@pytest.mark.parametrize("b,t,m", [(5, 545, 1030),     # more than 256 blocks of 16 neurons: groups of up to 16 chunks
                                   (9, 300, 1030),     # more than 256 blocks of 32: two groups of 5 chunks, the lanes hold 6
                                   (300, 530, 33), (1200, 290, 3)])   # 17 chunks in groups of 6, 10 in lanes for 8
def test_groups_of_fewer_chunks_where_the_blocks_are_many(hip, form, b, t, m):
    test_against_float64(hip, form, b, t, m)


def test_a_clamped_step_stops_what_is_not_a_number(hip):
    """A gradient that is no number at the final state ends where the potential was clamped, chunk by chunk as step by
    step."""
    b, t, m = 1, 200, 5
    x = torch.full((b, t, m), 0.1, device="cuda")
    x[:, 100:103] = -50.0                              # clamped there, in the fourth chunk of seven
    x[:, 191, :2] = -50.0                              # the sixth chunk's last step
    one, zero = torch.ones(m, device="cuda"), torch.zeros(m, device="cuda")
    am, a_syn, lo = 0.9 * one, 0.5 * one, -one
    f = hip.layerLifForward(x, zero, zero, am, a_syn, one, one, lo, True, 2, True, True)
    go = torch.ones_like(x)
    out = []
    for mode in (0, 1):
        hip.backwardTimeSplit(mode)
        out.append(hip.layerLifBackward(go, float("nan") * one, zero, x, f["ckpt_v"], f["ckpt_i"], zero, zero, am, a_syn, one,
                                        one, lo, True, 2, True, True, 1, 0.5, 1.0))
    assert torch.equal(out[0][0].isnan(), out[1][0].isnan()) and bool(out[0][0].isnan().any())
    assert torch.allclose(out[0][0].nan_to_num(), out[1][0].nan_to_num(), rtol=1e-5, atol=1e-7)
    f = hip.layerLifForward(x, zero, None, am, None, one, one, lo, True, 2, True, True)
    out = []
    for mode in (0, 1):
        hip.backwardTimeSplit(mode)
        out.append(hip.layerLifBackward(go, float("nan") * one, None, x, f["ckpt_v"], None, zero, None, am, None, one,
                                        one, lo, True, 2, True, True, 1, 0.5, 1.0))
    assert torch.equal(out[0][0].isnan(), out[1][0].isnan()) and not bool(out[1][0][:, :100].isnan().any())


def steep(hip, b, t, m, syn, quiet=()):
    """A layer without leak whose potential sits on the threshold in every step but the ``quiet`` ones, with a surrogate so
    narrow that every such step multiplies the adjoint by 1 - c s = -19: 32 of them by 8e40, more than a float holds."""
    one, zero = torch.ones(b * m, device="cuda"), torch.zeros(b * m, device="cuda")
    x = torch.ones(b, t, m, device="cuda")
    for lo, hi in quiet:
        x[:, lo:hi] = 0.0
    a_syn = zero if syn else None                      # forgets at once: the current is the input
    kw = dict(early=False, norm=False, cap=-1)
    args = (x, zero, zero if syn else None, one, a_syn, one, one, None, False, kw["cap"], kw["early"], kw["norm"])
    post, pre = hip.layerLifForward(*args, wantRecords=True), hip.layerLifForward(*args, wantPreReset=True)
    p0 = 0.05

    def backward(mode, go, gv, gi, rec=None):
        hip.backwardTimeSplit(mode)
        return hip.layerLifBackward(go, gv, gi, x, post["ckpt_v"], post["ckpt_i"], zero, zero if syn else None, one, a_syn,
                                    one, one, None, False, -1, False, False, 1, p0, 1.0, gradVRec=rec)
    v = pre["v_rec"]
    sg = torch.exp(-(v - 1.0).abs().double() / p0) / p0
    want = lambda go, gv, gi, rec=None: adjoint64(
        x, go, sg, v, post["i_rec"] if syn else x, post["v_rec"], zero, zero, gv, gi, rec,
        torch.zeros_like(x) if rec is not None and syn else None, one, a_syn, one, None, False, False)
    return backward, want, zero


@pytest.mark.parametrize("syn", [False, True])
@pytest.mark.parametrize("rec", [False, True])
@pytest.mark.parametrize("t", [96, 1000, 1100])
def test_chunks_whose_factors_overflow_pass_nothing_on_where_nothing_enters(hip, syn, rec, t):
    """A loss on the first steps only: exactly 0 enters every chunk but the first from later steps, whatever its factors.
    Three steps with factors of 19: about ten roundings, and the exponential's error of 2e-7 three times."""
    b, m = 2, 20
    backward, want, zero = steep(hip, b, t, m, syn)
    go = torch.zeros(b, t, m, device="cuda")
    go[:, :3] = torch.randn(b, 3, m, generator=gen(1)).cuda()
    qv = torch.zeros_like(go) if rec else None
    w, got, one = want(go, zero, zero, qv), backward(1, go, zero, zero, qv), backward(0, go, zero, zero, qv)
    for z in (got, one):
        assert bool(z[0].isfinite().all()) and not bool(z[0][:, 3:].any())
        for mine, ideal in ((z[0], w[0]), (z[1], w[1]), (z[3], w[3])) + (((z[2], w[2]),) if syn else ()):
            assert float((mine.double() - ideal).norm()) <= 2e-6 * float(ideal.norm())


@pytest.mark.parametrize("syn", [False, True])
def test_a_small_gradient_through_a_chunk_whose_factors_overflow(hip, syn):
    """1e-30 at the final state grows by 8e40 within one chunk: infinity times 1e-30 would be infinite."""
    b, t, m = 2, 96, 20
    backward, want, zero = steep(hip, b, t, m, syn, quiet=((0, 32), (64, 96)))
    go, gv = torch.zeros(b, t, m, device="cuda"), torch.full((b * m,), 1e-30, device="cuda")
    w, got, one = want(go, gv, zero), backward(1, go, gv, zero), backward(0, go, gv, zero)
    assert float(w[0].abs().max()) > 1e10
    for z in (got, one):                               # 32 factors: three roundings and the exponential's error each
        assert float((z[0].double() - w[0]).norm()) <= 2e-5 * float(w[0].norm())
    assert torch.equal(got[0], one[0])                 # passed on step by step, as one lane per neuron does it


def test_a_gradient_that_is_no_number_among_ordinary_neurons(hip):
    """One neuron's final state has a gradient that is no number: its block passes on chunk by chunk, the others fold."""
    b, t, m = 1, 300, 200
    x = (torch.randn(b, t, m, generator=gen(1)) * 0.8 + 0.4).cuda()
    one, zero = torch.ones(m, device="cuda"), torch.zeros(m, device="cuda")
    f = hip.layerLifForward(x, zero, zero, 0.9 * one, 0.5 * one, one, one, None, False, 2, True, True)
    go, gv = torch.randn(b, t, m, generator=gen(2)).cuda(), zero.clone()
    gv[70] = float("nan")
    out = []
    for mode in (0, 1):
        hip.backwardTimeSplit(mode)
        out.append(hip.layerLifBackward(go, gv, zero, x, f["ckpt_v"], f["ckpt_i"], zero, zero, 0.9 * one, 0.5 * one, one, one,
                                        None, False, 2, True, True, 1, 0.5, 1.0)[0])
    assert torch.equal(out[0].isnan(), out[1].isnan()) and bool(out[1][:, :, 70].isnan().all())
    assert int(out[1].isnan().sum()) == t
    assert float((out[0] - out[1]).nan_to_num().norm()) <= 4e-6 * float(out[0].nan_to_num().norm())
