"""The leaky-integrator layer kernels at step counts around their stages (8 or 16 steps), widths whose last block is partly
empty and one, two and four neurons per lane: forward bit for bit against the CPU oracle, backward against the recurrence
in float64 (two roundings per step, forgotten after 1 / (1 - alpha) < 20 steps: 20 * 2^-24 = 1.2e-6 in the 2-norm; the
decay factor's gradient adds fp32 sums of 8 to 24 terms that partly cancel: 2e-5)."""
import pytest
import torch

from _util import gen

pytestmark = pytest.mark.gpu


def check(b, t, m, early, norm, uniform, seed):
    from oracle import exodus_ref as ref
    from oracle import sinabs_cpu as sc
    from sinabs.exodus import _hip as hip
    g, n = gen(seed), b * m
    x = torch.randn(b, t, m, generator=g)
    alpha = 0.3 + 0.65 * torch.rand(n, generator=g)
    v0, gv = torch.randn(n, generator=g), torch.randn(n, generator=g)
    rows = sc.bt_to_rows(x)
    if norm:
        rows = (1.0 - alpha[:, None]) * rows
    if early:
        rows = rows * alpha[:, None]
    want = sc.rows_to_bt(ref.leaky_forward(rows.contiguous(), v0, alpha), b)
    xd, ad, vd = x.cuda(), alpha.cuda(), v0.cuda()
    out, last, total = hip.layerLeakyForward(xd, vd, ad, early, norm, wantSum=True)
    assert torch.equal(out.cpu(), want) and torch.equal(last.cpu(), want[:, -1].flatten())
    mass = float(want.double().abs().sum())
    assert abs(float(total) - float(want.double().sum())) <= 32 * 2.0 ** -24 * mass     # fp32 sums of at most 32 outputs
    go = torch.full((1,), 0.3) if uniform else torch.randn(b, t, m, generator=g)
    gx, ga, gi = hip.layerLeakyBackward(go.cuda(), gv.cuda(), out, xd, vd, ad, early, norm, True,
                                        shape=(b, t, m) if uniform else None)
    plain = hip.layerLeakyBackward(go.cuda(), gv.cuda(), None, None, None, ad, early, norm, False,
                                   shape=(b, t, m) if uniform else None)
    assert torch.equal(plain[0], gx) and torch.equal(plain[2], gi) and plain[1] is None
    a, h = alpha.double().view(b, m).cuda(), gv.double().view(b, m).cuda()
    x64, o64, go64 = xd.double(), out.double(), go.double().cuda().expand(b, t, m)
    k = 1.0 - a if norm else torch.ones_like(a)
    w_x, w_a = torch.empty_like(x64), torch.zeros_like(a)
    for s in range(t - 1, -1, -1):
        gt = h + go64[:, s]
        h = gt * a
        gs = h if early else gt
        w_a += gt * (o64[:, s - 1] if s else vd.double().view(b, m))
        if early:
            w_a += gt * k * x64[:, s]
        if norm:
            w_a -= gs * x64[:, s]
        w_x[:, s] = gs * k
    err = lambda z, w: float((z.double() - w).norm() / w.norm())
    assert err(gx, w_x) <= 1.2e-6 and err(gi, h.flatten()) <= 1.2e-6 * max(1.0, float(go64.norm() / h.norm()))
    assert err(ga, w_a.flatten()) <= 2e-5


@pytest.mark.parametrize("t", [1, 2, 7, 8, 9, 15, 16, 17, 24, 31, 32, 33, 40, 47, 48, 49, 100])
@pytest.mark.parametrize("m,early,norm,uniform", [(1, False, False, False), (70, True, True, False), (257, False, True, True),
                                                  (320, True, False, False)])
def test_stage_lengths(t, m, early, norm, uniform):
    from sinabs.exodus import _hip as hip
    mode = hip.backwardTimeSplit(0)                            # small layers run another kernel otherwise
    try:
        check(2, t, m, early, norm, uniform, 10 * t + m)
    finally:
        hip.backwardTimeSplit(mode)


@pytest.mark.parametrize("b,t,m", [(5, 23, 60002), (3, 17, 180004), (2, 41, 131074)])
@pytest.mark.parametrize("uniform", [False, True])
def test_several_neurons_per_lane(b, t, m, uniform):
    """From 262 144 neurons on a lane holds two, from 524 288 on four where their number allows it."""
    check(b, t, m, False, False, uniform, m)
    check(b, t, m, True, True, uniform, m + 1)


@pytest.mark.parametrize("b,t,m", [(5, 1, 60002), (3, 2, 180004), (3, 3, 180004)])
@pytest.mark.parametrize("uniform", [False, True])
def test_a_step_or_two_with_several_neurons_per_lane(b, t, m, uniform):
    check(b, t, m, False, False, uniform, m)
    check(b, t, m, True, True, uniform, m + 1)
