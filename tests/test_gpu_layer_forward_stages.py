"""The layer forward's stages (8 or 16 steps; a stage in which a potential calls for the quotient is done again) against
the CPU oracle, bit for bit: step counts around the stage and checkpoint lengths, neurons that now and then or always fire
more than twice per step, thresholds that are not positive, subtract values whose double overflows, a bound that is no
number, and widths whose last block is partly empty for one, two and four neurons per lane."""
import pytest
import torch

from _util import gen

pytestmark = pytest.mark.gpu


def check(b, t, m, cap, bound, seed, records=False, syn=False):
    from oracle import exodus_ref as ref
    from oracle import sinabs_cpu as sc
    from sinabs.exodus import _hip as hip
    g = gen(seed)
    n = b * m
    x = torch.randn(b, t, m, generator=g) * 0.5 + 0.1
    if n < 100000:
        x[torch.rand(b, t, m, generator=g) < 0.02] = 7.3          # sudden bursts
        x[:, :, m // 2] += 4.0                                    # one neuron fires many spikes in every step
    alpha = torch.rand(n, generator=g)
    v0 = torch.randn(n, generator=g) * 0.3
    th = 0.5 + torch.rand(n, generator=g)
    c = 0.3 + 0.5 * torch.rand(n, generator=g)
    lo = -0.5 * torch.ones(n)
    if n >= 8:
        th[1], th[n - 2] = -0.25, 0.0
        c[2] = 3e38
        if bound:
            lo[3] = float("nan")
    a_syn = 0.3 + 0.5 * torch.rand(n, generator=g) if syn else None
    rows = sc.bt_to_rows(x)
    if syn:
        rows = ref.leaky_forward((rows * a_syn[:, None]).contiguous(), torch.zeros(n), a_syn)
    ws, wv = ref.lif_forward(rows, v0, alpha, c, th, lo, bound, cap)
    d = lambda z: None if z is None else z.cuda()
    got = hip.layerLifForward(d(x), d(v0), torch.zeros(n).cuda() if syn else None, d(alpha), d(a_syn), d(c), d(th), d(lo),
                              bound, cap, True, False, wantRecords=records)
    vpost = wv - c[:, None] * ws
    same = lambda p, q: torch.equal(p.cpu().nan_to_num(nan=1234.5), q.nan_to_num(nan=1234.5))
    assert same(got["spikes"], sc.rows_to_bt(ws, b))
    assert same(got["v_last"], vpost[:, -1])
    if records:
        assert same(got["v_rec"], sc.rows_to_bt(vpost, b))
    every = hip.checkpointInterval()
    want_ck = torch.cat([v0[:, None], vpost[:, every - 1:-1:every]], 1)[:, :got["ckpt_v"].shape[1]]
    assert same(got["ckpt_v"], sc.rows_to_bt(want_ck.contiguous(), b))
    if cap != 1 and n < 100000:
        assert ws.max() > 1


@pytest.mark.parametrize("t", [1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 80, 97])
@pytest.mark.parametrize("m,cap,bound,records,syn", [(1, -1, False, False, False), (63, -1, True, False, True),
                                                     (257, 2, True, False, False), (130, 5, False, True, False),
                                                     (256, 1, False, False, True)])
def test_stage_lengths(t, m, cap, bound, records, syn):
    check(2, t, m, cap, bound, 100 * t + m, records, syn)


@pytest.mark.parametrize("b,t,m,cap", [(8, 41, 65538, -1), (3, 33, 180002, 2), (4, 19, 262148, -1), (1, 40, 1048580, 1)])
def test_several_neurons_per_lane(b, t, m, cap):
    """From 524 288 neurons on a lane holds two, from 1 048 576 on four where their number allows it."""
    check(b, t, m, cap, False, m)
    check(b, t, m, cap, True, m + 1, syn=True)


@pytest.mark.parametrize("b,t,m,cap", [(8, 1, 65538, -1), (3, 2, 180002, 2), (4, 3, 262148, -1), (1, 1, 1048580, 1)])
def test_a_step_or_two_with_several_neurons_per_lane(b, t, m, cap):
    check(b, t, m, cap, False, m)
    check(b, t, m, cap, True, m + 1, syn=True)


@pytest.mark.parametrize("b,t,m", [(4, 120, 131074), (2, 100, 524292)])
def test_stages_done_again_with_several_neurons_per_lane(b, t, m):
    """Long enough for waves to go to the exact steps and back several times (two and four neurons per lane)."""
    check(b, t, m, -1, False, m)
