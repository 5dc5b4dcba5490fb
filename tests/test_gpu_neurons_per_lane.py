"""The forward layer kernels at sizes on both sides of the rule that picks one, two or four neurons per lane: every batch
element equals, bit for bit, the same element computed alone (too few neurons for more than one per lane)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# per case: neurons per lane of the spiking and of the leaky forward
@pytest.mark.parametrize("b,t,m,spiking,leaky", [
    (32, 5, 131072, 4, 4),
    (33, 3, 131076, 4, 4),    # steps that do not fill whole sectors
    (27, 4, 65528, 4, 4),     # with shared sectors from 24 waves per compute unit on
    (16, 4, 65528, 2, 2),
    (32, 9, 32768, 2, 2),     # though four would leave 16 waves per compute unit
    (64, 17, 8192, 2, 2),     # 1024 blocks on 256 units
    (64, 17, 8176, 1, 2),     # below 16 waves per compute unit
    (32, 9, 8192, 1, 2),      # 8 waves per compute unit
    (32, 9, 8176, 1, 1),
    (64, 17, 12544, 1, 1),    # 1600 blocks of two per lane spread unevenly, 3136 of one do not
    (64, 9, 12545, 1, 1),     # odd
])
def test_every_batch_element_equals_itself_alone(b, t, m, spiking, leaky):
    from sinabs.exodus import _hip as hip
    assert hip.launchShape("forward", b, m)[0] == spiking and hip.launchShape("leaky forward", b, m)[0] == leaky
    assert hip.launchShape("forward", 1, m)[0] == 1 and hip.launchShape("leaky forward", 1, m)[0] == 1
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.empty(b, t, m, device="cuda").normal_(0.2, 0.8, generator=g)
    full = lambda n, v: torch.full((n,), v, device="cuda")

    def both(xx):
        n = xx.shape[0] * m
        out, last = hip.layerLeakyForward(xx, full(n, 0.1), full(n, 0.9), True, True)
        f = hip.layerLifForward(xx, full(n, 0.0), full(n, 0.0), full(n, 0.95), full(n, 0.8), full(n, 1.0), full(n, 1.0),
                                full(n, -1.0), True, -1, True, False)
        return out, last, f["spikes"], f["v_last"], f["i_last"], f["ckpt_v"], f["ckpt_i"]

    big = both(x)
    assert big[2].sum() > 0
    for k in (0, 1, b // 2, b - 1):
        for p, q in zip(big, both(x[k:k + 1].contiguous())):
            assert torch.equal(p[k] if p.ndim == 3 else p[k * m:(k + 1) * m], q[0] if q.ndim == 3 else q)
