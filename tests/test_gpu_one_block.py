"""A chunk of one sample in a single block, which writes the total itself: outputs, states, checkpoints to the bit as in a batch of
two, the total the sum of the output; on both sides of the limits in neurons (1024), steps (32) and their product (12288)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [1, 10, 12, 13, 16, 17, 31, 32, 33, 70])
@pytest.mark.parametrize("m", [1, 63, 64, 65, 256, 257, 384, 385, 1023, 1024, 1025])
def test_one_sample_as_in_a_batch(t, m):
    from sinabs.exodus import _hip as hip
    g = torch.Generator(device="cuda").manual_seed(t * 2000 + m)
    x = torch.empty(1, t, m, device="cuda").normal_(0.4, 1.0, generator=g)
    v0, i0 = (torch.randn(m, generator=g, device="cuda") * 0.3 for _ in range(2))
    full = lambda n, v: torch.full((n,), v, device="cuda")
    for syn, cap, low in ((False, -1, False), (True, 1, True), (True, 2, False), (False, 1, True), (False, 2, True), (True, -1, True)):
        def call(k):
            n = k * m
            return hip.layerLifForward(x.repeat(k, 1, 1), v0.repeat(k), i0.repeat(k) if syn else None, full(n, 0.9),
                                       full(n, 0.8) if syn else None, full(n, 1.0), full(n, 1.0), full(n, -0.3) if low else None, low,
                                       cap, True, False)
        one, two = call(1), call(2)
        for name in ("spikes", "v_last", "i_last", "ckpt_v", "ckpt_i"):
            p, q = one[name], two[name]
            assert p is None if q is None else torch.equal(p.flatten(), q.flatten()[:p.numel()]), name
        assert float(one["spike_sum"]) == float(one["spikes"].double().sum()) == float(two["spike_sum"]) / 2
    one, two = (hip.layerLeakyForward(x.repeat(k, 1, 1), v0.repeat(k), full(k * m, 0.9), True, True, wantSum=True) for k in (1, 2))
    assert torch.equal(one[0][0], two[0][1]) and torch.equal(one[1], two[1][:m])
    total, mass = float(one[0].double().sum()), float(one[0].double().abs().sum())
    assert abs(float(one[2]) - total) <= 16 * 2.0 ** -24 * mass     # fp32 sums of the outputs of 8 steps, then fp64
