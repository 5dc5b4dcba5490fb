"""Layers on both sides of the rule that gives small layers blocks of one wave: outputs, final states and totals of the forward
and leaky kernels equal those of a call on every batch element alone, and the totals are the sums of the outputs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,t,m,lanes", [
    (1, 3, 1, 64), (3, 40, 63, 64), (3, 40, 64, 64), (3, 40, 65, 64), (2, 33, 257, 64), (5, 7, 1000, 64),
    (8, 40, 4096, 64),        # 512 waves: two per compute unit, the last size with one wave per block
    (8, 40, 4097, 256),       # 520 waves
    (513, 5, 10, 256), (512, 5, 10, 64),
])
def test_small_and_larger_blocks(b, t, m, lanes):
    from sinabs.exodus import _hip as hip
    for kernel in ("forward", "leaky forward", "leaky backward alpha"):
        assert hip.launchShape(kernel, b, m) == (1, lanes)
    g = torch.Generator(device="cuda").manual_seed(b * m)
    x = torch.empty(b, t, m, device="cuda").normal_(0.2, 0.8, generator=g)
    go = torch.empty(b, t, m, device="cuda").normal_(0.0, 1.0, generator=g)
    full = lambda n, v: torch.full((n,), v, device="cuda")

    def every(xx, gg):
        n = xx.shape[0] * m
        out, last, total = hip.layerLeakyForward(xx, full(n, 0.1), full(n, 0.9), True, True, wantSum=True)
        gi, ga, gv = hip.layerLeakyBackward(gg, None, out, xx, full(n, 0.1), full(n, 0.9), True, True, True)
        f = hip.layerLifForward(xx, full(n, 0.0), full(n, 0.0), full(n, 0.95), full(n, 0.8), full(n, 1.0), full(n, 1.0),
                                full(n, -1.0), True, -1, True, False)
        assert float(f["spike_sum"]) == float(f["spikes"].double().sum())
        mass = float(out.double().abs().sum())
        assert abs(float(total) - float(out.double().sum())) <= 32 * 2.0 ** -24 * mass   # fp32 sums of at most 32 outputs
        return out, last, gi, ga, gv, f["spikes"], f["v_last"], f["i_last"], f["ckpt_v"], f["ckpt_i"]

    whole = every(x, go)
    for k in sorted({0, b // 2, b - 1}):
        for p, q in zip(whole, every(x[k:k + 1].contiguous(), go[k:k + 1].contiguous())):
            assert torch.equal(p[k] if p.ndim == 3 else p[k * m:(k + 1) * m], q[0] if q.ndim == 3 else q)


# 258, 1024 and 1040 waves
@pytest.mark.parametrize("b,t,m,lanes", [(2, 40, 8200, 64), (16, 40, 4096, 64), (16, 40, 4097, 256)])
def test_one_lane_backward_with_both_blocks(b, t, m, lanes):
    from sinabs.exodus import _hip as hip
    assert hip.launchShape("backward", b, m) == (1, lanes)
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.empty(b, t, m, device="cuda").normal_(0.2, 0.8, generator=g)
    go = torch.empty(b, t, m, device="cuda").normal_(0.0, 1.0, generator=g)
    full = lambda n, v: torch.full((n,), v, device="cuda")

    def backward(xx, gg):
        n = xx.shape[0] * m
        r = (full(n, 0.0), full(n, 0.0))
        c = (full(n, 0.95), full(n, 0.8), full(n, 1.0), full(n, 1.0), full(n, -1.0), True, -1, True, False)
        f = hip.layerLifForward(xx, *r, *c)
        return hip.layerLifBackward(gg, None, None, xx, f["ckpt_v"], f["ckpt_i"], *r, *c, hip.SURR_SINGLE_EXP, 0.5, 1.0)

    mode = hip.backwardTimeSplit(0)
    try:
        whole = backward(x, go)
        for k in (0, b - 1):
            for p, q in zip(whole, backward(x[k:k + 1].contiguous(), go[k:k + 1].contiguous())):
                assert torch.equal(p[k] if p.ndim == 3 else p[k * m:(k + 1) * m], q[0] if q.ndim == 3 else q)
    finally:
        hip.backwardTimeSplit(mode)
