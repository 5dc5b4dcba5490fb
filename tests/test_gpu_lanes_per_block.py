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

    mode = hip.backwardTimeSplit(0)                            # the kernels that the rule is for
    try:
        whole = every(x, go)
        for k in sorted({0, b // 2, b - 1}):
            for p, q in zip(whole, every(x[k:k + 1].contiguous(), go[k:k + 1].contiguous())):
                assert torch.equal(p[k] if p.ndim == 3 else p[k * m:(k + 1) * m], q[0] if q.ndim == 3 else q)
    finally:
        hip.backwardTimeSplit(mode)


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


# lanes per block of the forward that records both states, of the backward, and of the backward with gradients on state records or
# a surrogate tensor
@pytest.mark.parametrize("b,t,m,records,plain,more", [
    (6, 40, 4090, 64, 64, 64),                # 384 waves, sectors shared between blocks: the last for the recording forward
    (7, 40, 4090, 256, 64, 64),               # 448
    (8, 40, 4096, 64, 64, 64),                # 512, whole sectors
    (500, 5, 40, 64, 64, 64),                 # one wave per element: no neighbours
    (12, 40, 4090, 256, 64, 64),              # 768: the last for the backward with more tensors
    (13, 40, 4090, 256, 64, 256),             # 832
    (16, 40, 4090, 256, 64, 256),             # 1024
    (16, 40, 4096, 256, 64, 64),              # 1024, whole sectors: the last for the backward
    (16, 40, 4112, 256, 256, 256),            # 1040, whole sectors
])
def test_blocks_of_calls_with_more_tensors(b, t, m, records, plain, more):
    from sinabs.exodus import _hip as hip
    names = ("forward records", "backward", "backward more")
    assert tuple(hip.launchShape(k, b, m)[1] for k in names) == (records, plain, more)
    g = torch.Generator(device="cuda").manual_seed(b * m)
    x, go, gv, gi = (torch.empty(b, t, m, device="cuda").normal_(0.2, 0.8, generator=g) for _ in range(4))
    surr = torch.rand(b, t, m, device="cuda", generator=g)
    full = lambda n, v: torch.full((n,), v, device="cuda")

    def every(s):
        xx, n = x[s].contiguous(), x[s].shape[0] * m
        const = lambda i0, a_s: (full(n, 0.0), i0, full(n, 0.95), a_s, full(n, 1.0), full(n, 1.0), full(n, -1.0), True, -1, True, False)
        f = hip.layerLifForward(xx, *const(full(n, 0.0), full(n, 0.8)), wantRecords=True)
        assert float(f["spike_sum"]) == float(f["spikes"].double().sum())
        outs = [f[k] for k in ("spikes", "v_last", "i_last", "v_rec", "i_rec")]
        states = dict(gradVRec=gv[s].contiguous(), gradIRec=gi[s].contiguous())
        for syn_too, kind, more_grads in ((False, 1, {}), (True, 1, {}), (True, 1, states), (False, 0, dict(surr=surr[s].contiguous()))):
            c = const(full(n, 0.0), full(n, 0.8)) if syn_too else const(None, None)
            f = hip.layerLifForward(xx, *c)
            grads = hip.layerLifBackward(go[s].contiguous(), None, None, xx, f["ckpt_v"], f["ckpt_i"], *c, kind, 0.5, 1.0, **more_grads)
            outs += [r for r in grads if r is not None]
        return outs

    mode = hip.backwardTimeSplit(0)
    try:
        whole = every(slice(0, b))
        for k in sorted({0, b - 1}):
            for p, q in zip(whole, every(slice(k, k + 1))):
                assert torch.equal(p[k] if p.ndim == 3 else p[k * m:(k + 1) * m], q[0] if q.ndim == 3 else q)
    finally:
        hip.backwardTimeSplit(mode)
