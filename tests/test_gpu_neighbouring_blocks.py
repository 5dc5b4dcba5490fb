"""Layers whose steps share lines of memory between blocks: their blocks are dealt out to the XCDs in runs, which must leave no
block out and do none twice.  Everything a call writes equals what calls on the batch elements alone write (grids of a few
blocks, which stay as they are), for grids on both sides of every length of a run."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# blocks of the forward kernels: 2, 14 and 16 (runs of 1 and 2), 18 (two left over), 200, 202 (25) and 300 (37, four left over); in
# blocks of four waves 510 (63), 512 and 600 (32, 88 left over); two and four neurons per lane; half lines shared, and none.  More
# than 32 steps of at most one block per compute unit are another kernel's in the forward without records: 30 steps there
@pytest.mark.parametrize("b,t,m", [
    (1, 3, 65), (7, 3, 65), (8, 3, 65), (9, 30, 65), (9, 35, 65), (100, 3, 65), (101, 30, 65),
    (101, 33, 65), (150, 35, 65),
    (255, 3, 300), (256, 3, 300), (300, 30, 300), (5, 2, 110002), (5, 3, 1048580), (300, 3, 272), (300, 3, 288),
])
@pytest.mark.parametrize("syn,records", [(False, False), (True, True)])
def test_runs_of_blocks(b, t, m, syn, records):
    from sinabs.exodus import _hip as hip
    g = torch.Generator(device="cuda").manual_seed(b * m)
    x = torch.empty(b, t, m, device="cuda").normal_(0.2, 0.8, generator=g)
    go = torch.empty(b, t, m, device="cuda").normal_(0.0, 1.0, generator=g)
    a = 0.9 + 0.09 * torch.rand(m, generator=g, device="cuda")

    def every(xx, gg):
        n = xx.shape[0] * m
        full = lambda v: torch.full((n,), v, device="cuda")
        am = a.repeat(xx.shape[0])
        out, last, total = hip.layerLeakyForward(xx, full(0.1), am, True, True, wantSum=True)
        leaky = hip.layerLeakyBackward(gg, None, out, xx, full(0.1), am, True, True, True)
        plain = hip.layerLeakyBackward(gg, None, None, None, None, am, False, False, False)
        states = (full(0.0), full(0.0) if syn else None)
        consts = (am, full(0.8) if syn else None, full(1.0), full(1.0), full(-1.0), True, -1, True, False)
        f = hip.layerLifForward(xx, *states, *consts, wantRecords=records)
        assert float(f["spike_sum"]) == float(f["spikes"].double().sum())
        more = dict(gradVRec=gg, gradIRec=gg if syn else None) if records else {}
        lif = hip.layerLifBackward(gg, None, None, xx, f["ckpt_v"], f["ckpt_i"], *states, *consts, hip.SURR_SINGLE_EXP, 0.5, 1.0,
                                   **more)
        return [z for z in (out, last, *leaky, *plain, f["spikes"], f["v_last"], f["i_last"], f["v_rec"], f["i_rec"], f["ckpt_v"],
                            *lif) if z is not None]

    mode = hip.backwardTimeSplit(0)                            # the kernel that every width can have
    try:
        whole = every(x, go)
        for k in sorted({0, b // 3, b - 2, b - 1} & set(range(b))):
            for p, q in zip(whole, every(x[k:k + 1].contiguous(), go[k:k + 1].contiguous())):
                assert torch.equal(p[k] if p.ndim == 3 else p[k * m:(k + 1) * m], q[0] if q.ndim == 3 else q)
    finally:
        hip.backwardTimeSplit(mode)
