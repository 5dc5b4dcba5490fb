"""The (rows, time) kernels' driver for short rows (16-byte aligned tensors) against the driver with full address arithmetic (the
same data one element further): every output to the bit, per-row sums within what other groupings of their terms give; nothing
outside a tensor is written."""
import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = [1, 15, 16, 17, 31, 33, 63, 64, 65, 130, 257]


@pytest.mark.parametrize("t", [1, 2, 3, 4, 5, 7, 8, 9, 11, 12, 15, 16, 17, 23, 24, 25, 26, 27, 28, 31, 33, 39, 40, 44, 48, 55, 56, 58, 59,
                               60, 61, 62, 63, 65, 66, 79, 80, 81, 90, 99, 100, 101, 102, 117, 118, 119, 122, 149, 150, 151])
def test_short_rows_on_every_entry_point(t):
    from sinabs.exodus import _hip as hip
    g = torch.Generator().manual_seed(t)
    for case, n in enumerate(ROWS):
        R = lambda *s, sc=1.0, o=0.0: (torch.randn(*s, generator=g) * sc + o).cuda()
        U = lambda lo, hi: (lo + (hi - lo) * torch.rand(n, generator=g)).cuda()
        x, go, gv, gq = R(n, t, sc=0.7, o=0.25), R(n, t), R(n, t, sc=0.1), R(n, t, sc=0.1)
        nc, surr = (R(n, t) > -1.0).float(), R(n, t).abs()
        am, a_s, v0, i0, th = U(0.5, 1.0), U(0.3, 0.9), R(n, sc=0.3), R(n, sc=0.3), U(0.5, 1.5)
        c, lo = th * U(0.4, 1.0), -U(0.2, 1.2)
        use_lo, cap, de, ni = case % 2 == 0, (-1, 1, 2, 3)[case % 4], case % 3 != 0, case % 5 != 0
        low = lo if use_lo else None
        res = []
        for off in (4 * (case % 3), 4 * (case % 3) + 1):
            around = []

            def at(z):
                buf = torch.full((z.numel() + 64,), float("nan"), device="cuda")
                view = buf[off:off + z.numel()].view(z.shape)
                view.copy_(z)
                around.append((buf, z.numel()))
                return view
            zero = torch.zeros(n, t, device="cuda")
            xs, gos, gvs, gqs, ncs, ss = at(x), at(go), at(gv), at(gq), at(nc), at(surr)
            r = {}
            sp, vm = at(zero), at(zero)
            hip.lifForward(sp, vm, xs, v0, am, c, th, low, use_lo, cap)
            r["lif spikes"], r["lif v_mem"] = sp, vm
            for kind, extra in ((hip.SURR_SINGLE_EXP, None), (hip.SURR_PERIODIC_EXP, gvs), (hip.SURR_TENSOR, None),
                                (hip.SURR_TENSOR, gvs)):
                gi = at(zero)
                _, ga, g0 = hip.lifBackwardFused(gos, extra, vm, v0, am, c, th, low, use_lo, cap, kind, 0.5, 1.0, surr=ss,
                                                 needAlphaGrad=True, inputGrad=gi)
                tag = f"lif backward {kind} {extra is not None}"
                r[tag], r[tag + " alpha~"], r[tag + " init"] = gi, ga, g0
            out, gi = at(zero), at(zero)
            hip.leakyForward(xs, v0, am, output=out)
            _, ga, g0 = hip.leakyBackwardFused(gos, am, out, v0, needAlphaGrad=True, inputGrad=gi)
            r["leaky"], r["leaky backward"], r["leaky alpha~"], r["leaky init"] = out, gi, ga, g0
            r["leaky alpha alone~"] = hip.leakyBackwardAlpha(gos, out, v0, am)
            r["lif alpha alone~"] = hip.lifBackwardAlpha(ss, gos, vm, v0, ncs, am, c)
            s2, v2, i2 = at(zero), at(zero), at(zero)
            hip.synLifForward(xs, v0, i0, am, a_s, c, th, low, use_lo, cap, de, ni, out=(s2, v2, i2))
            r["syn spikes"], r["syn v_mem"], r["syn i_syn"] = s2, v2, i2
            for extra in (False, True):
                gi = at(zero)
                rows = hip.synLifBackward(gos, gvs if extra else None, gqs if extra else None, v2, i2, v0, i0, am, a_s, c, th, low,
                                          use_lo, cap, de, ni, hip.SURR_SINGLE_EXP, 0.5, 1.0, inputGrad=gi)
                r[f"syn backward {extra}"] = gi
                for name, z in zip(("alpha_mem~", "alpha_syn~", "v", "i"), rows[1:]):
                    r[f"syn {extra} {name}"] = z
            both = at(x)
            r["spike"], r["spike v"] = hip.spikeForward(both, 0.9, 0.8, 1.0, -0.5, use_lo, cap), both
            res.append(r)
            torch.cuda.synchronize()
            for buf, numel in around:
                assert bool(torch.isnan(buf[:off]).all() and torch.isnan(buf[off + numel:]).all()), (n, t)
        for name, p in res[0].items():
            q = res[1][name]
            if name.endswith("~"):
                # sums over t steps of terms of about 1, in fp32 within at most 32 of them, then in fp64
                assert torch.allclose(p, q, rtol=1e-5, atol=1e-5 * t), (n, t, name)
            else:
                assert torch.equal(p, q), (n, t, name)
