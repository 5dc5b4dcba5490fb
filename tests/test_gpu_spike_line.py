"""The forward kernel's spike count by one fused multiply-add: potentials on, just below and just above one and two thresholds,
for thresholds of every magnitude and kind, against the comparison and the quotient in numpy float32, bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

F = np.float32


def thresholds():
    rng = np.random.default_rng(1)
    powers = F(2.0) ** np.arange(-100, 101, 7).astype(F)
    free = np.exp2(rng.uniform(-100, 100, 60)).astype(F)
    edge = np.array([2.0 ** -101, 2.0 ** 101, 1e-40, 1e38, 0.0, -0.0, -1.0, np.inf, np.nan, 1.0, 0.1, 3.0], F)
    return np.concatenate([powers, np.nextafter(powers, F(np.inf)), np.nextafter(powers, F(0)), free, edge])


def steps(x, th, c, cap):
    """IAF neurons, (steps, neurons)"""
    v_post, out = np.zeros_like(th), []
    for row in x:
        v = v_post + row
        with np.errstate(all="ignore"):
            q = (v / th).astype(np.float64)
            q = np.where(np.isnan(q), 0.0, np.clip(np.trunc(q), 0.0, 4294967295.0))
            count = np.where(v >= th, np.minimum(q, cap), 0.0).astype(F)
            v_post = v - count * c
        out.append(count)
    return np.stack(out), v_post


@pytest.mark.parametrize("cap", [-1, 0, 1, 2, 5])
@pytest.mark.parametrize("subtract", ["threshold", "half", "infinite", "nan", "huge"])
@pytest.mark.parametrize("t", [1, 16, 40])
def test_potentials_around_the_threshold(cap, subtract, t):
    from sinabs.exodus import _hip as hip
    base = thresholds()
    near = [lambda a: a, lambda a: np.nextafter(a, F(np.inf)), lambda a: np.nextafter(a, F(-np.inf)),
            lambda a: a * F(0.5), lambda a: -a, lambda a: a * F(1.9999999), lambda a: a * F(0)]
    with np.errstate(all="ignore"):
        first = np.concatenate([f(base * F(k)) for k in (1, 2, 3) for f in near] +
                               [np.full_like(base, v) for v in (np.nan, -np.inf, 1e-45, 3e38)])
    th = np.tile(base, len(first) // len(base))
    c = {"threshold": th, "half": th * F(0.5), "infinite": np.full_like(th, np.inf), "nan": np.full_like(th, np.nan),
         "huge": np.full_like(th, 2.0 ** 127)}[subtract].astype(F)
    keep = ~(np.isinf(th) & (np.abs(first) > 1e38))             # infinity over infinity: no quotient
    th, c, first = th[keep], c[keep], first[keep]
    with np.errstate(all="ignore"):
        rest = [first * F(0)] * (t // 2) + [first] * (t - 1 - t // 2)
    x = np.stack([first] + [np.where(np.isnan(r), F(0), r) for r in rest])
    want, last = steps(x, th, c, 4294967295.0 if cap < 0 else float(cap))
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    one = torch.ones(len(th)).cuda()
    f = hip.layerLifForward(d(x)[None], 0 * one, None, one, None, d(c), d(th), None, False, cap, True, False)
    assert np.array_equal(f["spikes"].cpu().numpy()[0], want, equal_nan=True)
    assert np.array_equal(f["v_last"].cpu().numpy(), last, equal_nan=True)
