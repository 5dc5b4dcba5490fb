"""The range checks in one kernel: one bad value anywhere in a vector is found, in the call that carries it, and the values
on the edge, infinities and NaN are judged as torch's comparisons judge them."""
import pytest
import torch

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")


def flags(alphas, theta=None, low=None):
    from sinabs.exodus import _hip as hip
    host = torch.zeros(2, dtype=torch.int32, pin_memory=True)
    hip.checkParameters(host, alphas[0], alphas[1] if len(alphas) > 1 else None, theta, low)
    torch.cuda.synchronize()
    return host.tolist()


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 257, 1023, 1024, 1025, 131072, 524288, 524289, 1300001])
def test_one_bad_value_anywhere(n):
    good = torch.full((n,), 0.5, device="cuda")
    th, lo = torch.ones(n, device="cuda"), torch.zeros(n, device="cuda")
    assert flags([good], th, lo) == [0, 0] and flags([good, good]) == [0, 0]
    for at in sorted({0, n // 3, n // 2, n - 1}):
        bad = good.clone()
        bad[at] = 1.5
        lo_bad = lo.clone()
        lo_bad[at] = 1.0
        assert flags([bad], th, lo) == [1, 0] and flags([good, bad]) == [1, 0]
        assert flags([good], th, lo_bad) == [0, 1] and flags([bad, good], th, lo_bad) == [1, 1]


@pytest.mark.parametrize("value", [0.0, -0.0, 1.0, -1e-45, 1.0000001, INF, -INF, NAN])
def test_edges_as_torch_compares(value):
    a = torch.full((70,), 0.5, device="cuda")
    a[69] = value
    one = torch.ones_like(a)
    want = [int(((a < 0) | (a > 1)).any()), int((one <= a).any())]
    assert flags([a], one, a) == want


def test_the_call_that_carries_the_value_raises():
    from oracle import exodus_ref as ref
    from sinabs.exodus.spike import IntegrateAndFire
    x, one = torch.rand(300, 10).cuda(), torch.ones(300).cuda()
    bad = one * 0.9
    bad[299] = -0.1
    for _ in range(3):
        IntegrateAndFire.apply(x, one * 0.9, one * 0, one, None, -one, ref.Heaviside())
        with pytest.raises(ValueError, match="between 0 and 1"):
            IntegrateAndFire.apply(x, bad, one * 0, one, None, None, ref.Heaviside())
        with pytest.raises(ValueError, match="greater than"):
            IntegrateAndFire.apply(x, one * 0.9, one * 0, one, None, one, ref.Heaviside())


@pytest.mark.parametrize("mode", ["sync", "deferred"])
@pytest.mark.parametrize("one_kernel", [True, False])
def test_flags_are_host_memory_whatever_the_default_device(mode, one_kernel):
    from sinabs.exodus import _validate as val
    n = 40
    low = torch.zeros(n if one_kernel else 1, device="cuda")           # broadcast: checked by torch's operations
    good, bad, one = (torch.full((n,), v, device="cuda") for v in (0.5, 1.5, 1.0))
    val.set_mode(mode)
    try:
        with torch.device("cuda"):
            val.check_parameters([good], one, low)
            val.flush()
            with pytest.raises(ValueError, match="between 0 and 1"):
                val.check_parameters([bad], one, low)
                val.flush()
    finally:
        val.set_mode("sync")


@pytest.mark.parametrize("kind", ["LIF", "IAF"])
def test_layers_under_a_default_device(kind):
    import sinabs.exodus.layers as el
    x = torch.rand(2, 10, 30).cuda()
    layer = getattr(el, kind)(**dict(tau_mem=20.0) if kind == "LIF" else {}).cuda()
    want = layer(x)
    with torch.device("cuda"):
        layer = getattr(el, kind)(**dict(tau_mem=20.0) if kind == "LIF" else {})
        assert torch.equal(layer(x), want)
        with torch.no_grad():
            layer.spike_threshold.fill_(1.0)
            layer.reset_states()
            assert torch.equal(layer(x), want)
