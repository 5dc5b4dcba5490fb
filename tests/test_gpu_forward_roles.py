"""The forward kernel for small layers (a few waves share the work on 64 neurons) against the kernel of larger layers, to the bit:
a batch element alone gets the first, the same element among many gets the second."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def both(t, m, syn, cap, low, theta=1.0, c=None, poke=None, scale=1.0, decay_early=True, norm=True, elements=2, seed=0):
    from sinabs.exodus import _hip as hip
    many = 4 * torch.cuda.get_device_properties(0).multi_processor_count // max(1, m // 64) + 1
    g = torch.Generator(device="cuda").manual_seed(t * 1000 + m + seed)
    few = torch.empty(elements, t, m, device="cuda").normal_(0.3, 1.0, generator=g) * scale
    if poke is not None:
        poke(few)
    x = torch.cat([few, few[:1].expand(many, -1, -1)])
    a = 0.8 + 0.19 * torch.rand(m, generator=g, device="cuda")
    v0, i0 = (torch.randn(m, generator=g, device="cuda") * 0.3 for _ in range(2))

    def call(xx):
        n, k = xx.shape[0] * m, xx.shape[0]
        full = lambda v: torch.full((n,), v, device="cuda")
        return hip.layerLifForward(xx, v0.repeat(k), i0.repeat(k) if syn else None, a.repeat(k), full(0.8) if syn else None,
                                   full(theta if c is None else c), full(theta), full(-0.4) if low else None, low, cap,
                                   decay_early, norm)
    got, want = call(few), call(x)
    for name in ("spikes", "ckpt_v", "ckpt_i", "v_last", "i_last"):
        p, q = got[name], want[name]
        if p is None:
            assert q is None
            continue
        q = q[:elements] if q.ndim == 3 else q[:elements * m]
        assert p.shape == q.shape
        assert torch.equal(torch.nan_to_num(p, nan=7e30), torch.nan_to_num(q, nan=7e30)), name
    total = float(got["spikes"].double().sum())
    # the counts of 16 steps are added up in 32 bits: exact unless a count is beyond 2^20, as the quotients by tiny thresholds are
    assert abs(float(got["spike_sum"]) - total) <= (16 * 2.0 ** -24 * total if float(got["spikes"].max()) > 2 ** 20 else 0)
    return got


@pytest.mark.parametrize("t", [33, 47, 48, 49, 63, 64, 65, 80, 111, 112, 200])
@pytest.mark.parametrize("m", [1, 63, 64, 65, 200])
def test_ends_of_stages_and_blocks(t, m):
    for syn in (False, True):
        got = both(t, m, syn, -1, True, norm=False)
        assert float(got["spike_sum"]) > 0


@pytest.mark.parametrize("syn", [False, True])
@pytest.mark.parametrize("low", [False, True])
@pytest.mark.parametrize("cap", [-1, 0, 1, 2, 3])
def test_caps_and_potentials_beyond_two_thresholds(syn, low, cap):
    for scale in (1.0, 4.0, 40.0):                             # a double spike now and then, often, always
        both(150, 70, syn, cap, low, scale=scale, norm=False, decay_early=scale != 4.0)


@pytest.mark.parametrize("syn", [False, True])
def test_thresholds_and_values_that_the_short_count_does_not_cover(syn):
    def poke(x):
        x[0, 20, 3] = float("nan")
        x[0, 21, 4] = float("inf")
        x[1, 40, 5] = -float("inf")
        x[1, 70, 6] = 3e38
    for kw in (dict(poke=poke), dict(poke=poke, theta=-0.5), dict(theta=0.0), dict(theta=1e-35), dict(theta=3e37),
               dict(c=float("inf")), dict(c=0.0), dict(theta=0.7, c=0.9)):
        for cap in (-1, 1, 2):
            both(100, 40, syn, cap, True, **kw)


def test_the_last_size_and_the_first_beyond():
    from sinabs.exodus import _hip as hip
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    full = lambda n, v: torch.full((n,), v, device="cuda")
    for blocks in (cus, cus + 1):
        x = torch.randn(blocks, 40, 64, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda") + 0.2

        def call(xx):
            n = xx.shape[0] * 64
            return hip.layerLifForward(xx, full(n, 0.0), None, full(n, 0.9), None, full(n, 1.0), full(n, 1.0), None, False, -1, True, True)
        whole = call(x)
        for k in (0, blocks - 1):
            alone = call(x[k:k + 1].contiguous())
            assert torch.equal(alone["spikes"][0], whole["spikes"][k]) and torch.equal(alone["v_last"], whole["v_last"][k * 64:(k + 1) * 64])
        assert float(whole["spike_sum"]) == float(whole["spikes"].sum())


def test_without_checkpoints_and_into_one_total():
    """The entry point that adds to a total of the caller's, and a call whose backward pass is not wanted."""
    import ctypes
    from sinabs.exodus import _hip as hip
    b, t, m = 3, 70, 100
    n = b * m
    x = torch.randn(b, t, m, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda") + 0.2
    one, zero, a = torch.ones(n, device="cuda"), torch.zeros(n, device="cuda"), torch.full((n,), 0.9, device="cuda")
    want = hip.layerLifForward(x, zero, None, a, None, one, one, None, False, -1, True, True, wantCheckpoints=False)
    assert want["ckpt_v"] is None
    spikes, v_last, total = torch.empty_like(x), torch.empty(n, device="cuda"), torch.full((), 5.0, dtype=torch.float64, device="cuda")
    P = lambda z: None if z is None else ctypes.c_void_p(z.data_ptr())
    rc = hip.lib.exodus_layer_lif_forward(P(spikes), None, None, None, None, P(v_last), None, P(total), P(x), P(zero), None, P(a), None,
                                          P(one), P(one), None, 0, -1, 1, 1, 0, b, t, m,
                                          ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    assert torch.equal(spikes, want["spikes"]) and torch.equal(v_last, want["v_last"])
    assert float(total) == 5.0 + float(want["spikes"].double().sum())
