"""The total a layer forward call writes (its blocks' counts, added up by a second kernel) against the sum of what the kernel
wrote: layers whose last wave is partly empty, one neuron, wide lanes, more counts than the summing block has lanes, nothing
at all -- and the entry points that add everything to one double."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 5, 1), (2, 33, 63), (3, 40, 64), (2, 7, 65), (5, 70, 130), (30, 4, 700), (1, 3, 70001), (40, 17, 4098), (64, 9, 8192),
          (3, 2, 600000), (2, 0, 70), (0, 5, 70)]


@pytest.mark.parametrize("b,t,m", SHAPES)
def test_total_is_the_sum_of_the_output(b, t, m):
    from sinabs.exodus import _hip as hip
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(b * 1000 + t + m)
    x = torch.rand(b, t, m, device=dev, generator=g)
    zeros, ones = torch.zeros(b * m, device=dev), torch.ones(b * m, device=dev)
    res = hip.layerLifForward(x, zeros, None, ones, None, ones, ones, None, False, -1, True, False)
    assert res["spike_sum"].shape == () and float(res["spike_sum"]) == float(res["spikes"].sum(dtype=torch.float64))
    one = torch.zeros((), dtype=torch.float64, device=dev)
    ptr = lambda v: v.data_ptr()
    spikes, last = torch.empty_like(x), torch.empty_like(zeros)
    rc = hip.lib.exodus_layer_lif_forward(ptr(spikes), None, None, None, None, ptr(last), None, ptr(one), ptr(x), ptr(zeros),
                                          None, ptr(ones), None, ptr(ones), ptr(ones), None, 0, -1, 1, 0, 0, b, t, m,
                                          torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and float(one) == float(res["spike_sum"]) and torch.equal(spikes, res["spikes"])

    alpha = torch.full_like(ones, 0.9)
    out, _, total = hip.layerLeakyForward(x, zeros, alpha, False, False, wantSum=True)
    want = out.sum(dtype=torch.float64)
    # positive terms: fp32 partial sums over 8 steps of a lane's four neurons at most, float64 beyond
    assert abs(float(total) - float(want)) <= 32 * 2.0 ** -24 * float(want)
