"""A layer keeps per-neuron vectors and passed range checks for as long as its parameters are the same: tensors that are worked out
on access, replaced, or given other memory are not taken for the ones before, whatever addresses the allocators reuse."""
import pickle

import pytest
import torch
from torch.nn.utils import parametrize


class Scaled(torch.nn.Module):
    def forward(self, x):
        return x * 2.0


def layer_with(**kwargs):
    import sinabs.exodus.layers as el
    return el.LIF(**{**dict(tau_mem=20.0), **kwargs})


def vectors(layer, n):
    """(decay factors, thresholds, lower bounds or None) as a call without gradients gets them"""
    shape, dev = (1, n), torch.device("cpu")
    with torch.no_grad():
        stamps = layer._parameter_stamps()
        low = layer.min_v_mem
        return (layer._decay_factor("mem", stamps, shape, dev, False),
                layer._per_neuron("spike_threshold", layer.spike_threshold, stamps[2], shape, dev, False),
                None if low is None else layer._per_neuron("min_v_mem", low, stamps[3], shape, dev, False))


@pytest.mark.parametrize("n", [64, 4096, 65536])
def test_parameters_worked_out_on_access(n):
    layer = layer_with(tau_mem=torch.full((n,), 20.0), spike_threshold=torch.full((n,), 1.0))
    parametrize.register_parametrization(layer, "tau_mem", Scaled())
    parametrize.register_parametrization(layer, "spike_threshold", Scaled())
    for k in range(100):
        with torch.no_grad():
            layer.parametrizations.tau_mem.original.fill_(5.0 + k)
            layer.parametrizations.spike_threshold.original.fill_(1.0 + k)
        alpha, theta, _ = vectors(layer, n)
        assert torch.equal(alpha, torch.exp(-1.0 / torch.full((n,), 2.0 * (5.0 + k)))), k
        assert torch.equal(theta, torch.full((n,), 2.0 * (1.0 + k))), k


@pytest.mark.parametrize("n", [1, 64])
def test_stored_tensor_freed_and_replaced(n):
    layer = layer_with()
    for k in range(100):
        layer.min_v_mem = torch.full((1,), -1.0 - k)
        assert torch.equal(vectors(layer, n)[2], torch.full((n,), -1.0 - k)), k
        layer.min_v_mem = None


def test_parameter_given_other_memory():
    layer = layer_with()
    for k in range(100):
        layer.spike_threshold.data = torch.full((1,), 1.0 + k)
        assert torch.equal(vectors(layer, 8)[1], torch.full((8,), 1.0 + k)), k
        layer.spike_threshold.data = torch.zeros(3)


def test_attribute_found_by_a_rule_of_the_class():
    import sinabs.exodus.layers as el

    class Shared(el.LIF):
        settings = {"min_v_mem": -1.0}

        def __getattr__(self, name):
            return self.settings[name] if name in self.settings else super().__getattr__(name)

    layer = Shared(tau_mem=20.0)
    del layer.min_v_mem
    for low in (-1.0, -2.0, -3.0):
        layer.settings["min_v_mem"] = low
        assert torch.equal(vectors(layer, 8)[2], torch.full((8,), low))


@pytest.mark.parametrize("kind", ["LIF", "IAF"])
def test_decay_factor_by_a_rule_of_the_class(kind):
    import sinabs.exodus.layers as el

    class Own(getattr(el, kind)):
        @property
        def alpha_mem_calculated(self):
            return torch.sigmoid(self.w)

    layer = Own(**dict(tau_mem=20.0) if kind == "LIF" else {})
    layer.w = torch.nn.Parameter(torch.zeros(()))
    shape, dev = (1, 8), torch.device("cpu")
    seen = []
    for w in (0.0, 1.0, 2.0):
        with torch.no_grad():
            layer.w.fill_(w)
            stamps = layer._parameter_stamps()
            assert not any(stamps is s for s in seen)          # the range check is not skipped
            seen.append(stamps)
            assert torch.equal(layer._decay_factor("mem", stamps, shape, dev, False), torch.sigmoid(torch.full((8,), w)))
    layer._decay_factor("mem", layer._parameter_stamps(), shape, dev, False).sum().backward()
    assert layer.w.grad is not None and layer.w.grad != 0


def test_kept_while_nothing_changes_and_not_in_copies():
    layer = layer_with(min_v_mem=-1.0)
    first = vectors(layer, 8)
    assert all(a is b for a, b in zip(first, vectors(layer, 8)))
    stamps = layer._parameter_stamps()
    assert layer._parameter_stamps() is stamps
    with torch.no_grad():
        layer.tau_mem.mul_(2.0)
    second = vectors(layer, 8)
    assert second[0] is not first[0] and second[1] is first[1] and second[2] is first[2]
    other = pickle.loads(pickle.dumps(layer))
    assert other._kept.stamps is None and not other._kept.vectors
    assert torch.equal(vectors(other, 8)[0], second[0])


@pytest.mark.parametrize("before,after,same", [(1.0, 1.0, True), (1, 1.0, True), (float("nan"), float("nan"), True),
                                               (0.0, -0.0, False), (1.0, 2.0, False), (None, None, True), (None, 0.0, False)])
def test_numbers_by_their_bits(before, after, same):
    from sinabs.exodus import _hip
    kept = _hip.stamps(None, (before, 7.0))
    again = _hip.stamps(kept, (after, 7.0))
    assert (again is kept) == same and again[1] is kept[1]


def test_what_is_no_number_is_never_the_same():
    from sinabs.exodus import _hip
    value = object()
    kept = _hip.stamps(None, (value,))
    assert _hip.stamps(kept, (value,))[0] is not kept[0]


@pytest.mark.gpu
def test_the_range_check_sees_every_change():
    layer = layer_with(spike_threshold=torch.full((50,), 1.0), min_v_mem=0.0).cuda()
    parametrize.register_parametrization(layer, "spike_threshold", Scaled())
    x = torch.rand(2, 5, 50).cuda()
    with torch.no_grad():
        for k in range(20):
            layer.parametrizations.spike_threshold.original.fill_(1.0)
            layer(x)
            layer.parametrizations.spike_threshold.original.fill_(-1.0)
            with pytest.raises(ValueError, match="greater than"):
                layer(x)


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["tau_mem", "tau_syn"])
def test_gradient_of_a_parametrized_time_constant(which):
    """Also where nothing else asks for one: an input without a gradient, no trained parameter of the layer's own."""
    x = torch.rand(3, 20, 40).cuda()
    grads = []
    for parametrized in (False, True):
        layer = layer_with(tau_mem=20.0, tau_syn=10.0).cuda().requires_grad_(False)
        if parametrized:
            parametrize.register_parametrization(layer, which, Scaled())
            wanted = layer.parametrizations[which].original
            with torch.no_grad():
                wanted.mul_(0.5)
        else:
            wanted = getattr(layer, which)
        wanted.requires_grad_(True)
        layer(x).square().sum().backward()
        grads.append(wanted.grad)
    # the chain rule's factor of two is exact; the two gradients add the neurons up in another order
    assert grads[0].abs() > 0 and torch.allclose(grads[1], 2.0 * grads[0], rtol=1e-5)
