"""Whether a layer has a synapse is read off its parameters; the time constant it used to be worked out from agrees."""
import pytest


@pytest.mark.parametrize("train_alphas", [False, True])
@pytest.mark.parametrize("tau_syn", [None, 5.0])
@pytest.mark.parametrize("kind", ["LIF", "ExpLeak", "IAF"])
def test_agrees_with_the_time_constant(kind, tau_syn, train_alphas):
    import sinabs.exodus.layers as el
    if kind == "LIF":
        layer = el.LIF(tau_mem=20.0, tau_syn=tau_syn, train_alphas=train_alphas)
    elif kind == "ExpLeak":
        layer = el.ExpLeak(tau_mem=20.0, train_alphas=train_alphas)
    else:
        layer = el.IAF(tau_syn=tau_syn)
    assert layer._has_synapse() == (layer.tau_syn_calculated is not None)


def test_a_subclass_with_its_own_time_constant_is_asked():
    import sinabs.exodus.layers as el

    class Own(el.LIF):
        @property
        def tau_syn_calculated(self):
            return 3.0
    assert Own(tau_mem=20.0)._has_synapse()
    assert not el.LIF(tau_mem=20.0)._has_synapse()


@pytest.mark.parametrize("tau_syn", [None, 5.0])
def test_refused_where_the_time_constant_is(tau_syn):
    """train_alphas changed by hand: the parameter that would tell is not there."""
    import sinabs.exodus.layers as el
    layer = el.IAF(tau_syn=tau_syn)
    layer.train_alphas = True
    with pytest.raises(AttributeError):
        layer.tau_syn_calculated
    with pytest.raises(AttributeError):
        layer._has_synapse()
