"""brunel_with_plasticity's traces kept per neuron (its synapses' traces are the same for all plastic
synapses of a source, or of a target): windows with eager events, against the checker's dense
per-step plasticity; and the nets that go back to the per-synapse contract -- a layout whose
plastic synapses target Poisson neurons, imported synapse state that is not of that form --, alone
and in a batch. Weights as in the lazy contract's test (exp() differs by a few ulp between the
host's and the device's library: 3 steps' roundings per step); where the traces are per neuron
their per-step recurrence has the checker's roundings, so they are equal bit for bit."""
import numpy as np
import pytest

from oracle import oracle as O
from spice_amd import Batch, Layout, Snn
from tests.helpers import assert_state_close, assert_state_equal, brunel_ref_layout

pytestmark = pytest.mark.gpu

MODEL, DT = "brunel_with_plasticity", 1e-4


def _pair(lay, delay, seed=5):
    return O.CpuSnn(MODEL, lay, DT, delay, seed=seed, fixed_point=True), Snn(MODEL, Layout(*lay), DT, delay, seed=seed, fixed_point=True)


def _check(d, h, steps, traces_equal, what):
    assert_state_close(d.neurons(), h.neurons(), 1e-5, 1e-9, what)
    a, b = d.synapses(ell=False), h.synapses(ell=False)
    for k in b:
        if traces_equal and k != "W":
            np.testing.assert_array_equal(a[k].view(np.uint32), b[k].view(np.uint32), err_msg=f"{what} {k}")
        else:
            np.testing.assert_allclose(a[k], b[k], rtol=3 * steps * 2.0 ** -24, atol=1e-9, err_msg=f"{what} {k}")


@pytest.mark.parametrize("delay", [1, 2, 15])
def test_windows_match_dense(gpu, delay):
    h, d = _pair(brunel_ref_layout(1200), delay)
    done = 0
    for n in (200, 1, 10, 11, 89, 500):  # past 920 silent steps a weight can move
        d.run(n)
        h.run(n)
        done += n
        _check(d, h, done, True, f"after {done} steps")
    np.testing.assert_array_equal(np.sort(d.step(True)), np.sort(h.step(True)))
    d.close(), h.close()


def test_weights_move_with_the_traces(gpu):
    """Small imported traces (as after a long silence) make the events move the weights."""
    h, d = _pair(brunel_ref_layout(1000), 8)
    z = h.synapses(ell=False)
    src = np.repeat(np.arange(1000), np.diff(h.csr()[0]))
    dst = h.csr()[1]
    plastic = (src >= 500) & (src < 900) & (dst < 900)
    z["Zpre"] = np.where(plastic, np.float32(1e-4) * (1 + src % 7), 1.0).astype(np.float32)
    z["Zpost"] = np.where(plastic, np.float32(2e-4) * (1 + dst % 5), 1.0).astype(np.float32)
    for net in (h, d):
        net.set_synapses(z, ell=False)
    w0 = z["W"].copy()
    for n in (30, 70, 50):
        d.run(n)
        h.run(n)
    _check(d, h, 150, True, "after 150 steps")
    assert np.mean(d.synapses(ell=False)["W"] != w0) > 0.01
    # moving the clock drops the spikes in flight and keeps the synapses, traces included: as a
    # converted copy of the network that is given the same clock
    c = Snn.from_net(d, seed=5, fixed_point=True)
    before = d.synapses(ell=False)
    for net in (c, d):
        net.set_clock(1000, 0.1, 0.0)
    assert_state_equal(d.synapses(ell=False), before, "the clock moved")
    c.run(77), d.run(77)
    assert_state_equal(c.neurons(), d.neurons(), "after the clock moved")
    assert_state_equal(c.synapses(ell=False), d.synapses(ell=False), "after the clock moved")
    d.close(), h.close()


@pytest.mark.parametrize("case", ["poisson_targets", "trace", "non_plastic_trace", "weight"])
@pytest.mark.parametrize("batched", [False, True])
def test_back_to_the_per_synapse_contract(gpu, case, batched):
    lay = ([1000], [(0, 0, 0.1)]) if case == "poisson_targets" else brunel_ref_layout(1000)
    h = O.CpuSnn(MODEL, lay, DT, 6, seed=9, fixed_point=True)
    if batched:
        b = Batch(MODEL, [(Layout(*brunel_ref_layout(800)), 6, 4), (Layout(*lay), 6, 9)], DT, fixed_point=True)
        run, d = b.run, b.net(1)
    else:
        d = Snn(MODEL, Layout(*lay), DT, 6, seed=9, fixed_point=True)
        run = d.run
    run(130)
    h.run(130)
    _check(d, h, 130, False, "before the import")
    if case != "poisson_targets":
        z = h.synapses(ell=False)
        rp, dst = h.csr()
        src = np.repeat(np.arange(1000), np.diff(rp))
        plastic = (src >= 500) & (src < 900) & (dst < 900)
        e = np.flatnonzero(plastic if case != "non_plastic_trace" else ~plastic)[::3]
        if case == "weight":
            z["W"][e] = 0.001  # above the bound that the next step clamps to
        else:
            z["Zpost"][e] = 0.003
        d.set_synapses(z, ell=False)
        h.set_synapses(z, ell=False)
        got = d.synapses(ell=False)
        for k in z:
            np.testing.assert_array_equal(got[k], z[k], err_msg=k)
    for n in (40, 1, 260):
        run(n)
        h.run(n)
    if case == "non_plastic_trace":  # (the checker's dense plasticity leaves them alone, too)
        np.testing.assert_array_equal(d.synapses(ell=False)["Zpost"][e], np.float32(0.003))
    _check(d, h, 431, False, "after the import")
    if batched:
        alone = Snn(MODEL, Layout(*brunel_ref_layout(800)), DT, 6, seed=4, fixed_point=True)
        alone.run(431)
        assert_state_close(b.net(0).neurons(), alone.neurons(), 1e-5, 1e-9, "the batch's other net")
    h.close()


def test_factored_state_survives_conversion(gpu):
    h, d = _pair(brunel_ref_layout(900), 15)
    d.run(333), h.run(333)
    c = Snn.from_net(d, seed=5, fixed_point=True)
    assert_state_equal(c.synapses(ell=False), d.synapses(ell=False), "converted synapses")
    assert_state_equal(c.neurons(), d.neurons(), "converted neurons")
    x = Snn.from_net(h, seed=5, fixed_point=True)
    c.run(50), x.run(50)
    assert_state_close(c.neurons(), x.neurons(), 1e-5, 1e-9, "both conversions run on")
