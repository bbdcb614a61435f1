"""What a network keeps when its clock, its statistics or its launch shapes are changed between
runs."""
import numpy as np
import pytest

from oracle import oracle as O
from spice_amd import Batch, Layout, Snn
from tests.helpers import assert_state_equal, brunel_ref_layout, three_pop_layout

pytestmark = pytest.mark.gpu

DT = 1e-4


def _start(model, layout, delay, seed):
    """A network that is active from the first step on."""
    d = Snn(model, Layout(*layout), DT, delay, seed=seed, fixed_point=True)
    rng = np.random.default_rng(seed)
    n = sum(layout[0])
    s = d.neurons()
    s["V"] = rng.uniform(0.0, 0.025, n).astype(np.float32)
    d.set_neurons(s)
    if model == "brunel_with_plasticity":  # traces as after a long silence: events move the weights
        z = d.synapses(ell=False)
        rp, dst = d.csr()
        src = np.repeat(np.arange(n), np.diff(rp))
        plastic = (src >= n // 2) & (src < 9 * n // 10) & (dst < 9 * n // 10)
        for k in ("Zpre", "Zpost"):
            z[k] = np.where(plastic, np.float32(1e-4), np.float32(1.0))
        d.set_synapses(z, ell=False)
    return d


PLASTIC = [
    ("brunel_3pop_stdp", three_pop_layout(1500), 15),
    ("brunel_3pop_stdp", three_pop_layout(1500), 1),
    ("brunel_3pop_stdp_deferred", three_pop_layout(1500), 4),
    ("brunel_with_plasticity", brunel_ref_layout(1200), 9),
    ("brunel_with_plasticity", ([300, 900], [(0, 0, 0.05), (1, 0, 0.05), (1, 1, 0.05)]), 9),  # per-synapse contract
]


@pytest.mark.parametrize("model,layout,delay", PLASTIC)
@pytest.mark.parametrize("step", [0, 77])
def test_set_clock_keeps_the_plasticity_of_all_steps(gpu, model, layout, delay, step):
    """The synapses after set_clock() are those of the steps run before it, the last window's too."""
    a, b = _start(model, layout, delay, 3), _start(model, layout, delay, 3)
    before = a.synapses(ell=False)
    for net in (a, b):
        net.run(27)
    want = a.synapses(ell=False)
    assert not np.array_equal(before["W"], want["W"])
    b.set_clock(step, step * DT, 0.0)
    got = b.synapses(ell=False)
    for k in want:
        np.testing.assert_array_equal(got[k].view(np.uint32), want[k].view(np.uint32), err_msg=k)
    a.close(), b.close()


@pytest.mark.parametrize("model,layout,delay", PLASTIC)
def test_reset_stats_counts_from_here(gpu, model, layout, delay):
    """What earlier steps left to do is not counted after reset_stats()."""
    d = _start(model, layout, delay, 4)
    d.run(27)
    d.reset_stats()
    st = d.stats()
    assert all(v == 0 for v in st.values()), st
    d.close()


def test_a_smaller_network_leaves_a_larger_one_its_lds(gpu):
    """Both run the same kernel, at 144 KB (tiles of 1,024, 15 steps) and 76 KB (of 512) of LDS, and
    the larger one was made first."""
    lay, delay = three_pop_layout(3000), 15
    h = O.CpuSnn("brunel_3pop", lay, DT, delay, seed=8, fixed_point=True)
    large, small = (Snn("brunel_3pop", Layout(*lay), DT, delay, seed=8, fixed_point=True) for _ in range(2))
    large.set_launch(tile_w=1024, recv_block=1024)
    large.run(30)
    small.set_launch(tile_w=512, recv_block=1024)
    small.run(30)
    large.run(45)
    h.run(75)
    assert_state_equal(large.neurons(), h.neurons(), "the larger")
    small.run(45)
    assert_state_equal(small.neurons(), h.neurons(), "the smaller")
    large.close(), small.close(), h.close()


def test_launch_shapes_that_do_not_fit_leave_the_old_ones(gpu):
    """Tiles of 64 of 2.5 million neurons: 390 GB for the offsets of every row and tile. The network
    goes on with the shapes, counters and results that it had."""
    lay, delay = ([2500000], [(0, 0, 2e-6)]), 1
    h = O.CpuSnn("synth", lay, DT, delay, seed=9, fixed_point=True)
    d = Snn("synth", Layout(*lay), DT, delay, seed=9, fixed_point=True)
    for net in (h, d):
        net.run(9)
    before, stats = d.launch(), d.stats()
    with pytest.raises(MemoryError):
        d.set_launch(tile_w=64)
    assert d.launch() == before and d.stats() == stats
    for net in (h, d):
        net.run(6)
    assert_state_equal(d.neurons(), h.neurons(), "after the refused shapes")
    np.testing.assert_array_equal(np.sort(d.step(True)), np.sort(h.step(True)))
    d.set_launch(tile_w=2048)
    for net in (h, d):
        net.run(6)
        net.step()
    assert_state_equal(d.neurons(), h.neurons(), "after other shapes")
    d.close(), h.close()


def _fill(fill, room):
    """Takes the card's memory but `room` MB (the runtime may find some 200 more)."""
    import torch
    while torch.cuda.mem_get_info()[0] > (room << 20) + (16 << 30):
        fill.append(torch.empty(16 << 30, dtype=torch.uint8, device="cuda"))
    left = torch.cuda.mem_get_info()[0] - (room << 20)
    fill.append(torch.empty(left >> 21 << 21, dtype=torch.uint8, device="cuda"))
    if abs(torch.cuda.mem_get_info()[0] - (room << 20)) > 24 << 20:
        pytest.skip("the card's memory is used by others as well")


@pytest.mark.parametrize("room,fits", [(1300, False), (1800, True)])
def test_traces_that_do_not_fit_leave_the_network_as_it_was(gpu, room, fits):
    """Imported traces that differ between the synapses of a neuron make the network keep them per
    synapse: 2 x 1,220 MB here, for an import that takes 1,220 MB itself, with `room` MB of memory free;
    the by-target index, 780 MB, may make way (and the runtime finds about 200). If they do not fit the import raises MemoryError, and
    the network goes on as one that was not asked; with memory again, it is imported."""
    import torch
    model, lay, delay = "brunel_with_plasticity", brunel_ref_layout(80000), 15
    a, b = _start(model, lay, delay, 11), _start(model, lay, delay, 11)
    for net in (a, b):
        net.run(21)
    z = b.synapses(ell=False)
    assert z["W"].nbytes >> 20 in range(1200, 1230), z["W"].nbytes
    z["Zpre"] = np.random.default_rng(12).uniform(1e-4, 2e-4, z["W"].size).astype(np.float32)
    fill = []
    try:
        _fill(fill, room)
        if fits:
            a.set_synapses(z, ell=False)
        else:
            with pytest.raises(MemoryError):
                a.set_synapses(z, ell=False)
            for net in (a, b):
                net.run(40)
            assert_state_equal(a.neurons(), b.neurons(), "after the refused import")
    finally:
        del fill[:]
        torch.cuda.empty_cache()
    if not fits:
        a.set_synapses(z, ell=False)
    b.set_synapses(z, ell=False)
    for net in (a, b):
        net.run(40)
    assert_state_equal(a.neurons(), b.neurons(), "after the import")
    x, y = a.synapses(ell=False), b.synapses(ell=False)
    assert_state_equal(x, y, "after the import")
    a.close(), b.close()


def test_a_batch_whose_tables_could_not_be_made_makes_them_later(gpu):
    """A member's imported traces take the whole batch to traces per synapse (2 x 305 MB for the other
    member, whose index gives 195 back) at the next run: without the memory run() raises MemoryError,
    each time; with memory again it goes on as a batch that always had it."""
    import torch
    lay = brunel_ref_layout(40000)
    batches = [Batch("brunel_with_plasticity", [(Layout(*lay), 15, 21 + k) for k in range(2)], DT, fixed_point=True) for _ in range(2)]
    z = batches[0].net(0).synapses(ell=False)
    z["Zpre"] = np.random.default_rng(22).uniform(1e-4, 2e-4, z["W"].size).astype(np.float32)
    for b in batches:
        b.run(20)
        b.net(0).set_synapses(z, ell=False)
    fill = []
    try:
        _fill(fill, 100)
        for _ in range(2):
            with pytest.raises(MemoryError):
                batches[0].run(33)
    finally:
        del fill[:]
        torch.cuda.empty_cache()
    for b in batches:
        b.run(33)
    for k in range(2):
        x, y = (b.net(k) for b in batches)
        assert x.clock() == y.clock()
        assert_state_equal(x.neurons(), y.neurons(), f"net {k}")
        assert_state_equal(x.synapses(ell=False), y.synapses(ell=False), f"net {k}")
    for b in batches:
        b.close()


@pytest.mark.parametrize("model,delay", [("brunel_3pop", 15), ("brunel_3pop_stdp", 15), ("brunel_3pop_stdp", 1)])
def test_autotune_leaves_parts_that_have_no_effect(gpu, model, delay):
    """Windows of several steps, and of plastic models, have one workgroup per tile: the parts of a
    delivery are not varied (a time that differs by chance would be reported as theirs)."""
    d = Snn(model, Layout(*three_pop_layout(2000)), DT, delay, seed=10, fixed_point=True)
    cfg, us = d.autotune(warmup=50, steps=20)
    assert cfg["recv_parts"] == 1 and d.launch()["recv_parts"] == 1 and us > 0
    d.close()
