"""Window kernels (static networks: up to `delay` steps per launch, each tile delivered and
updated by one workgroup) against the CPU checker, fixed point and so bit for bit: delays below,
at and above the longest window and at multiples of the clock's slots, tiles of one wave, ragged
last tiles, tiles without inputs, wide tiles, rows with many and with no targets in a tile; runs
that end inside a window; and fp32 inputs past the tabulated sums."""
import numpy as np
import pytest

from oracle import oracle as O
from spice_amd import Batch, Layout, Snn
from tests.helpers import assert_state_equal, brunel_ref_layout, three_pop_layout

pytestmark = pytest.mark.gpu

DT = 1e-4
RUNS = (1, 2, 3, 4, 5, 7, 8, 15, 16, 29, 30, 31, 60, 1, 89)  # 301 steps


@pytest.mark.parametrize("model,layout,delay,launch", [
    ("brunel_3pop", three_pop_layout(1500), 2, (0, 0)),
    ("brunel_3pop", three_pop_layout(1500), 3, (64, 256)),
    ("brunel_3pop", three_pop_layout(1111), 4, (128, 1024)),
    ("brunel_3pop", three_pop_layout(2000), 15, (1024, 256)),
    ("brunel_3pop", three_pop_layout(1500), 16, (192, 512)),
    ("brunel_3pop", three_pop_layout(777), 40, (0, 0)),
    ("brunel", brunel_ref_layout(1500), 15, (64, 512)),  # half of the tiles receive nothing
    ("vogels_abbott", ([1300], [(0, 0, 0.3)]), 8, (256, 512)),
    ("vogels_abbott", ([2500], [(0, 0, 0.02)]), 5, (64, 256)),
    ("vogels_abbott", ([4200], [(0, 0, 0.02)]), 1, (4096, 1024)),
    ("synth", ([3000], [(0, 0, 0.001)]), 7, (64, 1024)),  # most segments empty
    ("synth", ([500], [(0, 0, 1.0)]), 12, (512, 256)),  # every row in full
    ("synth", ([65], [(0, 0, 0.5)]), 1, (0, 0)),
    ("synth", ([40], [(0, 0, 0.0)]), 3, (0, 0)),  # no synapse at all
])
def test_windows_bit_exact(gpu, model, layout, delay, launch):
    h = O.CpuSnn(model, layout, DT, delay, seed=81, fixed_point=True)
    d = Snn(model, Layout(*layout), DT, delay, seed=81, fixed_point=True)
    d.set_launch(tile_w=launch[0], recv_block=launch[1])
    done = 0
    for n in RUNS:
        d.run(n)
        h.run(n)
        done += n
        assert d.clock() == h.clock()
        assert_state_equal(d.neurons(), h.neurons(), f"{model} after {done} steps")
    for i in range(3):
        np.testing.assert_array_equal(np.sort(d.step(True)), np.sort(h.step(True)), err_msg=f"step {done + i}")
    ms = d.run_profiled(20)
    h.run(20)
    assert ms["receive"] == 0 and ms["update"] == 0 and ms["step"] > 0
    assert_state_equal(d.neurons(), h.neurons(), "after profiled steps")
    d.close(), h.close()


@pytest.mark.parametrize("model", ["vogels_abbott", "synth"])
@pytest.mark.parametrize("p", [0.004, 0.02, 0.05, 0.1, 0.3])
def test_segment_records_bit_exact(gpu, model, p):
    """Delay 1: records of 16, 32 and 64 bytes (segments of 1 to 13 targets, some longer than
    their record) and segments too long for any; the tiles change on the way (Vogels: all neurons
    fire at step 139)."""
    lay = ([2500], [(0, 0, p)])
    h = O.CpuSnn(model, lay, DT, 1, seed=23, fixed_point=True)
    d = Snn(model, Layout(*lay), DT, 1, seed=23, fixed_point=True)
    for w, block in ((256, 512), (320, 256), (64, 1024)):
        d.set_launch(tile_w=w, recv_block=block)
        d.run(149)
        h.run(149)
        assert_state_equal(d.neurons(), h.neurons(), f"tiles of {w}")
        s = h.step(True)
        np.testing.assert_array_equal(np.sort(d.step(True)), np.sort(s))
    assert d.stats()["events"] > 0
    d.close(), h.close()


@pytest.mark.parametrize("delay", [1, 6])
def test_fp32_inputs_past_the_tabulated_sums(gpu, delay):
    """Vogels-Abbott in fp32: the whole population's first spike gives every neuron hundreds of
    inputs of one value in one step, whose fp32 sum is the same in any order of adding them."""
    lay = ([900], [(0, 0, 0.4)])
    h = O.CpuSnn("vogels_abbott", lay, DT, delay, seed=5)
    d = Snn("vogels_abbott", Layout(*lay), DT, delay, seed=5)
    for n in (130, 5, 5, 5, 40):
        d.run(n)
        h.run(n)
        assert_state_equal(d.neurons(), h.neurons(), f"after {d.clock()[0]} steps")
    st = d.stats()
    assert st["spikes"] >= 900 and st["events"] > 64 * 900
    d.close(), h.close()


@pytest.mark.parametrize("delay,launch", [(1, (0, 0, 0, 0)), (2, (64, 256, 64, 1)), (3, (128, 512, 64, 7)), (9, (0, 0, 0, 0)), (10, (448, 1024, 1024, 300)),
                                          (12, (64, 512, 128, 64)), (255, (0, 0, 0, 0))])
def test_plastic_windows_bit_exact(gpu, delay, launch):
    """Pair STDP in windows (of up to 10 steps: the refractory promise allows (19 + 1) / 2), the
    passes of each beside the next: state and every weight against the checker's dense per-step
    plasticity, at window lengths on both sides of the clock's slots, over history words' ends
    and the ring of 256 steps, weights exported between windows."""
    lay = three_pop_layout(900)
    h = O.CpuSnn("brunel_3pop_stdp", lay, DT, delay, seed=33, fixed_point=True)
    d = Snn("brunel_3pop_stdp", Layout(*lay), DT, delay, seed=33, fixed_point=True)
    d.set_launch(tile_w=launch[0], recv_block=launch[1], flush_slots=launch[2], flush_grid=launch[3])
    for k, n in enumerate((60, 1, 2, 3, 4, 9, 10, 11, 21, 64, 130, 5, 200)):
        d.run(n)
        h.run(n)
        assert_state_equal(d.neurons(), h.neurons(), f"after run {k}")
        if k % 3 == 0:
            assert_state_equal(d.synapses(ell=False), h.synapses(ell=False), f"weights after run {k}")
    assert_state_equal(d.synapses(ell=False), h.synapses(ell=False), "weights")
    d.close(), h.close()


@pytest.mark.parametrize("batched", [False, True])
def test_imported_state_that_breaks_the_refractory_promise(gpu, batched):
    """Neuron state imported in mid-run lets neurons spike and accept input a few steps after a
    spike; windows rely on 19 refractory steps, so the steps until those spikes have arrived run
    one by one. Against the checker, weights included."""
    lay = three_pop_layout(700)
    h = O.CpuSnn("brunel_3pop_stdp", lay, DT, 15, seed=3, fixed_point=True)
    if batched:
        b = Batch("brunel_3pop_stdp", [(Layout(*lay), 15, 3), (Layout(*lay), 15, 4)], DT, fixed_point=True)
        run, net = b.run, b.net(0)
    else:
        net = Snn("brunel_3pop_stdp", Layout(*lay), DT, 15, seed=3, fixed_point=True)
        run = net.run
    run(157)
    h.run(157)
    for n in (40, 23, 60):
        s = h.neurons()
        s["V"] = np.full_like(s["V"], 0.021)
        s["Twait"] = np.full_like(s["Twait"], 4)
        net.set_neurons(s)
        h.set_neurons(s)
        run(n)
        h.run(n)
        assert_state_equal(net.neurons(), h.neurons(), "neurons")
    assert_state_equal(net.synapses(ell=False), h.synapses(ell=False), "weights")
    h.close()


@pytest.mark.parametrize("n", [16384, 16385, 20000])
def test_spikes_and_state_read_back(gpu, n):
    """Steps whose spikes (all neurons' at step 139) and networks whose state just fit, or do not
    fit, the pinned buffer of 16,384 words that small answers come through."""
    lay = ([n], [(0, 0, 0.0005)])
    h = O.CpuSnn("vogels_abbott", lay, DT, 1, seed=3, fixed_point=True)
    d = Snn("vogels_abbott", Layout(*lay), DT, 1, seed=3, fixed_point=True)
    d.run(135), h.run(135)
    sizes = []
    for i in range(10):
        want = np.sort(h.step(True))
        np.testing.assert_array_equal(np.sort(d.step(True)), want, err_msg=f"step {135 + i}")
        np.testing.assert_array_equal(np.sort(d.step_spikes_of_last()), want)
        assert_state_equal(d.neurons(), h.neurons(), f"step {135 + i}")
        sizes.append(len(want))
    assert min(sizes) == 0 and max(sizes) == n
    d.close(), h.close()


@pytest.mark.parametrize("model,layout,delay,launch", [
    ("synth", ([66000], [(0, 0, 0.005)]), 3, (1024, 512)),  # ids past 16 bits, 5 targets per segment
    ("vogels_abbott", ([700], [(0, 0, 0.1)]), 5, (64, 1024)),
    ("synth", ([901], [(0, 0, 0.9)]), 4, (64, 512)),  # 8 per lane: 57 targets per segment
    ("brunel_3pop", three_pop_layout(1500), 15, (640, 512)),
    ("synth", ([300], [(0, 0, 1.0)]), 1, (256, 256)),  # step by step, too long for records
    ("synth", ([257], [(0, 0, 1.0)]), 2, (64, 256)),
    ("synth", ([40000], [(0, 0, 0.025)]), 3, (0, 0)),  # the tiles that it is built with: 209 of 192
    ("vogels_abbott", ([20003], [(0, 0, 0.06)]), 6, (0, 0)),
    ("brunel_3pop_stdp", three_pop_layout(66000, 0.005), 15, (1024, 512)),  # beside the weights
    ("brunel_3pop_stdp", three_pop_layout(500), 3, (64, 256)),
])
def test_halved_row_store_bit_exact(gpu, model, layout, delay, launch):
    """Deliveries from the low halves of the target ids, 4 and 8 per lane: segments that begin and
    end anywhere in a piece, the row store's last ones, tiles on both sides of id 65,536."""
    h = O.CpuSnn(model, layout, DT, delay, seed=31, fixed_point=True)
    d = Snn(model, Layout(*layout), DT, delay, seed=31, fixed_point=True)
    d.set_launch(tile_w=launch[0], recv_block=launch[1])
    for n in (7, 160, 33):
        d.run(n)
        h.run(n)
        assert_state_equal(d.neurons(), h.neurons(), model)
    assert d.stats()["events"] > 0
    d.close(), h.close()


def _repeated_rows(n, base, seed, first):
    """Rows of `base` random targets from neuron `first` on; ten Poisson sources (of brunel_3pop) and two excitatory neurons
    also name two targets of one tile 66,000 to 140,000 times in all."""
    rng = np.random.default_rng(seed)
    rows = [np.sort(first + rng.choice(n - first, base, replace=False)) for _ in range(n)]
    sources = list(range(0, n // 5, max(1, n // 50)))[:10] + [n // 3, n // 2]
    for k, s in enumerate(sources):
        x = int(rng.integers(-(-first // 64), n // 64)) * 64
        more = np.repeat([x + 3, x + 40], [65536 + 7 * k, 400 + 6500 * k])
        rows[s] = np.sort(np.concatenate([rows[s], more]))
    rp = np.zeros(n + 1, np.int64)
    np.cumsum([r.size for r in rows], out=rp[1:])
    return rp, np.concatenate(rows).astype(np.int32), (max(r.size for r in rows) + 31) // 32 * 32


@pytest.mark.parametrize("model,n,base,delay", [
    ("brunel_3pop", 512, 40, 15),   # low halves, 8 per lane
    ("brunel_3pop", 1984, 40, 15),  # low halves, 4 per lane
    ("brunel_3pop", 9984, 5, 6),    # the row store itself
    ("brunel_3pop", 1984, 20, 1),   # records, and segments too long for any
    ("brunel_3pop_stdp", 512, 40, 15),
    ("brunel_3pop_stdp", 9984, 5, 1),
    ("brunel_with_plasticity", 1984, 20, 9),
])
def test_targets_named_many_times(gpu, model, n, base, delay):
    """More than 65,536 entries of a row in one tile, in windows of every length."""
    # (brunel_with_plasticity: targets in its LIF half, as windows need)
    rp, col, width = _repeated_rows(n, base, 91, n // 2 if model == "brunel_with_plasticity" else 0)
    h = O.CpuSnn.from_csr(model, rp, col, width, DT, delay, seed=91, fixed_point=True)
    d = Snn.from_csr(model, rp, col, width, DT, delay, seed=91, fixed_point=True)
    for k in (130, 1, 7, 62):
        d.run(k)
        h.run(k)
        assert_state_equal(d.neurons(), h.neurons(), model)
    np.testing.assert_array_equal(np.sort(d.step(True)), np.sort(h.step(True)))
    events = d.stats()["events"]
    assert events > 65536, events
    if model == "brunel_3pop_stdp":
        np.testing.assert_array_equal(d.synapses(ell=False)["W"].view(np.uint32), h.synapses(ell=False)["W"].view(np.uint32))
    d.close(), h.close()


@pytest.mark.parametrize("model,pops,p,delay", [
    ("synth", [299000, 1000], 0.05, 1),
    ("brunel_3pop_stdp", [150000, 50000, 1500, 500], 0.02, 15),
    ("synth", [200000], 0.0, 1),  # no synapse at all
])
def test_few_targets(gpu, model, pops, p, delay):
    """Many sources, few targets: the memory of the network is in proportion (the segment table has
    an entry for every row and tile, tiles without inputs included)."""
    import torch
    layout = (pops, [(s, len(pops) - 1, p) for s in range(len(pops))])
    free = torch.cuda.mem_get_info()[0]
    d = Snn(model, Layout(*layout), DT, delay, seed=93, fixed_point=True)
    taken = free - torch.cuda.mem_get_info()[0]
    assert taken < 3 << 30, taken
    h = O.CpuSnn(model, layout, DT, delay, seed=93, fixed_point=True)
    for k in (25, 3):
        d.run(k)
        h.run(k)
        assert_state_equal(d.neurons(), h.neurons(), model)
    np.testing.assert_array_equal(np.sort(d.step(True)), np.sort(h.step(True)))
    d.close(), h.close()


@pytest.mark.parametrize("model,layout,delay,launch", [
    ("brunel_3pop", three_pop_layout(1500), 15, (0, 0)),
    ("brunel_3pop", three_pop_layout(5000, 0.3), 15, (1024, 1024)),  # 200 targets per segment
    ("brunel_3pop", three_pop_layout(2100), 3, (192, 256)),
    ("brunel", brunel_ref_layout(1500), 1, (0, 0)),
    ("vogels_abbott", ([2500], [(0, 0, 0.02)]), 1, (0, 0)),      # records
    ("synth", ([9000], [(0, 0, 0.01)]), 7, (64, 512)),           # more than 63 tiles
    ("synth", ([3000], [(0, 0, 0.001)]), 1, (1024, 256)),
    ("brunel_3pop_stdp", three_pop_layout(1500), 15, (0, 0)),
    ("brunel_3pop_stdp", three_pop_layout(1500), 1, (128, 256)),
    ("brunel_3pop_stdp_deferred", three_pop_layout(1500), 4, (0, 0)),
    ("brunel_with_plasticity", brunel_ref_layout(1200), 9, (0, 0)),
    ("brunel_with_plasticity", ([300, 900], [(0, 0, 0.05), (1, 0, 0.05), (1, 1, 0.05)]), 9, (0, 0)),  # per-synapse contract
])
def test_offsets_in_place_of_the_segment_table(gpu, model, layout, delay, launch):
    """Networks declared wide enough for rows of 2^24 targets have 4-byte offsets of each tile's
    targets instead of the segment table (as do those whose table would take too much memory)."""
    h = O.CpuSnn(model, layout, DT, delay, seed=95, fixed_point=True)
    rp, col = h.csr()
    d = Snn.from_csr(model, rp, col, 1 << 24, DT, delay, seed=95, fixed_point=True)
    for k, (tw, bs) in ((100, (0, 0)), (31, launch), (8, launch)):
        d.set_launch(tile_w=tw, recv_block=bs)
        d.run(k)
        h.run(k)
        assert_state_equal(d.neurons(), h.neurons(), model)
    np.testing.assert_array_equal(np.sort(d.step(True)), np.sort(h.step(True)))
    if model.startswith("brunel_3pop_stdp"):
        np.testing.assert_array_equal(d.synapses(ell=False)["W"].view(np.uint32), h.synapses(ell=False)["W"].view(np.uint32))
    d.close(), h.close()


def test_row_of_more_than_2_24_targets(gpu):
    n, delay = 320, 4
    rows = [np.arange(k % 7, n, 7) for k in range(n)]
    rows[5] = np.sort(np.concatenate([np.full((1 << 24) + 9, 100), rows[5]]))
    rp = np.zeros(n + 1, np.int64)
    np.cumsum([r.size for r in rows], out=rp[1:])
    col, width = np.concatenate(rows).astype(np.int32), (rows[5].size + 31) // 32 * 32
    h = O.CpuSnn.from_csr("brunel_3pop", rp, col, width, DT, delay, seed=6, fixed_point=True)
    d = Snn.from_csr("brunel_3pop", rp, col, width, DT, delay, seed=6, fixed_point=True)
    fired = 0
    for k in range(60):
        d.run(20)
        h.run(20)
        assert_state_equal(d.neurons(), h.neurons(), f"after {20 * k + 20} steps")
        fired = d.stats()["events"] >> 24
        if fired:
            break
    assert fired  # neuron 5, a Poisson source
    d.close(), h.close()
