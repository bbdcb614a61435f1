"""Performance cases of the simulator: what its users have it do, through the public Python API.

A case is one pass of a user's program with the network (or batch, server, buffers) already in
hand: a stretch of simulation followed by reading the state back, a control loop that takes the
spikes of every step, a graph generated into the caller's buffers, a sweep stepped as one batch,
a group of jobs served. Networks are the library's benchmark networks and their smaller and odd
sized relatives, at the launch shapes a new network has. dt is 0.1 ms throughout.

Which accumulation a case uses: the Brunel networks mix inputs of two or more weights, so their
fp32 sums depend on the order in which the inputs arrive, and a spike that moves by one step makes
whole runs incomparable; their cases use the fixed-point mode, whose results are the same bits on
every run. Vogels-Abbott inputs of one kind are all equal (any order of adding them rounds alike)
and synth counts integers, so those cases use the default fp32 mode.
"""
import math

import numpy as np
import torch

from spice_amd import Batch, Layout, Server, Snn
from spice_amd.models import MODELS
from spice_amd.snn import generate_graph

DT = 1e-4  # s


# ---- the cases -------------------------------------------------------------------------------
def _run(name, model, n, p, delay, steps, fixed, weights=False):
    return {"name": name, "kind": "run", "model": model, "n": n, "p": p, "delay": delay, "steps": steps, "fixed": fixed,
            "weights": weights}


def listed():
    return [
        # interactive control of a small network (the CPU-sized Vogels-Abbott network of 4,000
        # neurons, built from the user's own connectivity): every step's spikes are read back
        {"name": "control_loop_4000", "kind": "control", "n": 4000, "p": 0.02, "delay": 1, "steps": 10},
        # the smallest benchmark network (1e6 synapses), a fifth of a second of biological time:
        # a step is a few microseconds, so launches and latency are all there is
        _run("brunel_1e6", "brunel_3pop", 3162, 0.1, 15, 2000, True),
        # conductance-based network at 1e8 synapses, delay of one step
        _run("vogels_1e8", "vogels_abbott", 70710, 0.02, 1, 1000, False),
        # the same model at 1e9 synapses with the reference benchmark's delay of 8 steps
        _run("vogels_1e9_delay8", "vogels_abbott", 223606, 0.02, 8, 400, False),
        # the reference's synthetic network: many neurons, sparse rows, 4,000 spikes a step
        _run("synth_1e9", "synth", 800640, 0.00156, 1, 200, False),
        # the largest network: 1e10 synapses
        _run("brunel_1e10", "brunel_3pop", 316228, 0.1, 15, 200, True),
        # pair STDP at 1e9 synapses, the library's headline workload
        _run("stdp_1e9", "brunel_3pop_stdp", 100000, 0.1, 15, 400, True),
        # pair STDP at 1e7 synapses on the user's own connectivity (each neuron connected to a tenth
        # of the others), the learned weights read back after the stretch
        _run("stdp_1e7_weights", "brunel_3pop_stdp", 10000, 0.1, 15, 2000, True, True),
        # the reference's plastic benchmark network (per-synapse traces)
        _run("brunel_plus_6e8", "brunel_with_plasticity", 109544, 0.1, 15, 150, True),
        # network construction: the random graph of the reference's set-up benchmark (1e9 synapses)
        # into buffers that the caller owns
        {"name": "graph_1e9", "kind": "graph", "layout": "single", "n": 141421, "p": 0.05},
        # a parameter sweep: 48 networks of 1e4 to 1e7 synapses, each with its own input rate,
        # stepped together
        {"name": "sweep_48", "kind": "batch", "model": "brunel_3pop", "nets": 48, "lo": 1e4, "hi": 1e7, "steps": 500, "mix": 7},
        # jobs of three models built, stepped in batched chunks, streamed and released by a server
        {"name": "serve_12", "kind": "serve", "jobs": 12, "lo": 1e5, "hi": 3e6, "steps": 1000, "mix": 3},
    ]


def draw(rng):
    def between(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    kind = rng.choice(["run"] * 9 + ["control", "graph", "graph", "batch", "serve"])
    if kind == "control":
        return {"kind": "control", "n": int(between(500, 6000)), "p": 0.02, "delay": rng.randint(1, 8), "steps": rng.randint(4, 20)}
    if kind == "graph":
        p = between(0.002, 0.1)
        return {"kind": "graph", "layout": rng.choice(["single", "three"]), "n": int(math.sqrt(between(1e5, 6e8) / p)), "p": p}
    if kind == "batch":
        return {"kind": "batch", "model": rng.choice(["brunel_3pop", "vogels_abbott"]), "nets": rng.randint(3, 48), "lo": 1e4,
                "hi": between(1e6, 1e7), "steps": rng.randint(100, 500), "mix": rng.randint(0, 1 << 20)}
    if kind == "serve":
        return {"kind": "serve", "jobs": rng.randint(2, 12), "lo": 1e5, "hi": between(1e6, 3e6), "steps": rng.randint(200, 1000),
                "mix": rng.randint(0, 1 << 20)}
    model = rng.choice(["brunel", "brunel_3pop", "brunel_3pop", "vogels_abbott", "vogels_abbott", "vogels_abbott", "synth", "synth",
                        "brunel_3pop_stdp", "brunel_3pop_stdp", "brunel_with_plasticity"])
    plastic = bool(MODELS[model][2])
    syn = between(1e5, 3e8 if plastic else 1e9)
    p = 0.02 if model == "vogels_abbott" else between(0.002, 0.05) if model == "synth" else rng.uniform(0.06, 0.1)
    delay = rng.choice([1, 1, 2, 4, 8, 15, rng.randint(1, 24)])
    if plastic or model in ("brunel", "brunel_3pop"):
        delay = max(delay, rng.choice([1, 8, 15]))
    steps = int(min(2000, max(60, 1e11 / syn)) * rng.uniform(0.6, 1.0))
    if model == "brunel_with_plasticity":
        steps = min(steps, 300)
    return {"kind": "run", "model": model, "n": int(math.sqrt(syn / p)), "p": p, "delay": delay, "steps": steps,
            "fixed": model not in ("vogels_abbott", "synth"), "weights": plastic and syn < 3e6}


# ---- networks --------------------------------------------------------------------------------
def _three_pop(n, p):
    npois = n // 5
    ne = (n - npois) * 4 // 5
    return [npois, ne, n - npois - ne], [(s, d, p) for s in range(3) for d in range(3)]


def _layout(model, n, p):
    if model in ("brunel", "brunel_with_plasticity"):  # the reference's: Poisson half, recurrent half
        return Layout([n // 2, n - n // 2], [(0, 1, p), (1, 1, p)])
    if model.startswith("brunel_3pop"):
        return Layout(*_three_pop(n, p))
    return Layout([n], [(0, 0, p)])


def _start_state(model, n, rng):
    """Initial state of a trial: membrane potentials spread below the threshold (from the
    models' uniform initial value all neurons would fire their first spikes together)."""
    if model == "synth":
        return {"N": np.zeros(n, np.int32)}
    if model == "vogels_abbott":
        return {"V": rng.uniform(-0.06, -0.05, n).astype(np.float32), "Gex": rng.uniform(0.0, 0.1, n).astype(np.float32),
                "Gin": rng.uniform(0.0, 0.5, n).astype(np.float32), "Twait": np.zeros(n, np.int32)}
    return {"V": rng.uniform(0.0, 0.015, n).astype(np.float32), "Twait": np.zeros(n, np.int32)}


def _random_csr(n, p, seed):
    """A user's own connectivity: each pair connected with probability p, rows sorted."""
    rng = np.random.default_rng(seed)
    src, dst = np.nonzero(rng.random((n, n), dtype=np.float32) < p)
    rp = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(src, minlength=n), out=rp[1:])
    return rp, dst.astype(np.int32)


def _even_csr(n, p, seed):
    """A user's own connectivity with the same number of targets for every neuron, one in each
    of as many equal stretches of the network."""
    k = max(1, int(n * p))
    edge = np.arange(k + 1, dtype=np.int64) * n // k
    rng = np.random.default_rng(seed)
    col = edge[:-1] + (rng.random((n, k), dtype=np.float32) * (edge[1:] - edge[:-1])).astype(np.int64)
    return np.arange(n + 1, dtype=np.int64) * k, np.minimum(col, edge[1:] - 1).astype(np.int32).reshape(-1), k


def _mix(case, models):
    """Sizes, models and parameters of a group of networks: part of the case, not of its inputs."""
    rng = np.random.default_rng(case["mix"])
    out = []
    for k in range(case.get("nets") or case["jobs"]):
        model = models[k % len(models)]
        syn = float(np.exp(rng.uniform(np.log(case["lo"]), np.log(case["hi"]))))
        p = 0.02 if model == "vogels_abbott" else 0.1
        n = max(20, int(round(math.sqrt(syn / p))))
        rate = float(rng.uniform(5, 30))
        steps = int(case["steps"] * rng.uniform(0.5, 1.0))
        out.append((model, n, p, 1 if model == "vogels_abbott" else 15, [rate] if model.startswith("brunel") else None, steps))
    return out


SERVED = ["brunel_3pop", "vogels_abbott", "brunel_3pop", "vogels_abbott", "brunel_3pop_stdp"]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "control":
        rp, col = _random_csr(case["n"], case["p"], seed)
        width = (int(np.diff(rp).max()) + 31) // 32 * 32
        net = Snn.from_csr("vogels_abbott", rp, col, width, DT, case["delay"], seed=seed)
        net.set_neurons(_start_state("vogels_abbott", case["n"], np.random.default_rng(seed + 1)))
        return {"kind": kind, "net": net, "steps": case["steps"], "n": case["n"]}
    if kind == "run":
        if case["weights"]:
            rp, col, k = _even_csr(case["n"], case["p"], seed)
            net = Snn.from_csr(case["model"], rp, col, (k + 31) // 32 * 32, DT, case["delay"], seed=seed, fixed_point=case["fixed"])
        else:
            net = Snn(case["model"], _layout(case["model"], case["n"], case["p"]), DT, case["delay"], seed=seed,
                      fixed_point=case["fixed"])
        net.set_neurons(_start_state(case["model"], case["n"], np.random.default_rng(seed + 1)))
        return {"kind": kind, "net": net, "steps": case["steps"], "weights": case["weights"]}
    if kind == "graph":
        lay = Layout(*_three_pop(case["n"], case["p"])) if case["layout"] == "three" else Layout(case["n"], case["p"])
        # (rows are never longer than the layout's ELL width; the entries past the graph's end stay 0)
        return {"kind": kind, "layout": lay, "seed": seed, "row_ptr": torch.empty(case["n"] + 1, dtype=torch.int64, device="cuda"),
                "col": torch.zeros(case["n"] * lay.max_degree(), dtype=torch.int32, device="cuda")}
    if kind == "batch":
        nets = [(_layout(m, n, p), d, seed + 1 + k, par) for k, (m, n, p, d, par, _) in enumerate(_mix(case, [case["model"]]))]
        return {"kind": kind, "batch": Batch(case["model"], nets, DT, fixed_point=True), "steps": case["steps"]}
    counts = {}

    def sink(job, first, offsets, ids):
        n = sizes[job]
        counts[job] = counts.get(job, 0) + np.bincount(ids, minlength=n)

    sizes = {}
    jobs = [(m, _layout(m, n, p), d, par, steps, n) for m, n, p, d, par, steps in _mix(case, SERVED)]
    return {"kind": kind, "server": Server(budget_bytes=50e9, chunk_steps=500, on_spikes=sink), "jobs": jobs, "seed": seed,
            "sizes": sizes, "counts": counts, "next": 1}


def run(state):
    kind = state["kind"]
    if kind == "control":
        net = state["net"]
        raster = np.zeros((state["steps"], state["n"]), bool)
        for t in range(state["steps"]):
            raster[t, net.step(spikes=True)] = True
        return {"raster": raster, "neurons": net.neurons()}
    if kind == "run":
        net = state["net"]
        net.run(state["steps"])
        out = {"neurons": net.neurons()}
        if state["weights"]:
            out["synapses"] = net.synapses(ell=False)
        return out
    if kind == "graph":
        col = state["col"]
        nnz, width = generate_graph(state["layout"], state["seed"], state["row_ptr"].data_ptr(), col.data_ptr(), col.numel())
        return {"row_ptr": state["row_ptr"], "col": col, "nnz": nnz, "width": width}
    if kind == "batch":
        b = state["batch"]
        b.run(state["steps"])
        nets = [b.net(i).neurons() for i in range(len(b))]
        return {k: np.concatenate([s[k] for s in nets]) for k in nets[0]}
    sv, sizes, counts = state["server"], state["sizes"], state["counts"]
    first = state["next"]  # the server numbers its jobs from 1
    state["next"] += len(state["jobs"])
    for k, (m, lay, d, par, steps, n) in enumerate(state["jobs"]):
        sizes[first + k] = n
        sv.submit(m, lay, DT, steps, delay=d, seed=state["seed"] + 1 + k, params=par, fixed_point=True)
    recs = [sv.wait(first + k) for k in range(len(state["jobs"]))]
    spikes = np.concatenate([np.zeros(sizes[r["id"]], np.int64) + counts.pop(r["id"], 0) for r in recs])
    return {"spikes_of_neuron": spikes, "digest": np.array([r["digest"] for r in recs], np.uint64).view(np.int64),
            "events": np.array([r["events"] for r in recs], np.int64)}


# ---- what a pass cannot do without -----------------------------------------------------------
def _spikes_per_step(model, n):
    """Typical activity of the models (spikes a step), for the bytes that delivery needs."""
    if model == "synth":
        return 0.005 * n
    if model == "vogels_abbott":
        return 10.5 * DT * n
    if model in ("brunel", "brunel_with_plasticity"):
        return (0.5 * 20 + 0.5 * 34) * DT * n
    return (0.2 * 20 + 0.8 * 14) * DT * n


def _net_bytes(model, n, p, steps):
    """Of `steps` steps of a network: neuron state read and written; per spike its id, row bounds
    and the target ids (and, of plastic models, the weights) of its row; per plastic spike its
    row's and its target's synapses read and written."""
    _, nattrs, sattrs = MODELS[model]
    state = 2 * 4 * len(nattrs) * n
    spk = _spikes_per_step(model, n)
    row = n * p * (0.5 if model in ("brunel", "brunel_with_plasticity") else 1.0)
    ev = spk * row
    per = 20 * spk + ev * 4
    if sattrs:
        per += ev * 4 + ev * 0.5 * 2 * 8 * len(sattrs)
    return steps * (state + per), steps * (4 * n + 2 * ev)


def work(case):
    kind = case["kind"]
    if kind in ("control", "run"):
        b, f = _net_bytes(case.get("model", "vogels_abbott"), case["n"], case["p"], case["steps"])
        return {"bytes": b, "flops": f}
    if kind == "graph":
        nnz = case["p"] * case["n"] ** 2
        return {"bytes": 4 * nnz + 8 * case["n"], "flops": 60 * nnz}  # logarithm and division in double
    total = [0.0, 0.0]
    for m, n, p, _, _, steps in _mix(case, [case["model"]] if kind == "batch" else SERVED):
        b, f = _net_bytes(m, n, p, case["steps"] if kind == "batch" else steps)
        if kind == "serve":
            b, f = b + 4 * p * n * n, f + 60 * p * n * n  # its graph is generated too
        total = [total[0] + b, total[1] + f]
    return {"bytes": total[0], "flops": total[1]}


# ---- the same in 64 bits ---------------------------------------------------------------------
def exact(case, seed):
    """The control loop's membrane potentials and conductances: the Vogels-Abbott equations
    (Euler steps, exponential conductances) in double precision. The other cases' networks run
    long enough to amplify any rounding, and return whole numbers or fixed-point sums."""
    if case["kind"] != "control":
        return None
    n, steps, delay = case["n"], case["steps"], case["delay"]
    rp, col = _random_csr(n, case["p"], seed)
    s = _start_state("vogels_abbott", n, np.random.default_rng(seed + 1))
    v, gex, gin = (s[k].astype(np.float64) for k in ("V", "Gex", "Gin"))
    wait = s["Twait"].copy()
    nexc = int(np.float32(0.8) * np.float32(n))
    dt, wex, win = float(np.float32(DT)), 0.4 * 16e6 / n**2, 5.1 * 16e6 / n**2
    fired = []
    for t in range(steps):
        for src in fired[t - delay] if t >= delay else ():
            if src < nexc:
                gex[col[rp[src]:rp[src + 1]]] += wex
            else:
                gin[col[rp[src]:rp[src + 1]]] += win
        wait -= 1
        ready = wait <= 0
        spike = ready & (v > np.float64(np.float32(-0.05)))
        drift = ((-0.06 - v) + gex * (0.0 - v) + gin * (-0.08 - v) + 0.02) * (dt * 50.0)
        v = np.where(spike, -0.06, np.where(ready, v + drift, v))
        wait[spike] = 50
        gex -= gex * (dt * 200.0)
        gin -= gin * (dt * 100.0)
        fired.append(np.flatnonzero(spike))
    return {"raster": None, "neurons": {"V": v, "Gex": gex, "Gin": gin, "Twait": None}}
