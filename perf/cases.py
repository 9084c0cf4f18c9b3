"""Timed cases of the framework's public entry points.

The phonon engine (psim_amd.Engine, psim_amd.Model, psim_amd.run_batch) from the smallest run a
program makes to the benchmark's L-shape, in each simulation type and on both tally paths, and the
warm-start surrogate (psim_amd.surrogate.Surrogate): prediction, gradients and training.

listed()       the named cases
draw(rng)      one more case of the same ranges
prepare(c, s)  what a program holds before the call, made from seed s
run(state)     one pass
work(c)        bytes and floating-point operations the pass cannot do without
exact(c, s)    the pass's outputs in 64 bits, where they have such a value
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

import psim_amd
from psim_amd import configs, surrogate

LAYER_DIMS = [surrogate.N_FEATURES] + [surrogate.HIDDEN] * surrogate.LAYERS + [16]

# What a Monte Carlo pass cannot do without, for work() alone: FP64 operations of one event (drift,
# three edge predicates, one crossing; a scatter's draws and rates), and the events themselves. A
# phonon lives LIFE x sqrt(simulated ns) on average and meets RATE scatters and wall hits per ns of
# its life (the engine's counters on the listed cases; a bar's hits grow with its sensors).
FP64_PER_EVENT = 150.0
LIFE = {"bar": 0.195, "lshape": 0.85, "film": 0.86, "batch": 0.24}
RATE = {"bar": 161.0, "lshape": 146.0, "film": 209.0, "batch": 318.0}


def listed() -> list:
    return [
        # The smallest run: a quick look at a bar, replayed from its graph as a seed sweep does.
        {"name": "bar_5e3_graph", "kind": "bar", "graph": True, "sensors": 10, "phonons": 5000, "steps": 400,
         "sim_ns": 2.0, "spec": 0.0},
        # The 1000 x 100 nm bar at its configured size, a whole model run with its interpretation.
        {"name": "bar_1e5", "kind": "bar", "graph": False, "sensors": 10, "phonons": 100_000, "steps": 2000,
         "sim_ns": 10.0, "spec": 0.0},
        # A bar cut into many sensors: more tallies than the LDS holds.
        {"name": "bar_1000_sensors", "kind": "bar", "graph": False, "sensors": 1000, "phonons": 1_000_000,
         "steps": 1000, "sim_ns": 0.5, "spec": 1.0},
        # The L-shape of the benchmark, at its size: full mode, steady state.
        {"name": "lshape_1e7", "kind": "lshape", "type": 0, "phonons": 10_000_000, "steps": 5000, "sim_ns": 10.0,
         "spec": 0.3},
        # The L-shape with every step recorded (periodic snapshots).
        {"name": "lshape_periodic", "kind": "lshape", "type": 1, "phonons": 1_600_000, "steps": 2500, "sim_ns": 5.0,
         "spec": 0.3},
        # The heated film, every step recorded, phonons born in a burst.
        {"name": "film_3e6", "kind": "film", "phonons": 3_000_000, "steps": 3000, "sim_ns": 3.0},
        # Structures of the batched-geometry family as one run.
        {"name": "batch_32", "kind": "batch", "type": 0, "count": 32, "phonons": 0, "steps": 2000, "sim_ns": 10.0},
        # Relaxations of a few structures, every step recorded: how the surrogate's data are made.
        {"name": "relax_8", "kind": "batch", "type": 1, "count": 8, "phonons": 100_000, "steps": 1000, "sim_ns": 10.0},
        # The start field of one structure.
        {"name": "predict_101", "kind": "predict", "rows": 101},
        # The start fields of a thousand structures (a validation set).
        {"name": "predict_100003", "kind": "predict", "rows": 100_003},
        # Loss and gradients of one ragged batch.
        {"name": "gradients_5003", "kind": "gradients", "rows": 5003},
        # Training: a few mini-batches of the default size, from the initial weights to the new ones.
        {"name": "fit_6x4096", "kind": "fit", "batch": 4096, "batches": 6},
    ]


def _log(rng: random.Random, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["bar", "bar", "lshape", "film", "batch", "predict", "gradients", "fit"])
    if kind == "bar":
        many = rng.random() < 0.4
        steps = _log(rng, 200, 2000)
        return {"kind": kind, "graph": rng.random() < 0.5, "sensors": _log(rng, 100, 1000) if many else rng.randint(4, 40),
                "phonons": _log(rng, 3e3, 2e6), "steps": steps, "sim_ns": steps * (0.0005 if many else rng.choice([0.001, 0.005])),
                "spec": rng.choice([0.0, 0.3, 1.0])}
    if kind == "lshape":
        steps = _log(rng, 500, 4000)
        return {"kind": kind, "type": rng.choice([0, 1]), "phonons": _log(rng, 2e4, 4e6), "steps": steps,
                "sim_ns": steps * 0.002, "spec": rng.choice([0.0, 0.3, 1.0])}
    if kind == "film":
        steps = _log(rng, 500, 4000)
        return {"kind": kind, "phonons": _log(rng, 2e4, 5e6), "steps": steps, "sim_ns": steps * 0.001}
    if kind == "batch":
        kind_type = rng.choice([0, 1])
        return {"kind": kind, "type": kind_type, "count": _log(rng, 2, 10 if kind_type else 32),
                "phonons": _log(rng, 1e4, 2e5), "steps": _log(rng, 300, 1000 if kind_type else 2000),
                "sim_ns": 10.0}
    if kind == "predict":
        return {"kind": kind, "rows": _log(rng, 1, 2e5)}
    if kind == "gradients":
        return {"kind": kind, "rows": _log(rng, 16, 3e4)}
    return {"kind": "fit", "batch": _log(rng, 64, 8192), "batches": rng.randint(2, 8)}


def _model(case: dict, rng: random.Random) -> dict:
    """The case's structure in the input schema, walls moved by up to 5 K."""
    if case["kind"] == "bar":
        return configs.linear_bar(num_sensors=case["sensors"], t_hot=310.0 + rng.uniform(-5, 5),
                                  t_cold=290.0 + rng.uniform(-5, 5), spec=case["spec"], num_phonons=case["phonons"],
                                  num_measurements=case["steps"], sim_time=case["sim_ns"]).to_dict()
    if case["kind"] == "lshape":
        return configs.lshape(num_phonons=case["phonons"], num_measurements=case["steps"], sim_time=case["sim_ns"],
                              t_hot=320.0 + rng.uniform(-5, 5), t_cold=280.0 + rng.uniform(-5, 5), spec=case["spec"],
                              sim_type=case["type"], step_interval=100 if case["type"] else 0).to_dict()
    return configs.film_transient(num_phonons=case["phonons"], num_measurements=case["steps"],
                                  sim_time=case["sim_ns"], burst_temp=320.0 + rng.uniform(-5, 5))


def _structures(case: dict, rng: random.Random) -> list:
    # the sensor counts and budgets of the family's first structures, so that every seed's batch is
    # the same size; everything else is drawn
    sizes = random.Random(0)
    out = []
    for _ in range(case["count"]):
        size, p = configs.batch_geometry_params(sizes), configs.batch_geometry_params(rng)
        p["n_sensors"] = size["n_sensors"]
        p["phonons"] = case["phonons"] or size["phonons"]
        p["kinked"], p["theta"] = size["kinked"], size["theta"]
        p["length"], p["width"], p["spec"] = size["length"], size["width"], size["spec"]
        out.append(p)
    return out


def _rows(rows: int, seed: int):
    """Inputs and targets: sensors of structures of the family, their shape near the linear one."""
    rng = random.Random(seed)
    some = np.concatenate([surrogate.features(configs.batch_geometry_params(rng)) for _ in range(24)])
    g = np.random.default_rng(seed)
    x = some[g.integers(0, len(some), rows)]
    x *= (1.0 + 0.02 * g.standard_normal(x.shape, np.float32))
    t = (1.0 - 2.0 * x[:, 8] + 0.1 * np.sin(5.0 * x[:, 14]) + 0.005 * g.standard_normal(rows)).astype(np.float32)
    return x, t


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    rng = random.Random(seed)
    if kind in ("bar", "lshape", "film"):
        engine = psim_amd.Engine(0)
        model = psim_amd.Model(_model(case, rng))
        state = {"call": "graph" if case.get("graph") else "model", "engine": engine, "model": model, "seed": seed}
        if case.get("graph"):
            model.upload(engine, seed)
        return state
    if kind == "batch":
        models = [psim_amd.Model(configs.geometry_from_params(p, case["steps"], case["sim_ns"], sim_type=case["type"],
                                                              step_interval=100 if case["type"] else 0))
                  for p in _structures(case, rng)]
        return {"call": "batch", "engine": psim_amd.Engine(0), "models": models, "seed": seed}
    if kind == "predict":
        return {"call": "predict", "net": surrogate.load_weights(), "x": _rows(case["rows"], seed)[0]}
    net = surrogate.Surrogate(seed=seed)
    if kind == "gradients":
        x, t = _rows(case["rows"], seed)
        return {"call": "gradients", "net": net, "x": x, "t": t}
    x, t = _rows(case["batch"] * case["batches"], seed)
    return {"call": "fit", "net": net, "x": x, "t": t, "batch": case["batch"], "first": net.initial_params(seed)}


def _results(model) -> dict:
    r = model.results(0)
    return {"measurements": r.measurements, "temps": r.temps, "fluxes": r.fluxes, "counts": r.counts,
            "raw_flux": r.raw_flux, "counters": dict(r.counters)}


def run(state: dict):
    call = state["call"]
    if call == "model":
        state["model"].run(state["engine"], state["seed"])
        return _results(state["model"])
    if call == "graph":
        m = state["model"]
        return state["engine"].run_graph(m.num_sensors, m.num_record, state["seed"])
    if call == "batch":
        counters = psim_amd.run_batch(state["engine"], state["models"], state["seed"])
        got = [m.results(0) for m in state["models"]]
        # at most a few arrays, whole: the models' fields one after the other
        return {"counters": counters, "measurements": np.concatenate([r.measurements for r in got]),
                "temps": np.concatenate([r.temps.ravel() for r in got]),
                "fluxes": np.concatenate([r.fluxes.ravel() for r in got]),
                "counts": np.concatenate([r.counts.ravel() for r in got])}
    if call == "predict":
        return state["net"].predict(state["x"])
    if call == "gradients":
        loss, grad = state["net"].gradients(state["x"], state["t"])
        return {"loss": loss, "grad": grad}
    net = state["net"]
    net.set_params(state["first"])  # a training from the initial weights; resets the optimiser
    history = net.fit(state["x"], state["t"], epochs=1, batch=state["batch"], lr=1e-3)
    return {"history": history, "params": net.params()}


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("predict", "gradients", "fit"):
        rows = case["rows"] if kind != "fit" else case["batch"] * case["batches"]
        weights = sum(a * b for a, b in zip(LAYER_DIMS[:-2], LAYER_DIMS[1:-1])) + surrogate.HIDDEN
        params = weights + surrogate.HIDDEN * surrogate.LAYERS + 1
        if kind == "predict":  # inputs in, one value a row out, the bf16 weights once
            return {"bytes": rows * (4 * surrogate.N_FEATURES + 4) + 2 * params, "flops": 2.0 * rows * weights}
        # forward, weight gradients, input gradients of all layers but the first
        flops = rows * (6.0 * weights - 2.0 * surrogate.N_FEATURES * surrogate.HIDDEN)
        if kind == "gradients":
            return {"bytes": rows * (4 * surrogate.N_FEATURES + 4) + 6 * params, "flops": flops}
        # each step reads and writes the FP32 weights and two moments
        return {"bytes": rows * (4 * surrogate.N_FEATURES + 4) + 24.0 * params * case["batches"], "flops": flops}
    if kind == "batch":
        sizes = _structures(case, random.Random(0))
        phonons = sum(p["phonons"] for p in sizes)
        sensors = sum(p["n_sensors"] for p in sizes)
        every_step = case["type"] == 1
    else:
        phonons = case["phonons"]
        sensors = case["sensors"] if kind == "bar" else 40 if kind == "lshape" else 30
        every_step = kind == "film" or (kind == "lshape" and case["type"] == 1)
    recorded = case["steps"] if every_step else 0.1 * case["steps"]
    life = min(case["sim_ns"], LIFE[kind] * math.sqrt(case["sim_ns"]))
    rate = RATE[kind] + (3.0 * sensors if kind == "bar" else 0.0)
    # counts and fluxes of every sensor and recorded step, raw and interpreted; the model once
    out = (24.0 if case.get("graph") else 48.0) * sensors * recorded
    return {"bytes": out + 1000.0 * sensors, "flops": FP64_PER_EVENT * phonons * life * rate}


def _forward64(x, layers):
    acts = [x]
    for i, (w, b) in enumerate(layers):
        z = acts[-1] @ w + b
        acts.append(torch.relu(z) if i + 1 < len(layers) else z)
    return acts


def exact(case: dict, seed: int):
    """Surrogate outputs in float64 of the FP32 weights and inputs; a Monte Carlo run has no such
    value (its tallies are sums over random trajectories), nor has a training run through Adam."""
    if case["kind"] not in ("predict", "gradients"):
        return None
    state = prepare(case, seed)
    net = state["net"]
    layers = [(torch.from_numpy(w.astype(np.float64)).cuda(), torch.from_numpy(b.astype(np.float64)).cuda())
              for w, b in net.layer_views(net.params())]
    x = torch.from_numpy(state["x"].astype(np.float64)).cuda()
    if case["kind"] == "predict":
        return torch.cat([_forward64(x[i:i + 16384], layers)[-1][:, 0] for i in range(0, len(x), 16384)])
    t = torch.from_numpy(state["t"].astype(np.float64)).cuda()
    acts = _forward64(x, layers)
    d = acts[-1][:, 0] - t
    dz = torch.zeros_like(acts[-1])
    dz[:, 0] = 2.0 * d / len(x)
    grads = []
    for i in range(len(layers) - 1, -1, -1):
        grads.append((acts[i].t() @ dz, dz.sum(0)))
        if i:
            dz = (dz @ layers[i][0].t()) * (acts[i] > 0)
    grad = torch.cat([torch.cat([w.reshape(-1), b]) for w, b in reversed(grads)])
    return {"loss": float((d * d).mean()), "grad": grad}
