"""Timed cases of the framework: the work its users have it do, through the public entry points.

    listed()             the cases, as plain dicts
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what a program holds before the call: the configuration, buffers, weights
    run(state)           one pass through the entry points; returns the outputs
    work(case)           the bytes and floating-point operations a pass cannot do without
    exact(case, seed)    the outputs of the floating-point cases computed in 64 bits

The kinds of work:
    standalone  EngineApp.start_standalone: configuration in, epicurve CSV and interventions
                report out, the way the command line runs one region.
    region      Simulation + one step() call over the whole run + the final citizen states: a
                program that embeds one region. Small, ordinary and very large populations.
    calls       the same with the hours asked for in calls of a fixed length, as a program that
                reports progress or a listener that takes every hour's row as it is made.
    ensemble    Batch: independent replicates in shared launches; rows of every replicate.
    states      the citizen-state message of the current hour formatted into device memory.
    train       Adam steps of the surrogate network on host mini-batches, then its parameters.
    predict     the surrogate network's answers for a set of parameter points.
"""
import copy
import ctypes
import math
import tempfile

import numpy as np
import torch

import epirust_amd as G
from epirust_amd import surrogate

# The disease, work and transport parameters of the framework's own 10k, 1M and 10M-agent
# configurations; a case sets the sizes, the hours, the starting infections and the interventions.
BASE = {
    "population": {"Auto": {"number_of_agents": 0, "public_transport_percentage": 0.2, "working_percentage": 0.7}},
    "disease": {"regular_transmission_start_day": 5, "high_transmission_start_day": 20, "last_day": 23,
                "asymptomatic_last_day": 9, "mild_infected_last_day": 12, "regular_transmission_rate": 0.025,
                "high_transmission_rate": 0.25, "death_rate": 0.2, "percentage_asymptomatic_population": 0.3,
                "percentage_severe_infected_population": 0.3, "exposed_duration": 48, "pre_symptomatic_duration": 48},
    "geography_parameters": {"grid_size": 0, "hospital_beds_percentage": 0.003},
    "hours": 0,
    "interventions": [],
    "starting_infections": {"exposed": 0, "infected_mild_asymptomatic": 0, "infected_mild_symptomatic": 0,
                            "infected_severe": 0},
}
INPUTS, OUTPUTS = 9, 600  # of the surrogate: parameters of a point; 100 days x 6 compartments


def listed():
    return [
        # The smallest whole run: the 10,000-agent configuration from JSON to CSV. Every launch
        # and every host step shows; the kernels themselves are tiny.
        {"name": "standalone_10k", "kind": "standalone", "agents": 10000, "grid": 250, "hours": 2400, "exposed": 20,
         "lockdown": 0, "hospital": 0, "vaccinate_from": 0},
        # One region of the surrogate's sweep: an ordinary size with a lockdown and daily vaccination.
        {"name": "region_100k_interventions", "kind": "region", "agents": 100000, "grid": 632, "hours": 2400,
         "exposed": 50, "lockdown": 1000, "hospital": 0, "vaccinate_from": 720},
        # The headline workload: 1,000,000 agents on 2000 x 2000, 2,399 hours.
        {"name": "region_1m", "kind": "region", "agents": 1000000, "grid": 2000, "hours": 2400, "exposed": 10,
         "lockdown": 0, "hospital": 0, "vaccinate_from": 0},
        # The largest region: 10,000,000 agents on 6000 x 6000 with lockdown, hospital growth and
        # daily vaccination, 60 days.
        {"name": "region_10m_interventions", "kind": "region", "agents": 10000000, "grid": 6000, "hours": 1440,
         "exposed": 20000, "lockdown": 100000, "hospital": 10000, "vaccinate_from": 720},
        # A large odd-sized region stepped in calls of 50 hours: most calls begin and end inside a day.
        {"name": "calls_333k_by_50h", "kind": "calls", "agents": 333331, "grid": 1171, "hours": 601, "call": 50,
         "exposed": 100, "lockdown": 0, "hospital": 0, "vaccinate_from": 0},
        # Hour at a time: every row handed to the program's listeners as it is made.
        {"name": "hourly_1m", "kind": "calls", "agents": 1000000, "grid": 2000, "hours": 241, "call": 1, "exposed": 10,
         "lockdown": 0, "hospital": 0, "vaccinate_from": 0},
        {"name": "hourly_20k", "kind": "calls", "agents": 19997, "grid": 283, "hours": 241, "call": 1, "exposed": 20,
         "lockdown": 0, "hospital": 0, "vaccinate_from": 0},
        # The judged ensemble of one sweep point: 32 seeds of a 100,000-agent region.
        {"name": "ensemble_32x100k", "kind": "ensemble", "sims": 32, "agents_from": 100000, "agents_to": 100000,
         "hours": 2400, "exposed": 50, "lockdown": 1000, "hospital": 0, "vaccinate_from": 720},
        # 64 replicates of mixed sizes, 20,000 to 500,000 agents.
        {"name": "replicates_64_mixed", "kind": "ensemble", "sims": 64, "agents_from": 20000, "agents_to": 500000,
         "hours": 2400, "exposed": 20, "lockdown": 0, "hospital": 0, "vaccinate_from": 0},
        # One hour's citizen-state message at 1,000,000 agents.
        {"name": "states_1m", "kind": "states", "agents": 1000000, "grid": 2000, "hours": 2400, "exposed": 1000,
         "lockdown": 0, "hospital": 0, "vaccinate_from": 0},
        # One epoch of the surrogate's training set of 6,144 points: 12 Adam steps of 512.
        {"name": "surrogate_epoch_512", "kind": "train", "batch": 512, "steps": 12, "hidden": 512, "layers": 4},
        # The surrogate's answers for its 500 held-out points.
        {"name": "surrogate_predict_500", "kind": "predict", "points": 500, "hidden": 512, "layers": 4},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["region", "region", "region", "standalone", "calls", "calls", "ensemble", "ensemble", "states",
                       "train", "predict"])
    if kind == "train":
        return {"kind": kind, "batch": _log_uniform(rng, 64, 1024), "steps": rng.randint(4, 16),
                "hidden": 8 * rng.randint(16, 64), "layers": rng.randint(2, 4)}
    if kind == "predict":
        return {"kind": kind, "points": _log_uniform(rng, 1, 4096), "hidden": 8 * rng.randint(16, 64),
                "layers": rng.randint(2, 4)}
    if kind == "ensemble":
        sims = _log_uniform(rng, 4, 64)
        lo = _log_uniform(rng, 10000, 100000)
        hi = min(500000, lo * rng.randint(1, 5))
        return {"kind": kind, "sims": sims, "agents_from": lo, "agents_to": hi, "hours": rng.randint(480, 2400),
                "exposed": rng.randint(20, 100), "lockdown": rng.choice([0, lo // 100]), "hospital": 0,
                "vaccinate_from": rng.choice([0, 24 * rng.randint(10, 30)])}
    top = {"region": 10000000, "standalone": 100000, "calls": 1000000, "states": 4000000}[kind]
    n = _log_uniform(rng, {"region": 20000, "standalone": 3000, "calls": 3000, "states": 10000}[kind], top)
    case = {"kind": kind, "agents": n, "grid": int(round(rng.uniform(1.95, 2.5) * math.sqrt(n))),
            "exposed": max(20, n // rng.randint(500, 5000)), "lockdown": rng.choice([0, max(20, n // 100)]),
            "hospital": rng.choice([0, max(10, n // 1000)]),
            "vaccinate_from": rng.choice([0, rng.randint(100, 900)])}
    if kind == "calls":
        case["call"] = rng.choice([1, 1, _log_uniform(rng, 2, 200)])
        case["hours"] = (96 if case["call"] == 1 else 240) + rng.randint(1, 240)
    elif kind == "states":
        case["hours"] = 2400
    else:
        case["hours"] = min(rng.randint(480, 2400), max(120, int(1.2e10 / n)))
    return case


def _config(case, agents, grid, seed, rate=1.0):
    c = copy.deepcopy(BASE)
    c["population"]["Auto"]["number_of_agents"] = agents
    c["geography_parameters"]["grid_size"] = grid
    c["hours"] = case["hours"]
    c["starting_infections"]["exposed"] = case["exposed"]
    c["disease"]["regular_transmission_rate"] *= rate
    c["disease"]["high_transmission_rate"] *= rate
    if case["lockdown"]:
        c["interventions"].append({"Lockdown": {"at_number_of_infections": case["lockdown"],
                                                "essential_workers_population": 0.1}})
    if case["hospital"]:
        c["interventions"].append({"BuildNewHospital": {"spread_rate_threshold": case["hospital"]}})
    if case["vaccinate_from"]:
        c["interventions"] += [{"Vaccinate": {"at_hour": h, "percent": 0.001}}
                               for h in range(case["vaccinate_from"], case["hours"], 24)]
    c["seed"] = seed
    return c


def _sizes(case):
    """The replicates' populations, spread evenly over the logarithm of the range, odd sizes among them."""
    lo, hi, k = math.log(case["agents_from"]), math.log(case["agents_to"]), case["sims"]
    return [int(round(math.exp(lo + (hi - lo) * ((i * 37) % k) / max(k - 1, 1)))) for i in range(k)]


def _widths(case):
    return [INPUTS] + [case["hidden"]] * case["layers"] + [OUTPUTS]


def _network(case, seed):
    """He-normal weights and small biases, flattened W0, b0, W1, b1, ... as the library keeps them."""
    rng, w, parts = np.random.default_rng(seed), _widths(case), []
    for k, n in zip(w[:-1], w[1:]):
        parts += [rng.standard_normal(k * n) * math.sqrt(2.0 / k), 0.01 * rng.standard_normal(n)]
    return np.concatenate(parts).astype(np.float32)


def _points(n, seed):
    """Points of the unit cube and standardized curves, as the surrogate's fit hands them to its networks."""
    rng = np.random.default_rng(seed + 1)
    x = rng.random((n, INPUTS)).astype(np.float32)
    # smooth in the point, unit variance, plus one run's noise
    phase = x @ rng.standard_normal((INPUTS, 6)).astype(np.float32)
    day = np.linspace(0.0, 3.0, OUTPUTS // 6, dtype=np.float32)
    t = np.sqrt(2.0) * np.sin(phase[:, None, :] + day[None, :, None]).reshape(n, OUTPUTS)
    return x, (t + 0.1 * rng.standard_normal((n, OUTPUTS))).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "seed": seed}
    if kind == "train":
        s["x"], s["t"] = _points(case["batch"] * case["steps"], seed)
        s["net"] = surrogate.MLP(_widths(case), seed=seed, max_batch=max(case["batch"], 1024))
        s["net"].set_params(_network(case, seed))
    elif kind == "predict":
        s["x"], _ = _points(case["points"], seed)
        s["net"] = surrogate.MLP(_widths(case), seed=seed)
        s["net"].set_params(_network(case, seed))
    elif kind == "ensemble":
        rng = np.random.default_rng(seed)
        s["configs"] = [_config(case, n, int(round(2.0 * math.sqrt(n))), seed + i, float(rng.uniform(0.8, 1.6)))
                        for i, n in enumerate(_sizes(case))]
    else:
        s["config"] = _config(case, case["agents"], case["grid"], seed)
        if kind == "standalone":
            s["dir"] = tempfile.mkdtemp()
        if kind != "standalone":
            # the longest record: {"citizen_id":"","state":"?","location":{"x":,"y":}} and a comma, id and cell digits
            longest = 54 + len(str(case["agents"])) + 2 * len(str(case["grid"] + 1))
            s["text"] = torch.zeros(case["agents"] * longest, dtype=torch.uint8, device="cuda")
            s["length"] = torch.zeros(1, dtype=torch.int64, device="cuda")
        if kind == "states":
            s["sim"] = G.Simulation(s["config"])
            s["sim"].step(68)  # an evening hour: the population is spread over houses and transport
        torch.cuda.synchronize()
    return s


def _text(s, sim):
    """The current hour's citizen-state records in the program's own device buffer, and their length."""
    L = G.lib()
    rc = L.epi_citizen_states_text_noalloc(sim._h, s["text"].data_ptr(), s["text"].numel(), s["length"].data_ptr())
    if rc:
        raise G.EpiError(rc, L.epi_last_error().decode())
    return {"text": s["text"], "length": s["length"]}


def _whole(values, count):
    """A result table of the run's full length: a run that stops early leaves the rest empty."""
    table = np.zeros((count,) + values.shape[1:], dtype=values.dtype)
    table[: len(values)] = values
    return table


def _report(s, sim, rows):
    case = s["case"]
    events = np.array(sim.events(), dtype=np.uint32).reshape(-1, 2)
    return {"rows": _whole(rows, case["hours"] - 1), "events": _whole(events, 16 + case["hours"] // 12),
            "states": _text(s, sim)}


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "standalone":
        csv = G.EngineApp.start_standalone(s["config"], s["dir"])
        report = np.fromfile(csv[: -len(".csv")] + "_interventions.json", dtype=np.uint8)
        return {"csv": _whole(np.fromfile(csv, dtype=np.uint8), 64 * case["hours"]),
                "interventions": _whole(report, 1024 + 8 * case["hours"])}
    if kind == "region":
        with G.Simulation(s["config"]) as sim:
            rows, _ = sim.step(case["hours"] - 1)
            return _report(s, sim, rows)
    if kind == "calls":
        with G.Simulation(s["config"]) as sim:
            rows, stopped = [], False
            while not stopped:
                got, stopped = sim.step(case["call"])
                rows.append(got)
            return _report(s, sim, np.concatenate(rows))
    if kind == "ensemble":
        with G.Batch(s["configs"]) as batch:
            rows, _ = batch.step(case["hours"] - 1)
        return {"rows": np.stack([_whole(r, case["hours"] - 1) for r in rows])}
    if kind == "states":
        return _text(s, s["sim"])
    if kind == "train":
        b = case["batch"]
        loss = [s["net"].train_step(s["x"][k * b:(k + 1) * b], s["t"][k * b:(k + 1) * b], 1e-3)
                for k in range(case["steps"])]
        return {"loss": np.array(loss, dtype=np.float32), "params": s["net"].params()}
    return {"curves": s["net"].forward(s["x"])}


def work(case):
    kind = case["kind"]
    if kind in ("train", "predict"):
        w = _widths(case)
        params = sum(k * n + n for k, n in zip(w[:-1], w[1:]))
        io = 4 * (INPUTS + OUTPUTS)
        if kind == "predict":
            return {"bytes": 2.0 * params + io * case["points"], "flops": 2.0 * params * case["points"]}
        # forward, input gradients and weight gradients; weights and both moments read and written
        return {"bytes": case["steps"] * (24.0 * params + io * case["batch"]),
                "flops": 6.0 * params * case["batch"] * case["steps"]}
    if kind == "ensemble":
        agents = sum(_sizes(case))
        cells = sum(int(round(2.0 * math.sqrt(n))) ** 2 for n in _sizes(case))
    else:
        agents, cells = case["agents"], case["grid"] ** 2
    if kind == "states":
        return {"bytes": 8.0 * agents + 62.0 * agents, "flops": 0}
    # An hour reads and writes every agent's cell and state (4 B each) and every cell's
    # occupant (1 B), in the 18 hours of a day in which anyone moves or falls ill.
    return {"bytes": 0.75 * (case["hours"] - 1) * (16.0 * agents + 2.0 * cells), "flops": 0}


def _gelu(z):
    return 0.5 * z * (1.0 + np.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def _gelu_slope(z):
    t = np.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3))
    return 0.5 * (1.0 + t) + 0.5 * z * (1.0 - t * t) * math.sqrt(2.0 / math.pi) * (1.0 + 3.0 * 0.044715 * z * z)


def _layers(case, flat):
    w, at, out = _widths(case), 0, []
    for k, n in zip(w[:-1], w[1:]):
        out.append((flat[at:at + k * n].reshape(k, n), flat[at + k * n:at + k * n + n]))
        at += k * n + n
    return out


def _forward(layers, x):
    a, kept = x, []
    for i, (W, b) in enumerate(layers):
        z = a @ W + b
        kept.append((a, z))
        a = z if i == len(layers) - 1 else _gelu(z)
    return a, kept


def exact(case, seed):
    """Simulations return counts and text, which are whole; the network's outputs in 64 bits."""
    if case["kind"] == "predict":
        x, _ = _points(case["points"], seed)
        layers = _layers(case, _network(case, seed).astype(np.float64))
        return {"curves": _forward(layers, x.astype(np.float64))[0]}
    if case["kind"] != "train":
        return None
    b = case["batch"]
    x, t = (v.astype(np.float64) for v in _points(b * case["steps"], seed))
    p = _network(case, seed).astype(np.float64)
    m, v, losses = np.zeros_like(p), np.zeros_like(p), []
    for k in range(case["steps"]):
        layers = _layers(case, p)
        y, kept = _forward(layers, x[k * b:(k + 1) * b])
        d = y - t[k * b:(k + 1) * b]
        losses.append(np.mean(d * d))
        dz, grads = 2.0 * d / d.size, []
        for i in range(len(layers) - 1, -1, -1):
            grads[:0] = [(kept[i][0].T @ dz).ravel(), dz.sum(axis=0)]
            if i:
                dz = (dz @ layers[i][0].T) * _gelu_slope(kept[i - 1][1])
        g = np.concatenate(grads)
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        p = p - 1e-3 * (m / (1.0 - 0.9 ** (k + 1))) / (np.sqrt(v / (1.0 - 0.999 ** (k + 1))) + 1e-8)
    return {"loss": np.array(losses), "params": p}
