"""The workloads whose speed matters, as single passes through the public API.

A case is one of five things a program does with this framework:

  tick     the reference's own loop (Simulator::sim_tick): a move dispatch and a collision
           dispatch, each waited for, then the whole entity buffer read back for the renderer.
           Library-default options, the reference's constant speed and its 10 m radius.
  run      one map advanced by many fused ticks, then the entities and the pair counts read.
  batch    many independent scenarios advanced together, then every scenario's state read.
  grad     one calibration step: a differentiable run of every scenario and its adjoint.
  predict  a differentiable run alone (what a calibration compares its observations with).

A pass continues from where the handle's last pass ended, as such programs do; the differentiable
ones start from the handle's initial state every time.  The maps are the package's own generators;
the agents come from the seed.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "movement-sim_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import msim  # noqa: E402
from msim import autotune  # noqa: E402
from msim import scenarios as S  # noqa: E402
from msim.adjoint import DiffRun  # noqa: E402

NODE_SPACING = 1000.0 / 31.0  # metres between lattice nodes, as in every lattice workload of the package
WARM_TICKS = 1  # the insert-only first tick, made before a program's loop

# The tuner's choices for the workload shapes it was run on (msim/tuned.json): the small map keeps
# the classic layout, everything larger the bucket-sorted state.
TUNED_SMALL = {"binning": 1, "collide_mode": 2, "reorder_interval": 32, "segment_log2": 12, "table_width_log2": 8}
TUNED_CITY = {"binning": 3, "bin_unroll": 2, "segment_log2": 11, "table_width_log2": 8, "graph_ticks": 100}
TUNED_DENSE = {"binning": 3, "bin_unroll": 4, "segment_log2": 12, "graph_ticks": 100}
TUNED_BATCH = {"binning": 3, "segment_log2": 12, "graph_ticks": 50}
LAYOUTS = {"library": {}, "untuned": dict(autotune.DEFAULT), "small": TUNED_SMALL, "city": TUNED_CITY,
           "dense": TUNED_DENSE, "batch": TUNED_BATCH, "batch-untuned": dict(autotune.BATCH_DEFAULT)}


def listed():
    return [
        # The smallest interactive run: launches, waits and one 640 KB readback per tick.
        {"name": "tick-10k", "kind": "tick", "agents": 10_000, "nodes": 1_024, "radius": 10.0, "layout": "library"},
        # The reference's compile-time agent count, one rendered tick.
        {"name": "tick-1M", "kind": "tick", "agents": 1_000_000, "nodes": 150_000, "radius": 10.0,
         "layout": "library"},
        # The plain small benchmark between two looks at it.
        {"name": "run-10k", "kind": "run", "agents": 10_000, "nodes": 1_024, "radius": 1.0, "layout": "small",
         "ticks": 200, "map": "lattice", "zipf": False, "read": "state"},
        # A town of no special size, nobody having tuned anything, cells larger than a metre.
        {"name": "run-123k", "kind": "run", "agents": 123_457, "nodes": 17_003, "radius": 2.5, "layout": "untuned",
         "ticks": 150, "map": "lattice", "zipf": False, "read": "state"},
        # The city-scale benchmark.
        {"name": "run-1M-city", "kind": "run", "agents": 1_000_000, "nodes": 150_000, "radius": 1.0, "layout": "city",
         "ticks": 500, "map": "city", "zipf": False, "read": "entities"},
        # The dense stress benchmark at half its size: skewed road occupancy, crowded cells.
        {"name": "run-8M-dense", "kind": "run", "agents": 8_000_000, "nodes": 490_000, "radius": 1.0,
         "layout": "dense", "ticks": 200, "map": "lattice", "zipf": True, "read": "entities"},
        # A handful of villages together, untuned: launch latency shared by 16 scenarios.
        {"name": "batch-16", "kind": "batch", "scenarios": 16, "agents_lo": 1_000, "agents_hi": 20_000,
         "radius": 1.0, "layout": "batch-untuned", "ticks": 200},
        # The batched benchmark's ragged sizes, an eighth of its scenarios.
        {"name": "batch-64", "kind": "batch", "scenarios": 64, "agents_lo": 1_000, "agents_hi": 500_000,
         "radius": 1.0, "layout": "batch", "ticks": 200},
        # Calibration while it is being set up, on toy scenarios: many small launches.
        {"name": "grad-3k", "kind": "grad", "scenarios": 2, "agents": 1_501, "nodes": 400, "radius": 1.0,
         "ticks": 40, "every": 20, "alpha": 0.02, "arrivals": "frozen"},
        # The calibration benchmark's scenarios, fewer of them and a tenth of its ticks.
        {"name": "grad-800k", "kind": "grad", "scenarios": 8, "agents": 100_000, "nodes": 20_000, "radius": 1.0,
         "ticks": 100, "every": 50, "alpha": 0.01, "arrivals": "carry"},
        # The hidden run a calibration observes, odd sizes and a wider radius.
        {"name": "predict-350k", "kind": "predict", "scenarios": 7, "agents": 50_021, "nodes": 10_000,
         "radius": 2.0, "ticks": 150, "every": 50, "alpha": 0.02},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tick", "run", "run", "batch", "grad", "predict"])
    if kind == "tick":
        n = _log_int(rng, 1_000, 1_000_000)
        return {"kind": kind, "agents": n, "nodes": max(64, n // rng.randint(5, 12)),
                "radius": rng.choice([1.0, 2.5, 10.0]), "layout": "library"}
    if kind == "run":
        n = _log_int(rng, 5_000, 4_000_000)
        layout = rng.choice(["small", "untuned"] if n < 60_000 else ["untuned", "city", "dense"])
        return {"kind": kind, "agents": n, "nodes": max(64, n // rng.randint(5, 16)),
                "radius": rng.choice([0.75, 1.0, 2.5]), "layout": layout, "ticks": rng.randint(60, 300),
                "map": "lattice", "zipf": rng.random() < 0.3, "read": rng.choice(["state", "entities"])}
    if kind == "batch":
        lo = _log_int(rng, 200, 5_000)
        return {"kind": kind, "scenarios": rng.randint(3, 40), "agents_lo": lo,
                "agents_hi": lo * rng.randint(2, 40), "radius": rng.choice([1.0, 2.5]),
                "layout": rng.choice(["batch", "batch-untuned"]), "ticks": rng.randint(60, 220)}
    agents = _log_int(rng, 500, 60_000)
    case = {"kind": kind, "scenarios": rng.randint(1, 8), "agents": agents, "nodes": max(64, agents // rng.randint(4, 8)),
            "radius": rng.choice([1.0, 1.5]), "ticks": rng.randint(20, 90), "every": rng.randint(10, 50),
            "alpha": rng.choice([0.0, 0.01, 0.02])}
    if kind == "grad":
        case["arrivals"] = rng.choice(["frozen", "carry"])
    return case


# ---- inputs -----------------------------------------------------------------

_maps = {}


def _map(kind, nodes):
    """(roads, connections, side length) of the map every seed of a case shares."""
    if (kind, nodes) not in _maps:
        if kind == "city":
            size = 12_000.0 * math.sqrt(nodes / 150_000)
            xy, edges = S.city_graph(n_nodes=nodes, size=size, sigma=size / 8.0, seed=S.MASTER_SEED + 2)
        else:
            side = max(4, int(round(math.sqrt(nodes))))
            size = NODE_SPACING * (side - 1)
            xy, edges = S.lattice_graph(side=side, size=size, seed=nodes)
        _maps[kind, nodes] = S.build_roads(xy, edges) + (size,)
    return _maps[kind, nodes]


def _agents(roads, n, seed, zipf=False):
    """(entities, speeds) of n agents as scenarios.place_agents draws them, drawn on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dev = torch.device("cuda")

    def uniform(*shape):
        return torch.rand(*shape, generator=g, device=dev)

    n_roads = roads.shape[0]
    if zipf:
        w = (torch.arange(1, n_roads + 1, device=dev, dtype=torch.float64) + S.ZIPF_Q) ** -1.1
        cdf = torch.cumsum(w, 0)
        rank = torch.searchsorted(cdf / cdf[-1], torch.rand(n, generator=g, device=dev, dtype=torch.float64))
        road = torch.randperm(n_roads, generator=g, device=dev)[rank.clamp_(max=n_roads - 1)]
    else:
        road = torch.randint(n_roads, (n,), generator=g, device=dev)
    ends = torch.from_numpy(np.concatenate([roads["start_pos"], roads["end_pos"]], axis=1)).to(dev)[road]
    a, b = ends[:, :2], ends[:, 2:]
    rec = torch.zeros(n, 16, device=dev)
    rec[:, 0:3] = uniform(n, 3)
    rec[:, 3] = 1.0
    rec[:, 8:10] = a + (b - a) * uniform(n, 1)
    rec[:, 10:12] = torch.where(uniform(n, 1) < 0.5, a, b)
    words = rec.view(torch.int32)
    words[:, 4:8] = torch.randint(-(1 << 31), 1 << 31, (n, 4), generator=g, device=dev, dtype=torch.int32)
    words[:, 14] = road.to(torch.int32)
    speed = 0.8 + 0.8 * uniform(n)
    return rec.cpu().numpy().view(msim.ENTITY_DTYPE).reshape(n), speed.cpu().numpy()


def _batch_sizes(case):
    """Agents and nodes of every scenario: log-uniform, the same for every seed."""
    rng = np.random.default_rng(case["scenarios"])
    lo, hi = math.log(case["agents_lo"]), math.log(case["agents_hi"])
    agents = np.exp(rng.uniform(lo, hi, case["scenarios"])).astype(int)
    return [(int(n), max(64, int(n / rng.uniform(2.0, 8.0)))) for n in agents]


def _scenarios(case, seed):
    """The case's scenarios: one for tick and run, several for the rest."""
    kind = case["kind"]
    if kind in ("tick", "run"):
        sizes = [(case["agents"], case["nodes"])]
    elif kind == "batch":
        sizes = _batch_sizes(case)
    else:
        sizes = [(case["agents"], case["nodes"])] * case["scenarios"]
    out = []
    for k, (n, nodes) in enumerate(sizes):
        roads, conns, size = _map(case.get("map", "lattice"), nodes)
        ents, speed = _agents(roads, n, 1000 * seed + k, case.get("zipf", False))
        # the reference's agents all walk at its constant speed
        out.append(S.Scenario(kind, roads, conns, ents, None if kind == "tick" else speed,
                              msim.push_consts(size, size, case["radius"]), 0, (size, size)))
    return out


def prepare(case, seed):
    torch.cuda.init()
    scs = _scenarios(case, seed)
    kind = case["kind"]
    if kind in ("tick", "run"):
        sc = scs[0]
        sim = msim.Simulation(sc.roads, sc.conns, sc.entities, sc.pc, speed=sc.speed, **LAYOUTS[case["layout"]])
        sim.run_ticks(WARM_TICKS)
        sim.sync()
        return {"case": case, "sim": sim}
    if kind == "batch":
        b = msim.Batch(scs, **LAYOUTS[case["layout"]])
        b.run_ticks(WARM_TICKS)
        b.sync()
        return {"case": case, "batch": b}
    b = msim.Batch(scs)
    diff = DiffRun(b, case["ticks"], checkpoint_every=case["every"], arrival_gradient=case.get("arrivals", "frozen"))
    theta, alpha, observed = _parameters(case, seed, scs)
    grad = kind == "grad"
    return {"case": case, "diff": diff, "theta": theta.cuda().requires_grad_(grad),
            "alpha": alpha.cuda().requires_grad_(grad), "observed": observed.cuda()}


def _parameters(case, seed, scs):
    """theta per map road tied over the scenarios, alpha, and the positions a calibration observes."""
    g = torch.Generator().manual_seed(seed)
    theta = torch.exp(0.2 * torch.randn(scs[0].roads.shape[0], generator=g))
    start = torch.from_numpy(np.concatenate([sc.entities["pos"] for sc in scs]))
    observed = start + 25.0 * torch.randn(start.shape, generator=g)
    return theta, torch.tensor(case["alpha"]), observed


# ---- one pass ---------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "tick":
        sim = state["sim"]
        sim.dispatch()
        sim.sync()
        sim.dispatch()
        sim.sync()
        return _fields(sim.entities())
    if kind == "run":
        sim = state["sim"]
        sim.run_ticks(case["ticks"])
        out = sim.state() if case["read"] == "state" else _fields(sim.entities())
        total, per_tick = sim.pairs(case["ticks"])
        return dict(out, pairs=np.int64(total), pairs_per_tick=per_tick)
    if kind == "batch":
        b = state["batch"]
        b.run_ticks(case["ticks"])
        states = [b.state(s) for s in range(b.n_scen)]
        total, last = b.pairs()
        out = {k: np.concatenate([st[k] for st in states]) for k in states[0]}
        return dict(out, pairs=total.astype(np.int64), pairs_last=last)
    theta, alpha = state["theta"], state["alpha"]
    pos = state["diff"](theta.repeat(case["scenarios"]), alpha)
    if kind == "predict":
        return {"pos": pos}
    loss = ((pos - state["observed"]) ** 2).sum(dim=1).mean()
    g_theta, g_alpha = torch.autograd.grad(loss, (theta, alpha))
    return {"pos": pos.detach(), "loss": loss.detach(), "theta": g_theta, "alpha": g_alpha}


def _fields(ents):
    return {k: ents[k] for k in ents.dtype.names}


def _agent_ticks(case):
    kind = case["kind"]
    if kind == "tick":
        return case["agents"], 1
    if kind == "run":
        return case["agents"], case["ticks"]
    if kind == "batch":
        return sum(n for n, _ in _batch_sizes(case)), case["ticks"]
    return case["agents"] * case["scenarios"], case["ticks"]


def work(case):
    """Per agent and tick: position, target and speed read, position and neighbour count written (32 B),
    about 30 operations for the step and the nearest neighbours; per agent and pass the 48 or 64 bytes read
    back.  The adjoint reads a tick's position, target, road and speed, and reads and writes its two
    binary64 adjoint values (60 B, about 60 operations)."""
    n, ticks = _agent_ticks(case)
    kind = case["kind"]
    moved, ops = 32.0, 30.0
    back = {"tick": 64.0, "run": 64.0 if case.get("read") == "entities" else 48.0, "batch": 48.0}.get(kind, 8.0)
    if kind == "grad":
        moved, ops = moved + 60.0, ops + 60.0
    return {"bytes": n * (ticks * moved + back), "flops": n * ticks * ops}


# ---- what a pass returns, in 64 bits ----------------------------------------

EXACT_AGENT_TICKS = 30_000_000
EXACT_DIFF_AGENTS = 3_000  # pairs are found over all agents of a scenario
EXACT_DIFF_TICKS = 60


def exact(case, seed):
    n, ticks = _agent_ticks(case)
    if case["kind"] in ("grad", "predict"):
        if case["agents"] > EXACT_DIFF_AGENTS or ticks > EXACT_DIFF_TICKS:
            return None
        return _exact_diff(case, seed)
    if n * ticks > EXACT_AGENT_TICKS:
        return None
    parts = [_walk(sc, ticks) for sc in _scenarios(case, seed)]
    pos, tgt, head = (np.concatenate([p[k] for p in parts]) for k in range(3))
    if case["kind"] == "batch" or case.get("read") == "state":
        return {"pos": pos, "tgt": tgt, "dir": head, "road": None, "rng": None, "ncount": None, "pairs": None}
    return {"pos": pos, "target": tgt, "direction": head}


def _walk(sc, ticks):
    """Positions, targets and headings after `ticks` moves.  The positions are carried in 64 bits beside the
    32-bit walk that takes the decisions (arrivals, draws), which are defined on 32-bit values."""
    n = sc.entities.shape[0]
    f = np.float32
    p = sc.entities["pos"].astype(f)
    t = sc.entities["target"].astype(f)
    road = sc.entities["roadIndex"].astype(np.int64)
    rng = sc.entities["randomState"].astype(np.uint32)
    speed = np.full(n, 1.4, f) if sc.speed is None else sc.speed.astype(f)
    exact_pos = p.astype(np.float64)
    head = np.zeros((n, 2))
    s64 = speed.astype(np.float64)[:, None]
    for _ in range(ticks):
        d = t - p
        length = np.sqrt(d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1])
        go = length > speed
        with np.errstate(invalid="ignore", divide="ignore"):
            p = np.where(go[:, None], p + (d / length[:, None]) * speed[:, None], t)
            head = _heading(exact_pos, t, s64)
        exact_pos = np.where(go[:, None], exact_pos + head, t)
        at = np.flatnonzero(~go)
        t[at], road[at], rng[at] = _route(sc, t[at], road[at], rng[at])
        head[at] = _heading(exact_pos[at], t[at].astype(np.float64), s64[at])
    return exact_pos, t.astype(np.float64), head


def _heading(p, t, speed):
    d = t - p
    length = np.sqrt((d * d).sum(1, keepdims=True))
    return np.where(length > 0, d / np.where(length > 0, length, 1.0), 0.0) * speed


def _route(sc, at, road, rng):
    """The route choice of agents that stand on their targets `at`."""
    roads = sc.roads
    at_start = (at == roads["start_pos"][road]).all(1)
    count = np.where(at_start, roads["start_count"][road], roads["end_count"][road]).astype(np.int64)
    index = np.where(at_start, roads["start_index"][road], roads["end_index"][road]).astype(np.int64)
    drawn = count > 2
    # one xorshift128 step for those that draw
    old = rng.copy()
    u = rng[:, 3].copy()
    u ^= u << np.uint32(11)
    u ^= u >> np.uint32(8)
    x = u ^ old[:, 0] ^ (old[:, 0] >> np.uint32(19))
    rng[drawn, 1:] = old[drawn, :3]
    rng[drawn, 0] = x[drawn]
    frac = x.astype(np.float32) * np.float32(2.3283064365386963e-10)
    offset = np.ceil(np.float32(1.0) + frac * count.astype(np.float32)).astype(np.int64) - 1
    offset = np.where(drawn, offset, 1)
    nxt = np.where(count > 1, sc.conns[np.where(count > 1, index + offset, 0)].astype(np.int64), road)
    start, end = roads["start_pos"][nxt], roads["end_pos"][nxt]
    leaves_start = (at == start).all(1)
    return np.where(leaves_start[:, None], end, start), nxt, rng


def _exact_diff(case, seed):
    """The differentiable run in 64 bits, its gradient by torch's autograd over the run."""
    scs = _scenarios(case, seed)
    theta, alpha, observed = _parameters(case, seed, scs)
    theta = theta.double().requires_grad_(True)
    alpha = alpha.double().requires_grad_(True)
    carry = case.get("arrivals") == "carry"
    final = []
    for sc in scs:
        p = torch.from_numpy(sc.entities["pos"].astype(np.float64))
        t = sc.entities["target"].astype(np.float32)
        road = sc.entities["roadIndex"].astype(np.int64)
        rng = sc.entities["randomState"].astype(np.uint32)
        v = torch.from_numpy(sc.speed.astype(np.float64))
        for tick in range(case["ticks"]):
            if tick:  # the first tick only enters the agents
                T = torch.from_numpy(t.astype(np.float64))
                s = v * theta[torch.from_numpy(road)]
                d = T - p
                length = d.square().sum(1).sqrt()
                arrived = (length <= s).detach()
                safe = torch.where(length > 0, length, torch.ones_like(length))
                moved = p + d / safe[:, None] * s[:, None]
                at = np.flatnonzero(arrived.numpy())
                t[at], new_road, rng[at] = _route(sc, t[at], road[at], rng[at])
                snapped = T
                if carry and at.size:
                    road[at] = new_road
                    T2 = torch.from_numpy(t.astype(np.float64))
                    e = T2 - T
                    u2 = e / e.square().sum(1).sqrt().clamp_min(1e-300)[:, None]
                    left = (1 - length / s) * v * theta[torch.from_numpy(road)]
                    over = torch.where(arrived[:, None], left[:, None] * u2, torch.zeros_like(T))
                    snapped = T + (over - over.detach())
                road[at] = new_road
                p = torch.where(arrived[:, None], snapped, moved)
            p = p + alpha * _push(p, case["radius"])
        final.append(p)
    pos = torch.cat(final)
    if case["kind"] == "predict":
        return {"pos": pos.detach()}
    loss = ((pos - observed.double()) ** 2).sum(1).mean()
    g = torch.autograd.grad(loss, (theta, alpha))
    return {"pos": pos.detach(), "loss": loss.detach(), "theta": g[0], "alpha": g[1]}


def _push(p, radius):
    """Sum over each agent's neighbours of (1 - |x|^2 / R^2)^3 x."""
    with torch.no_grad():
        i, j = torch.nonzero(torch.cdist(p, p) < radius * 1.001, as_tuple=True)
        i, j = i[i != j], j[i != j]
    x = p[i] - p[j]
    h = 1 - x.square().sum(1) / radius ** 2
    w = torch.where(h > 0, h, torch.zeros_like(h)) ** 3
    return torch.zeros_like(p).index_add(0, i, w[:, None] * x)
