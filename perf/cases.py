"""The work that a program built on this framework has it do, as timed cases.

Five kinds of work:

run       a simulation held by models.Simulation steps some more and its population is read
          back (a logged or watched run, or the end of one)
batch     many simulations of one model stepped together through models.Batch, and every
          population read back
index     the index of a spatial message list (fgx_spatial_build_records), the spatial
          sort of an agent list (fgx_agent_sort) or a bucket index (fgx_bucket_build) on
          device buffers
turnover  deaths and births of one agent list: compaction, then the append of new agents
stats     sum, minimum, maximum and squared deviations of one logged agent variable

Steps are enqueued launch by launch (option "graphs" off), as those of every model with
host functions between its layers are; the kernels are those a captured step replays.

Everything the framework computes is defined to the bit: lists keep a stated order, sums
over neighbours follow the message order, random draws are keyed by agent and step.  A
multi-step run that rounds one sum differently ends in another state, so runs are compared
exactly; only the statistics, sums in double precision whose order is open, have a
tolerance.
"""
import math

import numpy as np
import torch

from flamegpu2_amd import fgx, serving, workloads
from flamegpu2_amd.models import Batch, Simulation

TORCH = {"f32": torch.float32, "f64": torch.float64, "i32": torch.int32, "u32": torch.int32, "i64": torch.int64}
STATS_CODE = {"f32": 0, "f64": 1, "i32": 2, "u32": 3, "i64": 4}
BYTES = {"f32": 4, "f64": 8, "i32": 4, "u32": 4, "i64": 8}


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # the smallest simulation a service admits: launches and latency
        {"name": "boids-1k", "kind": "run", "model": "boids", "n": 1024, "steps": 100},
        # the circles example at its own size
        {"name": "circles-16k", "kind": "run", "model": "circles", "n": 16384, "steps": 50},
        # a population of an odd size watched after every step
        {"name": "circles-watched", "kind": "run", "model": "circles", "n": 50021, "steps": 1},
        # the benchmark's 2^20 boids
        {"name": "boids-1m", "kind": "run", "model": "boids", "n": 1 << 20, "steps": 25},
        # births and deaths every step in a small population
        {"name": "predprey-20k", "kind": "run", "model": "predprey", "n": 20000, "predators": 1999, "width": 150.0, "steps": 20},
        # predator-prey at its configured populations, of which the predators are watched
        {"name": "predprey-1m", "kind": "run", "model": "predprey", "n": 1000000, "predators": 250000, "width": 1000.0, "steps": 10},
        # an ensemble of circles with the bin width its tuner settles on
        {"name": "batch-64", "kind": "batch", "count": 64, "n_lo": 1024, "n_hi": 131072, "steps": 10, "bins_per_radius": 2},
        # the message index of a moving flock: agents in last step's order, about one bin apart
        {"name": "index-3d-1m", "kind": "index", "what": "messages", "dims": 3, "n": 1 << 20, "per_bin": 4.0, "order": "moved"},
        # the index of a large 2-D list that arrives in no order (the first step of a run)
        {"name": "index-2d-8m", "kind": "index", "what": "messages", "dims": 2, "n": 8388593, "per_bin": 25.0, "order": "random"},
        # the spatial sort of an ordinary agent list
        {"name": "sort-250k", "kind": "index", "what": "agents", "dims": 3, "n": 250007, "per_bin": 8.0, "order": "moved"},
        # deaths and births of a large population
        {"name": "turnover-1m", "kind": "turnover", "n": 1000003, "deaths": 0.1, "births": 0.05},
        # one logged variable of the benchmark's population
        {"name": "stats-1m", "kind": "stats", "n": 1 << 20, "dtype": "f32"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "predprey", "batch", "index", "index", "turnover", "stats"])
    if kind == "run":
        steps = 1 if rng.random() < 0.25 else _log(rng, 5, 100)
        n = _log(rng, 1024, min(1 << 20, 25 * (1 << 20) // steps))
        return {"kind": "run", "model": rng.choice(["circles", "boids"]), "n": n, "steps": steps}
    if kind == "predprey":
        n = _log(rng, 5000, 500000)
        return {"kind": "run", "model": "predprey", "n": n, "predators": max(16, int(n * rng.uniform(0.01, 0.25))),
                "width": round(math.sqrt(n) * rng.uniform(0.9, 1.4) / 5.0) * 5.0, "steps": rng.randint(1, 20)}
    if kind == "batch":
        return {"kind": "batch", "count": rng.randint(4, 64), "n_lo": 1024, "n_hi": _log(rng, 8192, 131072),
                "steps": rng.randint(1, 10), "bins_per_radius": rng.choice([1, 2])}
    if kind == "index":
        what = rng.choice(["messages", "messages", "agents", "bucket"])
        return {"kind": "index", "what": what, "dims": 1 if what == "bucket" else rng.choice([2, 3]),
                "n": _log(rng, 1000, 8000000), "per_bin": round(rng.uniform(2.0, 24.0), 2),
                "order": rng.choice(["moved", "random"])}
    if kind == "turnover":
        return {"kind": "turnover", "n": _log(rng, 1000, 4000000), "deaths": round(rng.uniform(0.0, 0.5), 3),
                "births": round(rng.uniform(0.0, 0.3), 3)}
    return {"kind": "stats", "n": _log(rng, 1000, 16000000), "dtype": rng.choice(["f32", "f32", "i32", "u32", "f64", "i64"])}


# ---------------------------------------------------------------- inputs

def _population(case, seed):
    """Model library, parameters and {agent: arrays} of a run."""
    n = case["n"]
    if case["model"] == "predprey":
        params, prey, pred = workloads.predprey(n, case["predators"], seed=seed, width=case["width"])
        # populations in balance, so that a pass costs the same however long the run has been
        # going: prey are born as often as they die (1 % a step), predators hunt, eat nothing
        # and do not starve
        params[2], params[3], params[4], params[6] = 0.0, 0.01, 0.01, 1e9
        return "predator_prey", params, {"Prey": prey, "Predator": pred}
    lib, _, request = serving.MODELS[case["model"]]
    params, pops = request(n, seed)
    if case["model"] == "boids":
        params[5] = 1e-3   # steering so weak that the flock stays spread out, for the same reason
    return lib, params, pops


def _batch_plans(case, seed):
    sizes = np.random.default_rng(case["count"])   # the ensemble's plan; its populations come from the seed
    rng = np.random.default_rng(seed)
    plans = []
    for k in range(case["count"]):
        n = int(np.exp(sizes.uniform(np.log(case["n_lo"]), np.log(case["n_hi"]))))
        params, arrs = workloads.circles(n, seed=int(rng.integers(1 << 31)), radius=float(sizes.uniform(1.0, 3.0)))
        plans.append((params, int(seed) * 1000 + k, arrs))
    return plans


def _grid(case):
    """Bins per axis and total: as near `per_bin` elements a bin as a whole number of bins allows."""
    if case["what"] == "bucket":
        keys = max(1, int(case["n"] / case["per_bin"]))
        return keys, keys
    g = max(3, int(round((case["n"] / case["per_bin"]) ** (1.0 / case["dims"]))))
    return g, g ** case["dims"]


def _index_inputs(case, seed):
    """Variables of the list: positions, two or three velocity parts, id (32 bits each)."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    n, dims = case["n"], case["dims"]
    g, _ = _grid(case)
    ids = torch.randperm(n, generator=gen, device="cuda", dtype=torch.int32) + 1
    if case["what"] == "bucket":
        key = torch.randint(0, g, (n,), generator=gen, device="cuda", dtype=torch.int32)
        if case["order"] == "moved":   # mostly in order: one in eight has changed its key
            key = torch.sort(key).values
            swap = torch.rand(n, generator=gen, device="cuda") < 0.125
            new = torch.randint(0, g, (n,), generator=gen, device="cuda", dtype=torch.int32)
            key = torch.where(swap, new, key)
        value = torch.rand(n, generator=gen, device="cuda") * 2 - 1
        return [key, ids, value]
    r, w = np.float32(0.05), np.float32(0.05) * np.float32(g)
    top = float(np.nextafter(w, np.float32(0)))
    pos = [torch.rand(n, generator=gen, device="cuda") * float(w) for _ in range(dims)]
    vel = torch.rand((dims, n), generator=gen, device="cuda") * 2 - 1
    vel = vel / vel.norm(dim=0, keepdim=True).clamp_min(1e-6) * 0.04
    if case["order"] == "moved":
        # the order of the last step's bins, then one step of movement with wrap-around
        key = torch.zeros(n, device="cuda", dtype=torch.int64)
        for a in reversed(range(dims)):
            key = key * g + (pos[a] / float(r)).to(torch.int64).clamp(0, g - 1)
        at = torch.argsort(key, stable=True)
        pos = [p[at] for p in pos]
        for a in range(dims):
            p = pos[a] + vel[a]
            p = torch.where(p < 0, p + float(w), p)
            pos[a] = torch.where(p >= float(w), p - float(w), p)
    pos = [p.clamp(0.0, top) for p in pos]
    return pos + [vel[a].contiguous() for a in range(dims)] + [ids]


def _turnover_inputs(case, seed):
    """Death and birth flags, the list's 7 variables, the new agents' 7 variables (last: id)."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    n = case["n"]

    def rand():
        return torch.rand(n, generator=gen, device="cuda")

    dead = (rand() < case["deaths"]).to(torch.int32)
    born = (rand() < case["births"]).to(torch.int32)
    ids = torch.randperm(n, generator=gen, device="cuda", dtype=torch.int32) + 1
    return dead, born, [rand() for _ in range(6)] + [ids], [rand() for _ in range(6)] + [torch.zeros_like(ids)]


def _stats_input(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    n, dt = case["n"], case["dtype"]
    if dt in ("f32", "f64"):
        return (torch.rand(n, generator=gen, device="cuda", dtype=TORCH[dt]) * 2 - 0.75)
    lo = 0 if dt == "u32" else -1000000
    return torch.randint(lo, 1000000, (n,), generator=gen, device="cuda", dtype=TORCH[dt])


def _ptrs(tensors):
    return [t.data_ptr() for t in tensors]


# ---------------------------------------------------------------- one pass

def prepare(case, seed):
    kind = case["kind"]
    if kind == "run":
        lib, params, pops = _population(case, seed)
        sim = Simulation(lib, params, seed=int(seed))
        sim.set_option("graphs", 0)
        for agent, arrays in pops.items():
            sim.set_agents(agent, arrays)
        return {"case": case, "sim": sim}
    if kind == "batch":
        plans = _batch_plans(case, seed)
        b = Batch("circles_spatial3D", plans[0][0])
        b.set_option("graphs", 0)
        b.set_option("bins_per_radius", case["bins_per_radius"])
        handles = [b.add(params, seed, 1 << 30, {"Circle": arrs}) for params, seed, arrs in plans]
        return {"case": case, "batch": b, "handles": handles}
    ctx = fgx.Context(0)
    if kind == "index":
        v = _index_inputs(case, seed)
        n, dims = case["n"], case["dims"]
        g, bins = _grid(case)
        s = {"case": case, "ctx": ctx, "in": v, "out": [torch.zeros_like(t) for t in v], "bytes": [4] * len(v)}
        if case["what"] == "agents":
            w = float(np.float32(0.05) * np.float32(g))
            s["box"] = ([0.0] * dims, [w] * dims, 0.05)
            bits = fgx.agent_sort_key_bits(dims, *s["box"])
            s["len"] = fgx.scratch_bytes(fgx.FGX_OP_AGENT_SORT, n, 1 << bits)
        else:
            if case["what"] == "messages":
                w = float(np.float32(0.05) * np.float32(g))
                s["meta"] = fgx.spatial_meta(dims, [0.0] * dims, [w] * dims, 0.05)
                bins = s["meta"].bins
                s["rec_vars"] = [0, 1, 2 if dims == 3 else -1, len(v) - 1]
                s["records"] = torch.zeros((n, 4), dtype=torch.int32, device="cuda")
            s["keys"] = bins
            s["pbm"] = torch.zeros(bins + 1, dtype=torch.int32, device="cuda")
            s["len"] = fgx.scratch_bytes(fgx.FGX_OP_SPATIAL_BUILD, n, bins)
        s["scratch"] = torch.zeros(s["len"] // 4 + 1, dtype=torch.int32, device="cuda")
        return s
    if kind == "turnover":
        dead, born, old, new = _turnover_inputs(case, seed)
        n = case["n"]
        cap = 2 * n
        length = max(fgx.scratch_bytes(fgx.FGX_OP_COMPACT, n), fgx.scratch_bytes(fgx.FGX_OP_BIRTHS, n))
        return {"case": case, "ctx": ctx, "dead": dead, "born": born, "old": old, "new": new,
                "list": [torch.zeros(cap, dtype=t.dtype, device="cuda") for t in old],
                "count": torch.zeros(1, dtype=torch.int32, device="cuda"),
                "next_id": torch.full((1,), n + 1, dtype=torch.int32, device="cuda"), "cap": cap, "len": length,
                "scratch": torch.zeros(length // 4 + 1, dtype=torch.int32, device="cuda")}
    length = fgx.scratch_bytes(fgx.FGX_OP_STATS, 0)
    acc = torch.float64 if case["dtype"] in ("f32", "f64") else torch.int64
    return {"case": case, "ctx": ctx, "in": _stats_input(case, seed), "out": torch.zeros(4, dtype=acc, device="cuda"),
            "len": length, "scratch": torch.zeros(length // 4 + 1, dtype=torch.int32, device="cuda")}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "run":
        sim = s["sim"]
        sim.step(case["steps"])
        if case["model"] != "predprey":
            return list(sim.get_agents("Circle" if case["model"] == "circles" else "Boid"))
        got = list(sim.get_agents("Predator"))
        if case["n"] <= 50000:
            # prey come and go: their number varies with the seed, so they are given back in
            # arrays of one length, zero behind the last
            arrs, ids = sim.get_agents("Prey")
            got += [np.concatenate([a, np.zeros(2 * case["n"] + 4096 - len(a), a.dtype)]) for a in arrs + [ids]]
        return got
    if kind == "batch":
        b = s["batch"]
        b.step(case["steps"])
        got = [b.get_agents(h, "Circle") for h in s["handles"]]
        return [np.concatenate([arrs[k] for arrs, _ in got]) for k in range(4)] + [np.concatenate([ids for _, ids in got])]
    if kind == "index":
        n, vi, vo, scratch = case["n"], _ptrs(s["in"]), _ptrs(s["out"]), s["scratch"].data_ptr()
        pos = vi[:case["dims"]] + [None] * (3 - case["dims"])
        if case["what"] == "agents":
            mn, mx, r = s["box"]
            fgx.agent_sort(s["ctx"], case["dims"], mn, mx, r, n, *pos, vi, vo, s["bytes"], scratch, s["len"])
            return s["out"]
        if case["what"] == "bucket":
            fgx.bucket_build(s["ctx"], 0, s["keys"], n, vi[0], vi, vo, s["bytes"], s["pbm"].data_ptr(), scratch, s["len"])
            return s["out"] + [s["pbm"]]
        fgx.spatial_build_records(s["ctx"], s["meta"], n, *pos, vi, vo, s["bytes"], s["rec_vars"], s["records"].data_ptr(),
                                  s["pbm"].data_ptr(), scratch, s["len"])
        return s["out"] + [s["records"], s["pbm"]]
    if kind == "turnover":
        n, b, lst, scratch = case["n"], [4] * 7, _ptrs(s["list"]), s["scratch"].data_ptr()
        fgx.compact(s["ctx"], s["dead"].data_ptr(), 0, n, _ptrs(s["old"]), lst, b, s["count"].data_ptr(), scratch, s["len"])
        fgx.append_births(s["ctx"], s["born"].data_ptr(), n, _ptrs(s["new"]), lst, b, 6, s["count"].data_ptr(), s["cap"],
                          s["next_id"].data_ptr(), scratch, s["len"])
        return s["list"] + [s["count"], s["next_id"]]
    fgx.reduce_stats(s["ctx"], STATS_CODE[case["dtype"]], s["in"].data_ptr(), case["n"], s["out"].data_ptr(),
                     s["scratch"].data_ptr(), s["len"])
    # the fourth word is a double, whatever the type of the other three
    return [s["out"][:3], s["out"][3:].view(torch.float64)]


# ---------------------------------------------------------------- what a pass cannot do without

# state read and written once a step; operations on each candidate neighbour (distance,
# comparison) and the mean number of candidates in the searched bins
AGENT_BYTES = {"circles": 20, "boids": 28, "predprey": 20}
PAIR_FLOPS = {"circles": 9, "boids": 15, "predprey": 6}


def _candidates(case, radius=2.0):
    fine = (2.5 / 3.0) if case.get("bins_per_radius") == 2 else 1.0
    if case.get("model") == "boids":
        return 27 * 4.0 * fine ** 3
    if case.get("model") == "predprey":
        return (15.0 * fine) ** 2 * case["n"] / case["width"] ** 2
    return (3 * radius * fine) ** 3 * 0.85   # density 1; the box's faces cut some neighbourhoods


def work(case):
    kind = case["kind"]
    if kind == "run":
        n = case["n"] + case.get("predators", 0)
        return {"bytes": 2.0 * AGENT_BYTES[case["model"]] * n * case["steps"],
                "flops": float(n) * case["steps"] * PAIR_FLOPS[case["model"]] * _candidates(case)}
    if kind == "batch":
        lo, hi = case["n_lo"], case["n_hi"]
        n = case["count"] * (hi - lo) / math.log(hi / lo)
        return {"bytes": 2.0 * 20 * n * case["steps"], "flops": n * case["steps"] * 9 * _candidates(case)}
    n = float(case["n"])
    if kind == "index":
        _, bins = _grid(case)
        nvars = 3 if case["what"] == "bucket" else 2 * case["dims"] + 1
        table = 0 if case["what"] == "agents" else 4.0 * (bins + 1)
        return {"bytes": 8.0 * nvars * n + table + (16.0 * n if case["what"] == "messages" else 0.0), "flops": 0.0}
    if kind == "turnover":
        kept, born = n * (1 - case["deaths"]), n * case["births"]
        return {"bytes": 8.0 * n + 2.0 * 28 * kept + (24.0 + 28.0) * born, "flops": 0.0}
    return {"bytes": n * BYTES[case["dtype"]], "flops": 6.0 * n}


def tolerance(case):
    # sums in double whose order is open; everything else, integer statistics among it, is
    # defined to the bit (see the module's text)
    if case["kind"] == "stats":
        return {"rel": 1e-13, "max": 1e-12, "differ": 0.0}
    return "exact"


# ---------------------------------------------------------------- the same in 64 bits

def _keys(pos, grid, scale):
    """Bin of each element: z-major cell number of the clamped cells."""
    key = np.zeros(len(pos[0]), np.int64)
    for p, g, s in reversed(list(zip(pos, grid, scale))):
        key = key * g + np.clip(s(p), 0, g - 1)
    return key


def _cells(pos, key, bins):
    order = np.argsort(key, kind="stable")
    return order, np.concatenate([[0], np.cumsum(np.bincount(key, minlength=bins))])


def _one_step(case, seed):
    """One step of circles or boids: positions and forces in 64 bits; which bin an agent
    is in, and so the order of the result, from the 32-bit positions."""
    lib, params, pops = _population(case, seed)
    arrs, = pops.values()
    n = case["n"]
    boids = case["model"] == "boids"
    lo, hi, r = (params[0], params[1], params[2]) if boids else (np.float32(0), params[0], params[1])
    w = np.float32(hi - lo)
    grid = int(np.ceil(np.float32(w / r)))

    def cell(p):
        return np.floor((p - lo) / r).astype(np.int64)

    def sort_cell(p):
        return np.floor(((p - lo) / w) * np.float32(grid)).astype(np.int64)

    # agents are put in spatial order before they read their messages
    order = np.argsort(_keys(arrs[:3], [grid] * 3, [sort_cell] * 3), kind="stable")
    ids = np.arange(1, n + 1, dtype=np.int64)[order]
    a32 = [a[order] for a in arrs]
    c = [np.clip(cell(a32[k]), 0, grid - 1) for k in range(3)]
    at, start = _cells(a32[:3], (c[2] * grid + c[1]) * grid + c[0], grid ** 3)
    a = [x.astype(np.float64) for x in a32]
    rr, ww = float(r), float(w)
    fx = np.zeros((3, n))
    centre, heading, count = np.zeros((3, n)), np.zeros((3, n)), np.zeros(n, np.int64)
    me = np.arange(n)
    for dx in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dz in (-1, 0, 1):
                q = [c[0] + dx, c[1] + dy, c[2] + dz]
                if boids:
                    q = [v % grid for v in q]
                    live = np.ones(n, bool)
                else:
                    live = np.all([(v >= 0) & (v < grid) for v in q], axis=0)
                b = np.where(live, (q[2] * grid + q[1]) * grid + q[0], 0)
                s, e = start[b], np.where(live, start[b + 1], 0)
                for k in range(int(max(0, (e - s).max()))):
                    i = np.nonzero(s + k < e)[0]
                    j = at[s[i] + k]
                    i, j = i[me[i] != j], j[me[i] != j]
                    d = np.stack([a[x][j] - a[x][i] for x in range(3)])
                    if boids:
                        d = np.where(np.abs(d) > ww / 2, d - np.copysign(ww, d), d)
                    dist = np.sqrt((d * d).sum(axis=0))
                    near = (dist < rr) & (dist > 0 if not boids else True)
                    i, j, d, dist = i[near], j[near], d[:, near], dist[near]
                    count[i] += 1
                    if not boids:
                        fx[:, i] += np.sin(dist / rr * 3.141 * -2.0) * float(params[2]) * d / dist
                        continue
                    for x in range(3):
                        centre[x, i] += a[x][i] + d[x]
                        heading[x, i] += a[3 + x][j]
                    sep = float(params[3])
                    close = dist < sep
                    i, d, dist = i[close], d[:, close], dist[close]
                    fx[:, i] -= float(params[7]) * d * (1.0 - dist / sep) ** 2
    cnt = np.maximum(count, 1)
    if not boids:
        f = fx / cnt
        new = [np.clip(a[k] + f[k], 0.0, float(hi)) for k in range(3)]
        return [new + [np.sqrt((f * f).sum(axis=0))], ids]
    _, _, _, _, time_scale, global_scale, steer, _, match, vmin, vmax = [float(x) for x in params]
    some = count > 0
    p0, v0 = np.stack(a[:3]), np.stack(a[3:6])
    fx += np.where(some, (centre / cnt - p0) * steer + heading / cnt * match - v0, 0.0)
    v = v0 + fx * global_scale
    speed = np.sqrt((v * v).sum(axis=0))
    v = np.where(speed > vmax, v / speed * vmax, v)
    v = np.where(speed < vmin, v / speed * vmin, v)
    p = p0 + v * time_scale
    p = np.where(p < float(lo), p + ww, p)
    p = np.where(p > float(hi), p - ww, p)
    return [[*p, *v], ids]


def exact(case, seed):
    kind = case["kind"]
    if kind == "run":
        if case["steps"] != 1 or case["model"] == "predprey" or case["n"] > 200000:
            return None   # a run of many steps has no 64-bit counterpart: its states diverge
        return _one_step(case, seed)
    if kind == "batch":
        return None
    if kind == "index":
        v = [t.cpu().numpy() for t in _index_inputs(case, seed)]
        g, bins = _grid(case)
        w, r = np.float32(0.05) * np.float32(g), np.float32(0.05)
        if case["what"] == "bucket":
            key = v[0].astype(np.int64)
        elif case["what"] == "messages":
            g = int(np.ceil(w / r))
            bins = g ** case["dims"]
            key = _keys(v[:case["dims"]], [g] * case["dims"], [lambda p: np.floor(p / r).astype(np.int64)] * case["dims"])
        else:
            g = int(np.ceil(w / r))
            bits = int(math.floor(math.log2(g ** case["dims"]))) + 1
            key = np.zeros(case["n"], np.int64)
            for p in reversed(v[:case["dims"]]):
                key = key * g + np.floor((p / w) * np.float32(g)).astype(np.int64)
            key &= (1 << bits) - 1
        order = np.argsort(key, kind="stable")
        out = [x[order] for x in v]
        if case["what"] == "agents":
            return out
        pbm = np.concatenate([[0], np.cumsum(np.bincount(key, minlength=bins))])
        if case["what"] == "bucket":
            return out + [pbm.astype(np.int32)]
        rec = [out[0], out[1], out[2] if case["dims"] == 3 else np.zeros_like(out[0]), out[-1]]
        return out + [np.stack([x.view(np.int32) for x in rec], axis=1), pbm.astype(np.int32)]
    if kind == "turnover":
        dead, born, old, new = _turnover_inputs(case, seed)
        n = case["n"]
        dead, born = dead.cpu().numpy() != 0, born.cpu().numpy() != 0
        kept, births = int((~dead).sum()), int(born.sum())
        out = []
        for k in range(7):
            o, m = old[k].cpu().numpy(), new[k].cpu().numpy()
            x = np.zeros(2 * n, o.dtype)
            x[:kept] = o[~dead]
            x[kept:kept + births] = m[born] if k < 6 else np.arange(n + 1, n + 1 + births)
            out.append(x)
        return out + [np.array([kept + births], np.int32), np.array([n + 1 + births], np.int32)]
    x = _stats_input(case, seed)
    mean = x.double().mean()
    dev = float((x.double() - mean).square().sum())
    if case["dtype"] in ("f32", "f64"):
        first = torch.tensor([float(x.double().sum()), float(x.min()), float(x.max())], dtype=torch.float64)
    else:
        first = torch.tensor([int(x.long().sum()), int(x.min()), int(x.max())], dtype=torch.int64)
    return [first, torch.tensor([dev], dtype=torch.float64)]
