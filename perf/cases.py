"""Performance cases of the sampling framework.

Each case is one pass of a user's program through the public entry points of
c-saw_amd/csaw.py (and the C ABI it binds) on RMAT graphs of the sizes the
benchmark configurations use: RMAT-16 (edge factor 8), RMAT-20 (edge factor 5)
and RMAT-22 (edge factor 16), symmetrised, with FP32 edge weights.  A program
loads its graph once and keeps it, so the graphs live for the process; the
vertices it samples from, the sampling key and the plan over them are a case's
inputs.  How many edges a pass emits follows the drawn degrees, so a program
keeps edge buffers of the most its fanouts can give, and a pass fills the first
entries of them.
"""
import ctypes
import json
import os

import numpy as np
import torch  # before the library, so that both use one HIP runtime

import __graft_entry__

C = __graft_entry__.load_csaw()
L = C.lib()
MODELS = os.path.join(os.path.dirname(os.path.abspath(C.__file__)), "models")
BIAS = {"uniform": C.BIAS_UNIFORM, "degree": C.BIAS_DEGREE, "weight": C.BIAS_WEIGHT, "user": C.BIAS_USER}
GRAPHS = {"rmat16": (16, 8), "rmat20": (20, 5), "rmat22": (22, 16)}
STREAM_BUDGET = 512 << 20

_kept = {}


def _keep(key, make):
    if key not in _kept:
        _kept[key] = make()
    return _kept[key]


def _graph(name):
    scale, ef = GRAPHS[name]
    return _keep(name, lambda: C.Graph.rmat(scale, ef, weights=True))


def _host_graph(name):
    scale, ef = GRAPHS[name]
    return _keep("host_" + name, lambda: C.HostGraph.rmat(scale, ef))


def _cost_model():
    """The trained cost model that ships with the package."""
    def make():
        m = C.Mlp(1)
        with open(os.path.join(MODELS, "cost_model_gfx950.json")) as f:
            m.set_params(np.array(json.load(f)["params"], np.float32))
        return m
    return _keep("cost_model", make)


def _tuning():
    """The launch shapes that ship with the package for request mixes."""
    def make():
        t = C.Tuning()
        with open(os.path.join(MODELS, "tuning_gfx950_c4.json")) as f:
            for k, v in json.load(f).items():
                setattr(t, k, int(v))
        return t
    return _keep("tuning", make)


def _fanouts(case):
    return [int(x) for x in case["fanouts"].split(",")]


def _seeds(rng, V, n):
    return rng.integers(0, V, n, dtype=np.int32)


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one call of the sampler at the reference's default size: 1,000
        # subgraphs, two neighbours, two hops; what a call costs by itself
        {"name": "sample_small", "kind": "sample", "graph": "rmat16", "seeds": 1000, "fanouts": "2,2",
         "bias": "uniform", "dedup": 1},
        # one mini-batch of degree-biased neighbour sampling, edges to the host
        {"name": "sample_degree", "kind": "sample", "graph": "rmat20", "seeds": 8192, "fanouts": "25,10",
         "bias": "degree", "dedup": 1},
        # uniform neighbour sampling from a million vertices, edges kept on the GPU
        {"name": "plan_uniform", "kind": "plan", "graph": "rmat22", "seeds": 1048576, "fanouts": "25,10",
         "bias": "uniform", "dedup": 1, "cache": False},
        # degree bias without the per-graph CDF cache (the reference's default)
        {"name": "plan_degree", "kind": "plan", "graph": "rmat22", "seeds": 40000, "fanouts": "25,10",
         "bias": "degree", "dedup": 1, "cache": False},
        # three hops over FP32 edge weights with the CDF cache, an odd batch
        {"name": "plan_weight", "kind": "plan", "graph": "rmat22", "seeds": 30011, "fanouts": "15,10,5",
         "bias": "weight", "dedup": 1, "cache": True},
        # the reference's default collision policy (region remap)
        {"name": "plan_remap", "kind": "plan", "graph": "rmat22", "seeds": 8191, "fanouts": "10,10",
         "bias": "degree", "dedup": 2, "cache": True},
        # the benchmark's workload: 256 mixed requests, batched, learned
        # schedule, captured graph; every request's edges to GPU tensors
        {"name": "mix_256", "kind": "batch", "graph": "rmat22", "requests": 256, "lo": 64, "hi": 65536,
         "mix": 42},
        # a small serving batch of the same requests
        {"name": "serve_8", "kind": "batch", "graph": "rmat22", "requests": 8, "lo": 64, "hi": 1024, "mix": 7},
        # weighted random walks, the walk corpus read into a pinned buffer
        {"name": "walk_weight", "kind": "walk", "graph": "rmat22", "walkers": 1048576, "len": 80, "bias": "weight"},
        # multi-dimensional random walks from GPU tensors to GPU tensors
        {"name": "mdrw", "kind": "mdrw", "graph": "rmat22", "samples": 4096, "frontier": 64, "depth": 200},
        # a graph kept in host memory, streamed through a device budget
        {"name": "stream_degree", "kind": "stream", "graph": "rmat22", "seeds": 16384, "fanouts": "15,10,5",
         "bias": "degree", "partitions": 16},
        # training the cost model of the learned schedule on logged chunks
        {"name": "cost_model_train", "kind": "train", "rows": 6000, "epochs": 4, "batch": 256},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["sample", "sample", "plan", "plan", "plan", "batch", "batch", "walk", "walk", "mdrw", "stream",
                       "train"])
    fan = rng.choice(["2,2", "5,5", "25,10", "15,10,5", "10,10", "20", "64,3", "7,5,3"])
    if kind == "sample":
        return {"kind": kind, "graph": rng.choice(["rmat16", "rmat20"]), "seeds": _log(rng, 50, 16384),
                "fanouts": fan, "bias": rng.choice(sorted(BIAS)), "dedup": rng.choice([0, 1, 1])}
    if kind == "plan":
        dedup = rng.choice([0, 1, 1, 2])
        most = {0: 262144, 1: 131072, 2: 16384}[dedup]
        return {"kind": kind, "graph": rng.choice(["rmat20", "rmat22"]), "seeds": _log(rng, 100, most),
                "fanouts": fan, "bias": rng.choice(sorted(BIAS)), "dedup": dedup, "cache": rng.random() < 0.5}
    if kind == "batch":
        hi = rng.choice([512, 4096, 32768])
        return {"kind": kind, "graph": "rmat22", "requests": _log(rng, 3, 200), "lo": rng.choice([16, 64]), "hi": hi,
                "mix": rng.randint(1, 1 << 20)}
    if kind == "walk":
        return {"kind": kind, "graph": rng.choice(["rmat20", "rmat22"]), "walkers": _log(rng, 500, 700000),
                "len": rng.randint(8, 80), "bias": rng.choice(sorted(BIAS))}
    if kind == "mdrw":
        depth = rng.randint(20, 300)
        return {"kind": kind, "graph": rng.choice(["rmat20", "rmat22"]), "samples": _log(rng, 50, 8000),
                "frontier": _log(rng, 2, 2048), "depth": depth}
    if kind == "stream":
        return {"kind": kind, "graph": "rmat22", "seeds": _log(rng, 500, 16384),
                "fanouts": rng.choice(["25,10", "15,10,5", "10,10"]), "bias": rng.choice(["uniform", "degree", "user"]),
                "partitions": rng.choice([5, 8, 16])}
    return {"kind": kind, "rows": _log(rng, 300, 12000), "epochs": rng.randint(1, 4),
            "batch": rng.choice([64, 200, 256, 512])}


# ---------------------------------------------------------------- preparation
def _most(seeds, fanouts):
    return sum(int(np.prod(fanouts[:h + 1])) for h in range(len(fanouts))) * seeds


def _host_buffers(case):
    fan = _fanouts(case)
    n = _most(case["seeds"], fan)
    return {"src": np.zeros(n, np.int32), "dst": np.zeros(n, np.int32), "smp": np.zeros(n, np.int32),
            "hop_off": np.zeros((len(fan), case["seeds"] + 1), np.int64)}


def _device_buffers(specs):
    n = sum(_most(len(s["seeds"]), s["fanouts"]) for s in specs)
    h = sum(len(s["fanouts"]) * (len(s["seeds"]) + 1) for s in specs)
    out = {k: torch.zeros(n, dtype=torch.int32, device="cuda") for k in ("src", "dst", "smp")}
    out["hop_off"] = torch.zeros(h, dtype=torch.int64, device="cuda")
    return out


def _chunk_rows(rng, n):
    """Chunk features, log2 times and measured-variant masks as a logged run
    gives them: sizes and degrees over their logarithms, one bias kind each."""
    X = np.zeros((n, 16), np.float32)
    length = np.exp2(rng.uniform(3, 10, n))
    mean_d = np.exp2(rng.uniform(1, 17, n))
    max_d = mean_d * np.exp2(rng.uniform(0, 2, n))
    fan = rng.choice([5.0, 10.0, 15.0, 25.0], n)
    kind = rng.integers(0, 3, n)
    X[:, 0] = 1
    X[:, 1] = np.log2(length + 1) / 10
    X[:, 2] = np.log2(mean_d + 1) / 20
    X[:, 3] = np.log2(max_d + 1) / 20
    X[:, 4] = fan / 64
    X[:, 5] = fan / 64
    X[np.arange(n), 6 + kind] = 1
    X[:, 9] = rng.integers(0, 3, n) / 8
    X[:, 10] = np.minimum(fan / mean_d, 1)
    X[:, 11] = max_d <= 32
    X[:, 12] = max_d <= 1024
    X[:, 13] = max_d <= 8192
    X[:, 14] = np.log2(rng.uniform(1e3, 6e4, n)) / 24
    X[:, 15] = rng.integers(0, 8, n) / 8
    cost = np.log2(length * (1 + fan) * (1 + kind * np.log2(mean_d) / 4))
    T = (cost[:, None] + rng.normal(0, 0.5, (n, 5)) - 3).astype(np.float32)
    M = (rng.random((n, 5)) < 0.7).astype(np.float32)
    M[:, 1] = 1
    return X, T, M


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    key = int(rng.integers(1, 1 << 40))
    kind = case["kind"]
    if kind == "train":
        X, T, M = _chunk_rows(rng, case["rows"])
        m = C.Mlp(seed % 1000 + 1)
        return {"case": case, "mlp": m, "start": m.params(), "X": X, "T": T, "M": M, "key": key}
    if kind == "stream":
        hg = _host_graph(case["graph"])
        return {"case": case, "graph": hg, "seeds": _seeds(rng, hg.V, case["seeds"]), "key": key,
                "out": _host_buffers(case)}
    g = _graph(case["graph"])
    if kind == "sample":
        return {"case": case, "graph": g, "seeds": _seeds(rng, g.V, case["seeds"]), "key": key,
                "out": _host_buffers(case)}
    if kind == "walk":
        seeds = _seeds(rng, g.V, case["walkers"])
        W = torch.empty((case["walkers"], case["len"] + 1), dtype=torch.int32, pin_memory=True)
        return {"case": case, "plan": C.WalkPlan(g, seeds, case["len"], bias=BIAS[case["bias"]], key=key), "W": W}
    if kind == "mdrw":
        S, D = case["samples"], case["depth"]
        seeds = torch.from_numpy(_seeds(rng, g.V, S * case["frontier"])).cuda()
        return {"case": case, "graph": g, "seeds": seeds, "key": key,
                "src": torch.zeros(S * D, dtype=torch.int32, device="cuda"),
                "dst": torch.zeros(S * D, dtype=torch.int32, device="cuda"),
                "off": torch.zeros(S + 1, dtype=torch.int64, device="cuda")}
    if kind == "plan":
        spec = {"seeds": _seeds(rng, g.V, case["seeds"]), "fanouts": _fanouts(case), "bias": BIAS[case["bias"]],
                "dedup": case["dedup"], "key": key, "request": 0}
        return {"case": case, "plan": C.Plan(g, [spec], mode=C.MODE_PLAIN, cdf_cache=case["cache"]),
                "out": _device_buffers([spec])}
    specs = C.request_mix(case["requests"], case["lo"], case["hi"], mix_key=case["mix"])
    for s in specs:
        s["seeds"] = _seeds(rng, g.V, s["samples"])
        s["key"] = key
    return {"case": case, "plan": C.Plan(g, specs, mode=C.MODE_BATCHED, sched=C.SCHED_MLP, mlp=_cost_model(),
                                         tuning=_tuning(), use_graph=True, cdf_cache=True),
            "out": _device_buffers(specs)}


# ------------------------------------------------------------------- one pass
def _edges_to_tensors(plan, out):
    """Every request's edges, one after another, and its hop offsets."""
    at = to = 0
    for r, spec in enumerate(plan.specs):
        n = plan.n_edges(r)
        C._check(L.csaw_plan_copy_device(plan.h, r, out["src"].data_ptr() + 4 * at, out["dst"].data_ptr() + 4 * at,
                                         out["smp"].data_ptr() + 4 * at, out["hop_off"].data_ptr() + 8 * to, None,
                                         1 if r == len(plan.specs) - 1 else 0), "plan_copy_device")
        at += n
        to += len(spec["fanouts"]) * (len(spec["seeds"]) + 1)
    return out


def _edges_to_host(r, out):
    n = len(r["src"])
    for k in ("src", "dst", "smp"):
        out[k][:n] = r[k]
    out["hop_off"][:] = r["hop_off"]
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("plan", "batch"):
        state["plan"].run()
        return _edges_to_tensors(state["plan"], state["out"])
    if kind == "sample":
        r = C.sample(state["graph"], state["seeds"], _fanouts(case), bias=BIAS[case["bias"]], dedup=case["dedup"],
                     key=state["key"])
        return _edges_to_host(r, state["out"])
    if kind == "walk":
        state["plan"].run()
        steps = C.i64()
        C._check(L.csaw_walk_plan_result(state["plan"].h, state["W"].data_ptr(), ctypes.byref(steps), None, None),
                 "walk_plan_result")
        return {"walks": state["W"], "steps": steps.value}
    if kind == "mdrw":
        C._check(L.csaw_mdrw_noalloc(state["graph"].h, state["key"], 0, case["samples"], case["frontier"],
                                     case["depth"], state["seeds"].data_ptr(), state["src"].data_ptr(),
                                     state["dst"].data_ptr(), state["off"].data_ptr(), None, 1), "mdrw_noalloc")
        return {"src": state["src"], "dst": state["dst"], "off": state["off"]}
    if kind == "stream":
        r = C.stream_sample(state["graph"], state["seeds"], _fanouts(case), bias=BIAS[case["bias"]], key=state["key"],
                            budget_bytes=STREAM_BUDGET, partitions=case["partitions"])
        return _edges_to_host(r, state["out"])
    m = state["mlp"]
    m.set_params(state["start"])
    loss = m.train(state["X"], state["T"], state["M"], epochs=case["epochs"], batch=case["batch"],
                   shuffle_key=state["key"])
    return {"params": m.params(), "loss": np.array([loss], np.float32)}


# --------------------------------------------------------- what a pass needs
def _edges_per_seed(graph, bias, fanouts, dedup):
    """Mean edges a seed gives, from 4,096 seeds (sizes follow the degrees)."""
    def make():
        g = _graph(graph)
        seeds = _seeds(np.random.default_rng(5), g.V, 4096)
        n = len(C.sample(g, seeds, fanouts, bias=BIAS[bias], dedup=min(dedup, 1))["src"])
        return n / 4096.0
    return _keep(("edges", graph, bias, tuple(fanouts), min(dedup, 1)), make)


def work(case):
    """Per emitted edge: its neighbour id read (4 bytes) and the edge written
    (12), the frontier vertex it gave read once more (4 + 8 for its offset) and,
    with a bias, one CDF entry (4).  Per walk step: offset, CDF entry and id
    read, id written."""
    kind = case["kind"]
    if kind == "train":
        macs = 16 * 64 + 64 * 64 + 64 * 5
        return {"bytes": 104.0 * case["rows"] * (case["epochs"] + 1),
                "flops": 6.0 * macs * case["rows"] * case["epochs"] + 2.0 * macs * case["rows"]}
    if kind == "walk":
        return {"bytes": (4.0 + 8 + 4 + (0 if case["bias"] == "uniform" else 4)) * case["walkers"] * case["len"] / 2,
                "flops": 0.0}
    if kind == "mdrw":
        return {"bytes": 4.0 * case["samples"] * case["frontier"] + 28.0 * case["samples"] * case["depth"],
                "flops": 0.0}
    if kind == "batch":
        seeds = case["requests"] * (case["hi"] - case["lo"]) / np.log(case["hi"] / case["lo"])
        per = sum(_edges_per_seed(case["graph"], b, f, 1) for b in ("uniform", "degree", "weight")
                  for f in ([25, 10], [15, 10, 5])) / 6
        return {"bytes": 31.0 * seeds * per, "flops": 0.0}
    per = _edges_per_seed(case["graph"], case["bias"], _fanouts(case), case.get("dedup", 1))
    return {"bytes": (28.0 if case["bias"] == "uniform" else 32.0) * case["seeds"] * per, "flops": 0.0}


# ----------------------------------------------------------- 64-bit reference
def _philox(c0, c1, c2, c3, k0, k1):
    """Philox4x32-10 (Salmon et al., SC'11) over arrays of counters."""
    lo = np.uint64(0xFFFFFFFF)
    c = [np.asarray(x, np.uint64) for x in np.broadcast_arrays(c0, c1, c2, c3)]
    for r in range(10):
        if r:
            k0 = (k0 + 0x9E3779B9) & 0xFFFFFFFF
            k1 = (k1 + 0xBB67AE85) & 0xFFFFFFFF
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & lo, (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & lo]
    return c


def _bf16(x):
    """float64 -> nearest bfloat16 (ties to even), as float64."""
    return torch.from_numpy(x).to(torch.bfloat16).to(torch.float64).numpy()


def exact(case, seed):
    """Edges, walks and offsets are whole numbers; the trained parameters and
    the loss are computed here in 64 bits (working weights rounded to bfloat16
    after each step, as the model defines them)."""
    if case["kind"] != "train":
        return None
    state = prepare(case, seed)
    X, T, M = (state[k].astype(np.float64) for k in "XTM")
    n, key, lr = case["rows"], state["key"], float(np.float32(0.05))
    shapes = [(64, 16), (64,), (64, 64), (64,), (5, 64), (5,)]
    ends = np.cumsum([int(np.prod(s)) for s in shapes])
    p = state["start"].astype(np.float64)

    def parts(v):
        return [a.reshape(s) for a, s in zip(np.split(v, ends[:-1]), shapes)]

    def step(rows):
        w1, b1, w2, b2, w3, b3 = parts(_bf16(p))
        x, t, m = X[rows], T[rows], M[rows] != 0
        h1 = np.maximum(x @ w1.T + b1, 0)
        h2 = np.maximum(h1 @ w2.T + b2, 0)
        e = np.where(m, h2 @ w3.T + b3 - t, 0.0)
        cnt = max(m.sum(), 1)
        dy = e / cnt
        d2 = (dy @ w3) * (h2 > 0)
        d1 = (d2 @ w2) * (h1 > 0)
        g = [d1.T @ x, d1.sum(0), d2.T @ h1, d2.sum(0), dy.T @ h2, dy.sum(0)]
        return np.concatenate([a.reshape(-1) for a in g]), 0.5 * (e * e).sum() / cnt

    perm = np.arange(n)
    i = np.arange(n)
    for ep in range(case["epochs"]):
        o = _philox(i, ep, 2, 8 << 28, key & 0xFFFFFFFF, key >> 32)
        for k in range(n - 1, 0, -1):
            j = (((int(o[1][k]) << 32) | int(o[0][k])) * (k + 1)) >> 64
            perm[k], perm[j] = perm[j], perm[k]
        for b in range(0, n, case["batch"]):
            p = p - lr * step(perm[b:b + case["batch"]])[0]
    return {"params": p, "loss": np.array([step(np.arange(n))[1]])}
