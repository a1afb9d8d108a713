"""The work this engine is timed on: one call of a public entry point per case.

Sizes are the benchmark's and the tests' configurations (R-MAT with edge
factor 16 or 32, HBM budgets of 25% and 30%, 64-source batches, the star with
a 2,000-vertex path, ids past 2^32), scaled so that a graph can be built many
times, and generic ones (a weighted grid).  `listed` names one case for each
use; `draw` spreads sizes, stores and options over the same ranges.
"""
import math

import numpy as np
import torch

import thievory_amd as T

DAMPING, TOL, MAX_ITER = 0.85, 1e-7, 100  # the defaults of Graph.pr


def listed():
    return [
        # one query on a small graph: launches and host round trips only
        {"name": "bfs-rmat14-split25", "kind": "bfs", "graph": "rmat", "scale": 14, "ef": 16,
         "budget": 0.25, "part": 1 << 12},
        # a traversal of high diameter from a hub: thousands of tiny frontiers
        {"name": "bfs-star-path", "kind": "bfs", "graph": "star", "leaves": 19999, "path": 2001,
         "budget": 1.0, "part": 1 << 16},
        # the headline shape: undirected, edges out of HBM's budget, levels
        # read back by the caller
        {"name": "bfs-rmat25-split25", "kind": "bfs", "graph": "rmat", "scale": 25, "ef": 32,
         "budget": 0.25, "part": 1 << 16},
        # components of the same kind of graph
        {"name": "cc-rmat23-split25", "kind": "cc", "graph": "rmat", "scale": 23, "ef": 32,
         "budget": 0.25, "part": 1 << 16},
        # least reaching id on a directed graph, its edges in HBM
        {"name": "cc-directed-3M", "kind": "cc", "graph": "directed", "n": 3000017, "ef": 16,
         "budget": 1.0, "part": 1 << 16},
        # road-like: many buckets, each with a small frontier
        {"name": "sssp-grid-500", "kind": "sssp", "graph": "grid", "rows": 500, "cols": 500,
         "budget": 1.0, "part": 1 << 16},
        # weighted records, 30% of them in HBM
        {"name": "sssp-rmat23-split30", "kind": "sssp", "graph": "rmat", "scale": 23, "ef": 16,
         "budget": 0.3, "part": 1 << 16},
        # PageRank along out-edges, 25% of them in HBM
        {"name": "pr-push-2M-split25", "kind": "pr", "mode": "push", "n": 2000003, "ef": 16,
         "budget": 0.25, "part": 1 << 16},
        # PageRank along in-edges, all in HBM (the default store)
        {"name": "pr-pull-4M", "kind": "pr", "mode": "pull", "n": 4000037, "ef": 16,
         "budget": 1.0, "part": 1 << 16},
        # 64 queries at once on a resident graph
        {"name": "batch-bfs64-rmat22", "kind": "batch", "algo": "bfs", "scale": 22, "ef": 16,
         "k": 64, "budget": 1.0, "part": 1 << 16},
        {"name": "batch-sssp64-rmat20", "kind": "batch", "algo": "sssp", "scale": 20, "ef": 16,
         "k": 64, "budget": 1.0, "part": 1 << 16},
        # ids past 2^32, few of them with edges
        {"name": "wide-sssp-rmat18", "kind": "wide", "algo": "sssp", "scale": 18, "ef": 16,
         "stride": 16899, "budget": 1.0, "part": 1 << 16},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["bfs", "bfs", "path", "cc", "cc-directed", "sssp", "grid", "push", "pull",
                       "batch-bfs", "batch-sssp", "wide"])
    c = {"budget": rng.choice([1.0, 1.0, 0.5, 0.3, 0.25]), "part": rng.choice([1 << 12, 1 << 16])}
    if kind == "bfs":
        c.update(kind="bfs", graph="rmat", scale=rng.randint(10, 23), ef=rng.randint(8, 32))
    elif kind == "path":
        c.update(kind="bfs", graph="star", leaves=_log(rng, 500, 200000), path=_log(rng, 100, 4000))
    elif kind == "cc":
        c.update(kind="cc", graph="rmat", scale=rng.randint(10, 22), ef=rng.randint(4, 32))
    elif kind == "cc-directed":
        c.update(kind="cc", graph="directed", n=_log(rng, 1000, 3000000), ef=rng.randint(4, 16))
    elif kind == "sssp":
        c.update(kind="sssp", graph="rmat", scale=rng.randint(10, 21), ef=rng.randint(8, 20))
    elif kind == "grid":
        c.update(kind=rng.choice(["bfs", "sssp"]), graph="grid", rows=_log(rng, 20, 600),
                 cols=_log(rng, 20, 600))
    elif kind in ("push", "pull"):
        c.update(kind="pr", mode=kind, n=_log(rng, 1000, 2000000), ef=rng.randint(4, 16))
    elif kind in ("batch-bfs", "batch-sssp"):
        algo = kind.split("-")[1]
        c.update(kind="batch", algo=algo, scale=rng.randint(10, 21 if algo == "bfs" else 19),
                 ef=rng.randint(8, 20), k=_log(rng, 1, 64))
    else:
        scale = rng.randint(8, 18)
        c.update(kind="wide", algo=rng.choice(["bfs", "cc", "sssp"]), scale=scale,
                 ef=rng.randint(8, 16), stride=max(1, _log(rng, 1 << 20, 1 << 32) >> scale))
    return c


# ---- graphs -------------------------------------------------------------------


def _csr(n, src, dst):
    """Sorted unique edges without self-loops as (offsets, destinations)."""
    keep = src != dst
    key = torch.unique(src[keep] * n + dst[keep])
    off = torch.zeros(n + 1, dtype=torch.int64, device=key.device)
    off[1:] = torch.cumsum(torch.bincount(key // n, minlength=n), 0)
    return off, key % n


def _rmat_edges(n, ef, seed):
    """n * ef edges over n vertices with R-MAT's quadrants (a, b, c = 0.57,
    0.19, 0.19); ids past n fold back into the range."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    count = n * ef
    a, b, c = T.RMAT_ABC
    src = torch.zeros(count, dtype=torch.int64, device="cuda")
    dst = torch.zeros(count, dtype=torch.int64, device="cuda")
    for _ in range(max(1, (n - 1).bit_length())):
        r = torch.rand(count, generator=gen, device="cuda")
        src = src * 2 + (r >= a + b)
        dst = dst * 2 + (((r >= a) & (r < a + b)) | (r >= a + b + c))
    return src % n, dst % n


def _directed(n, ef, seed):
    return _csr(n, *_rmat_edges(n, ef, seed))


def _transpose(n, off, dst):
    """In-lists (offsets, sources) and out-degrees."""
    deg = off[1:] - off[:-1]
    src = torch.repeat_interleave(torch.arange(n, device=off.device), deg)
    ioff, isrc = _csr(n, dst, src)
    return ioff, isrc, deg


def _np(t, dtype):
    return t.cpu().numpy().astype(dtype)


def _star(leaves, path, seed):
    """A hub with `leaves` out-edges and a path of `path` vertices behind its
    last leaf; the ids are shuffled."""
    n = 1 + leaves + path
    name = np.random.default_rng(seed).permutation(n)
    src = np.concatenate([np.zeros(leaves, np.int64), np.arange(leaves, n - 1)])
    dst = np.arange(1, n)
    order = np.lexsort((name[dst], name[src]))
    off = np.zeros(n + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(name[src], minlength=n))
    return off, name[dst][order].astype(np.uint32), int(name[0])


def _grid(rows, cols, seed):
    """Four neighbours each way, one weight in [1, 64] per undirected edge."""
    rng = np.random.default_rng(seed)
    at = np.arange(rows * cols).reshape(rows, cols)
    u = np.concatenate([at[:, :-1].ravel(), at[:-1].ravel()])
    v = np.concatenate([at[:, 1:].ravel(), at[1:].ravel()])
    w = rng.integers(1, 65, len(u))
    src, dst, w = np.concatenate([u, v]), np.concatenate([v, u]), np.concatenate([w, w])
    order = np.lexsort((dst, src))
    off = np.zeros(rows * cols + 1, np.uint64)
    off[1:] = np.cumsum(np.bincount(src, minlength=rows * cols))
    return off, dst[order].astype(np.uint32), w[order].astype(np.uint32), int(
        rng.integers(rows * cols))


def _sources(off, k, seed):
    """k seeded vertices that have edges."""
    have = np.flatnonzero(np.diff(off.astype(np.int64)))
    return np.random.default_rng(seed).choice(have, k).astype(np.uint32)


def _store(g, case):
    part = case["part"]
    if case["budget"] >= 1.0:
        g.store_config(None, part)
    else:
        g.store_config(int(case["budget"] * g.m * g.edge_bytes), part)


# ---- a case ---------------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    state = {"kind": kind}
    if kind == "wide":
        scale, stride = case["scale"], case["stride"]
        with T.Graph.rmat(scale, case["ef"], seed=seed, weights=True) as small:
            off, dst, w, _ = small.export()
        deg = np.diff(off.astype(np.int64))
        ids = np.flatnonzero(deg).astype(np.uint64) * np.uint64(stride)
        loff = np.concatenate([[0], np.cumsum(deg[deg > 0])]).astype(np.uint64)
        n = (1 << scale) * stride + 12345
        g = T.Graph64(n, ids, loff, dst.astype(np.uint64) * np.uint64(stride), w)
        if case["budget"] < 1.0:
            g.store_config(int(case["budget"] * g.m * 16), case["part"])
        src = int(np.random.default_rng(seed).choice(ids))
        every = np.arange(1 << scale, dtype=np.uint64) * np.uint64(stride)
        state.update(g=g, algo=case["algo"], src=src, ids=every)
        return state
    if kind == "batch":
        g = T.Graph.rmat(case["scale"], case["ef"], seed=seed, weights=True)
        _store(g, case)
        state.update(g=g, algo=case["algo"], srcs=_sources(g.offsets(), case["k"], seed))
        return state
    if kind == "pr":
        off, dst = _directed(case["n"], case["ef"], seed)
        if case["mode"] == "push":
            g = T.Graph.from_arrays(_np(off, np.uint64), _np(dst, np.uint32))
        else:
            off, src, deg = _transpose(case["n"], off, dst)
            g = T.Graph.from_arrays(_np(off, np.uint64), _np(src, np.uint32),
                                    outdeg=_np(deg, np.uint32))
        _store(g, case)
        state.update(g=g, mode=case["mode"], out=np.empty(g.n, np.float32))
        return state
    src = None
    if case["graph"] == "rmat":
        g = T.Graph.rmat(case["scale"], case["ef"], seed=seed, weights=kind == "sssp")
        src = int(_sources(g.offsets(), 1, seed)[0])
    elif case["graph"] == "directed":
        off, dst = _directed(case["n"], case["ef"], seed)
        g = T.Graph.from_arrays(_np(off, np.uint64), _np(dst, np.uint32))
    elif case["graph"] == "star":
        off, dst, src = _star(case["leaves"], case["path"], seed)
        g = T.Graph.from_arrays(off, dst)
    else:
        off, dst, w, src = _grid(case["rows"], case["cols"], seed)
        g = T.Graph.from_arrays(off, dst, w if kind == "sssp" else None)
        g.set_option("symmetric", 1)
    _store(g, case)
    state.update(g=g, src=src, out=np.empty(g.n, np.uint32))
    return state


def run(state):
    g, kind = state["g"], state["kind"]
    if kind == "bfs":
        out, st = g.bfs(state["src"], out=state["out"])
        return {"levels": out, "reached": st.reached}
    if kind == "sssp":
        out, st = g.sssp(state["src"], out=state["out"])
        return {"distances": out, "reached": st.reached}
    if kind == "cc":
        return {"labels": g.cc(out=state["out"])[0]}
    if kind == "pr":
        return {"ranks": g.pr(state["mode"], DAMPING, TOL, MAX_ITER, out=state["out"])[0]}
    if kind == "batch":
        r = g.batch(state["algo"], state["srcs"])
        return {"hash": r["hash"].view(np.int64), "reached": r["reached"].view(np.int64),
                "depth": r["depth"]}
    r = g.cc() if state["algo"] == "cc" else getattr(g, state["algo"])(state["src"])
    return {"hash": np.array([r["hash"]], np.uint64).view(np.int64), "reached": r["reached"],
            "depth": r["depth"], "values": g.values(state["ids"]).view(np.int64)}


def work(case):
    """Records and per-vertex state read once, values written once."""
    kind, weighted = case["kind"], case["kind"] in ("sssp", "wide", "batch")
    if kind == "wide":
        n, k = (1 << case["scale"]) * case["stride"], 1 << case["scale"]
        # every value is written, then digested
        return {"bytes": 16.0 * n + 16.0 * k * case["ef"] + 24.0 * k, "flops": 0.0}
    if "scale" in case:
        n = 1 << case["scale"]
        m = n * case["ef"]
    elif case.get("graph") == "star":
        n = 1 + case["leaves"] + case["path"]
        m = n - 1
    elif case.get("graph") == "grid":
        n = case["rows"] * case["cols"]
        m = 4 * n - 2 * (case["rows"] + case["cols"])
        weighted = kind == "sssp"
    else:
        n = case["n"]
        m = n * case["ef"]
    rec = 8 if weighted else 4
    if kind == "pr":  # each iteration: every record, two reads and two writes a vertex
        return {"bytes": MAX_ITER * (rec * m + 16.0 * n), "flops": MAX_ITER * (m + 3.0 * n)}
    if kind == "batch":  # the lanes share the records; each has its own values
        return {"bytes": rec * m + (16.0 if case["algo"] == "bfs" else 8.0 * case["k"]) * n,
                "flops": 0.0}
    if kind in ("bfs", "cc") and case["graph"] == "rmat":
        # undirected: one word names a neighbour of each vertex, few lists are read
        return {"bytes": 12.0 * n, "flops": 0.0}
    return {"bytes": rec * m + 12.0 * n, "flops": 0.0}


def exact(case, seed):
    """PageRank's iterations in 64 bits; everything else is whole numbers."""
    if case["kind"] != "pr":
        return None
    n, tol = case["n"], float(np.float32(TOL))
    a = float(np.float32(DAMPING))
    off, dst = _directed(n, case["ef"], seed)
    deg = (off[1:] - off[:-1])
    src = torch.repeat_interleave(torch.arange(n, device="cuda"), deg)
    od = deg.double()
    inv = torch.where(deg > 0, 1.0 / od.clamp(min=1.0), torch.zeros_like(od))
    active = torch.ones(n, dtype=torch.bool, device="cuda")
    if case["mode"] == "push":
        rank = torch.full((n,), 1.0 - a, dtype=torch.float64, device="cuda")
        delta, res = rank * a * inv, torch.zeros_like(rank)
        for _ in range(MAX_ITER):
            give = torch.where(active, delta, torch.zeros_like(delta))
            res.index_add_(0, dst, give[src])
            active = res > tol
            rank += torch.where(active, res, torch.zeros_like(res))
            delta = torch.where(active, res * a * inv, delta)
            res = torch.where(active, torch.zeros_like(res), res)
            if not bool(active.any()):
                break
    else:
        rank = torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda")
        for _ in range(MAX_ITER):
            total = torch.zeros_like(rank).index_add_(0, dst, (rank * inv)[src])
            new = torch.where(active, (1.0 - a) + a * total, rank)
            active = active & ((new - rank).abs() > tol)
            rank = new
            if not bool(active.any()):
                break
    return {"ranks": rank}
