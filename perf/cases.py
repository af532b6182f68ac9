"""The calls this library is used for, as measurable cases.

Every case is one call of a public entry point on a graph that is already resident on the GPU
(the upload and its plan are what a program does once): PageRank in its directions and number
kinds, SpMV, personalised PageRank and the many-graph batch. Graphs are RMAT (the skewed degree
distribution of web and social graphs) or Erdos-Renyi (evenly spread sources, any vertex count),
at the sizes of bench.py and the tests.
"""
import math

import numpy as np
import torch

import accelgraph_amd as ag

DAMP = 0.85

KINDS = {"fixed64": ag.KIND_FIXED64, "fixed32": ag.KIND_FIXED32, "fixed16": ag.KIND_FIXED16,
         "quant32": ag.KIND_QUANT32, "quant16": ag.KIND_QUANT16, "quant8": ag.KIND_QUANT8}
KIND_BYTES = {"fixed64": 8, "fixed32": 4, "fixed16": 2, "quant32": 4, "quant16": 2, "quant8": 1,
              "f32": 4}
STORAGE = {"f32": ag.STORE_F32, "bf16": ag.STORE_BF16, "f16": ag.STORE_F16}

_device = None


def _dev():
    global _device
    if _device is None:
        _device = ag.Device(0)
    return _device


def listed():
    return [
        # the smallest call: a graph of a few thousand vertices, all launches and host work
        {"name": "pr_rmat12_l1", "op": "pagerank", "graph": "rmat", "scale": 12, "ef": 16,
         "kind": "f32", "storage": "f32", "stop": "l1", "tol": 1e-4, "iters": 100},
        # PageRank to L1 <= 1e-4 on RMAT-16, the small configuration of bench.py
        {"name": "pr_rmat16_l1", "op": "pagerank", "graph": "rmat", "scale": 16, "ef": 16,
         "kind": "f32", "storage": "f32", "stop": "l1", "tol": 1e-4, "iters": 100},
        # the headline: FP32 iterations on RMAT-25, the command line's 20 of them
        {"name": "pr_rmat25_20it", "op": "pagerank", "graph": "rmat", "scale": 25, "ef": 16,
         "kind": "f32", "storage": "f32", "stop": "none", "tol": 0.0, "iters": 20},
        # evenly spread sources and a vertex count that is no power of two, to convergence
        {"name": "pr_er5m_l1", "op": "pagerank", "graph": "er", "n": 5000011, "m": 80000000,
         "kind": "f32", "storage": "f32", "stop": "l1", "tol": 1e-6, "iters": 100},
        # the fixed-point pull under the reference's stop rule (bit-exact ranks)
        {"name": "pr_fixed32_rmat22", "op": "pagerank", "graph": "rmat", "scale": 22, "ef": 16,
         "kind": "fixed32", "storage": "f32", "stop": "active", "tol": 1e-4, "iters": 20},
        # a quantised pull on a graph whose contribution vector fits the caches
        {"name": "pr_quant16_rmat20", "op": "pagerank", "graph": "rmat", "scale": 20, "ef": 16,
         "kind": "quant16", "storage": "f32", "stop": "active", "tol": 1e-4, "iters": 20},
        # the push direction
        {"name": "pr_push_rmat22", "op": "push", "graph": "rmat", "scale": 22, "ef": 16,
         "kind": "f32", "iters": 10},
        # the data-driven pull over worklists
        {"name": "pr_dd_rmat19", "op": "data_driven", "graph": "rmat", "scale": 19, "ef": 16,
         "eps": 1e-4, "iters": 100},
        # one weighted FP32 product, x and y in host memory (bench.py's SpMV)
        {"name": "spmv_rmat22_w", "op": "spmv", "graph": "rmat", "scale": 22, "ef": 16,
         "weighted": True, "form": "f32"},
        # one fixed-point product on a mid-sized graph of odd size
        {"name": "spmv_fixed_er300k", "op": "spmv", "graph": "er", "n": 300007, "m": 4800011,
         "weighted": False, "form": "fixed"},
        # 64 personalised columns, 16-bit storage refined in FP32, to convergence
        {"name": "ppr64_rmat18", "op": "ppr", "graph": "rmat", "scale": 18, "ef": 16, "k": 64,
         "storage": "bf16", "tol": 1e-6, "iters": 300},
        # many small graphs in one solve
        {"name": "batch48", "op": "batch", "count": 48, "lo": 10, "hi": 15, "ef": 16,
         "tol": 1e-6, "iters": 100},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_graph(rng, lo, hi):
    """An RMAT or Erdos-Renyi graph of 2^lo to 2^hi vertices, 4 to 24 edges a vertex."""
    ef = rng.randint(4, 24)
    if rng.random() < 0.6:
        return {"graph": "rmat", "scale": rng.randint(lo, hi), "ef": ef}
    n = _log_int(rng, 1 << lo, 1 << hi)
    return {"graph": "er", "n": n, "m": n * ef + rng.randint(0, 1000)}


def draw(rng):
    op = rng.choice(["pagerank", "pagerank", "integer", "push", "data_driven", "spmv", "spmv",
                     "ppr", "batch"])
    if op == "pagerank":
        c = {"op": op, **_draw_graph(rng, 12, 24), "kind": "f32",
             "storage": rng.choice(["f32", "f32", "f32", "bf16", "f16"])}
        if rng.random() < 0.5:
            return {**c, "stop": "l1", "tol": rng.choice([1e-4, 1e-5, 1e-6]), "iters": 100}
        return {**c, "storage": "f32", "stop": "none", "tol": 0.0, "iters": rng.randint(1, 20)}
    if op == "integer":
        return {"op": "pagerank", **_draw_graph(rng, 12, 23), "kind": rng.choice(sorted(KINDS)),
                "storage": "f32", "stop": "active", "tol": 1e-4, "iters": rng.randint(5, 30)}
    if op == "push":
        return {"op": op, **_draw_graph(rng, 14, 22),
                "kind": rng.choice(["f32", "f32", "fixed64", "fixed32"]),
                "iters": rng.randint(2, 20)}
    if op == "data_driven":
        return {"op": op, **_draw_graph(rng, 14, 21), "eps": 1e-4, "iters": 100}
    if op == "spmv":
        return {"op": op, **_draw_graph(rng, 14, 22), "weighted": rng.random() < 0.5,
                "form": rng.choice(["f32", "f32", "fixed", "push", "push_fixed"])}
    if op == "ppr":
        return {"op": op, **_draw_graph(rng, 12, 19), "k": _log_int(rng, 1, 64),
                "storage": rng.choice(sorted(STORAGE)), "tol": 1e-6, "iters": 300}
    lo = rng.randint(8, 11)
    return {"op": op, "count": rng.randint(4, 60), "lo": lo, "hi": rng.randint(lo + 1, 15),
            "ef": rng.randint(6, 20), "tol": 1e-6, "iters": 100}


# ------------------------------------------------------------------ inputs

def _graph(case, seed):
    s = (ag.DEFAULT_SEED + 7919 * int(seed)) & 0x7FFFFFFF
    if case["graph"] == "rmat":
        return ag.Graph.rmat_gpu(_dev(), case["scale"], case["ef"], seed=s)
    return ag.Graph.erdos_renyi_gpu(_dev(), case["n"], case["m"], seed=s)


def _batch_graphs(case, seed):
    span = case["hi"] - case["lo"] + 1
    return [ag.Graph.rmat(case["lo"] + i % span, case["ef"],
                          seed=(ag.DEFAULT_SEED + 7919 * int(seed) + 104729 * i) & 0x7FFFFFFF)
            for i in range(case["count"])]


def _vector(case, g, seed):
    rng = np.random.default_rng(1000003 + int(seed))
    if case["form"] == "fixed":
        return rng.integers(0, 1 << 18, g.n, dtype=np.uint32)           # Q16.16 codes
    if case["form"] == "push_fixed":
        return rng.integers(0, 1 << 34, g.n, dtype=np.uint64)           # Q32.32 codes
    return rng.random(g.n, dtype=np.float32)


def _weights(case, g, seed):
    """Puts a weight on every edge of a weighted case's graph."""
    if case.get("weighted"):
        w = np.random.default_rng(2000003 + int(seed)).random(g.m, dtype=np.float32)
        g.set_weights(w + np.float32(1e-6))


def _seeds(case, n, seed):
    s = np.random.default_rng(3000017 + int(seed)).integers(0, n, case["k"], dtype=np.uint32)
    s[0] = ag.PPR_UNIFORM
    return s


def prepare(case, seed):
    if case["op"] == "batch":
        graphs = _batch_graphs(case, seed)
        b = ag.Batch(_dev(), graphs)
        for g in graphs:
            g.close()
        return {"case": case, "batch": b}
    g = _graph(case, seed)
    _weights(case, g, seed)
    state = {"case": case, "dg": _dev().upload(g, weights=bool(case.get("weighted")))}
    if case["op"] == "spmv":
        state["x"] = _vector(case, g, seed)
    if case["op"] == "ppr":
        state["seeds"] = _seeds(case, g.n, seed)
    g.close()
    return state


# ------------------------------------------------------------------ one call

STOPS = {"l1": ag.STOP_L1, "none": ag.STOP_NONE, "active": ag.STOP_ACTIVE}


def _pagerank_result(case, r):
    if case["kind"] == "f32":
        return {"ranks": r.ranks}
    # integer sums: the run's course is exact as well
    return {"ranks": r.ranks, "iterations": r.iterations,
            "active": r.hist_active.view(np.int32)}


def run(state):
    case, dg = state["case"], state.get("dg")
    op = case["op"]
    if op == "pagerank":
        kw = {"max_iterations": case["iters"], "stop_rule": STOPS[case["stop"]]}
        if case["stop"] == "active":
            kw["epsilon"] = case["tol"]
        else:
            kw.update(l1_tolerance=case["tol"], init=ag.INIT_UNIFORM)
        if case["kind"] == "f32":
            r = dg.pagerank(storage=STORAGE[case["storage"]], **kw)
        else:
            r = dg.pagerank(kind=KINDS[case["kind"]], **kw)
        return _pagerank_result(case, r)
    if op == "push":
        kind = ag.KIND_F32 if case["kind"] == "f32" else KINDS[case["kind"]]
        r = dg.pagerank(kind=kind, direction=ag.DIR_PUSH, max_iterations=case["iters"],
                        stop_rule=ag.STOP_NONE, init=ag.INIT_UNIFORM)
        return _pagerank_result(case, r)
    if op == "data_driven":
        r = dg.pagerank(direction=ag.DIR_DATA_DRIVEN, max_iterations=case["iters"],
                        epsilon=case["eps"])
        return {"ranks": r.ranks}
    if op == "spmv":
        call = {"f32": dg.spmv, "fixed": dg.spmv_fixed, "push": dg.spmv_push,
                "push_fixed": dg.spmv_push_fixed}[case["form"]]
        y, _ = call(state["x"])
        return {"y": y.view(np.int64) if y.dtype == np.uint64 else y}
    if op == "ppr":
        ranks, _, _ = dg.ppr(state["seeds"], max_iterations=case["iters"],
                             l1_tolerance=case["tol"], storage=STORAGE[case["storage"]])
        return {"ranks": ranks}
    ranks, _, _, _ = state["batch"].pagerank(max_iterations=case["iters"],
                                             l1_tolerance=case["tol"])
    return {"ranks": ranks}


# ------------------------------------------------------------------ the work of a call

def _size(case):
    if case["graph"] == "rmat":
        n = 1 << case["scale"]
        return n, n * case["ef"]
    return case["n"], case["m"]


def _iterations(case):
    """About how many iterations a call takes: RMAT graphs need some 8 per decade of the
    tolerance, evenly connected ones fewer than 2."""
    if case.get("stop", "l1") == "none" or case["op"] == "push":
        return case["iters"]
    tol = case.get("tol", case.get("eps", 1e-4))
    per_decade = 8.0 if case.get("graph", "rmat") == "rmat" else 1.7
    return max(1, min(case["iters"], round(-math.log10(tol) * per_decade)))


def work(case):
    op = case["op"]
    if op == "batch":
        span = case["hi"] - case["lo"] + 1
        n = sum(1 << (case["lo"] + i % span) for i in range(case["count"]))
        m, it = n * case["ef"], _iterations(case)
        return {"bytes": it * (4 * m + 20 * n) + 4 * n, "flops": it * 2 * m}
    n, m = _size(case)
    if op == "spmv":
        e = 8 if case["form"] in ("fixed", "push_fixed") else 4
        return {"bytes": (8 if case["weighted"] else 4) * m + (4 + 2 * e) * n, "flops": 2 * m}
    it = _iterations(case)
    if op == "ppr":
        # per iteration: the edge list, every column's rank twice and its contribution twice
        c = 4 if case["storage"] == "f32" else 2
        return {"bytes": it * (4 * m + 8 * n + (8 + 2 * c) * n * case["k"]) + 4 * n * case["k"],
                "flops": it * 2 * m * case["k"]}
    # per iteration: the edge list, offsets and out-degrees, ranks and contributions twice each
    c = KIND_BYTES[case.get("kind", "f32")]
    return {"bytes": it * (4 * m + 8 * n + 8 * n + 2 * c * n) + 4 * n, "flops": it * 2 * m}


# ------------------------------------------------------------------ the result in 64 bits

def _on_gpu(a, dtype):
    a = np.ascontiguousarray(a)
    return torch.from_numpy(a.view(np.int32) if a.dtype == np.uint32 else a).cuda().to(dtype)


class _Pull:
    """y[v] = sum over in-edges (u -> v) of x[u], for one or more columns, in 64 bits."""

    def __init__(self, g):
        self.src = _on_gpu(g.inv_src, torch.int64)      # row after row of the inverse graph
        self.len = _on_gpu(g.in_degree, torch.int64).split(1 << 22)    # some rows at a time
        self.edges = [int(d.sum()) for d in self.len]
        self.outdeg = _on_gpu(g.out_degree, torch.float64)

    def __call__(self, x, w=None):
        t = x[self.src]
        if w is not None:
            t = t * w
        return torch.cat([torch.segment_reduce(part, "sum", lengths=d, axis=0, initial=0, unsafe=True)
                          for part, d in zip(t.split(self.edges), self.len)])

    def iterate(self, rank, restart):
        od = self.outdeg if rank.dim() == 1 else self.outdeg[:, None]
        c = torch.where(od > 0, rank / od.clamp(min=1.0), torch.zeros_like(rank))
        return restart + DAMP * self(c)


def _solve(g, iters, stop, tol):
    """Scaled ranks from the uniform start; stops after the first iteration whose L1 change is
    within the tolerance."""
    p = _Pull(g)
    rank = torch.ones(g.n, dtype=torch.float64, device="cuda")
    for _ in range(iters):
        nxt = p.iterate(rank, 1.0 - DAMP)
        delta = float((nxt - rank).abs().sum()) / g.n
        rank = nxt
        if stop == "l1" and delta <= tol:
            break
    return rank / g.n


def exact(case, seed):
    op = case["op"]
    if op == "batch":
        return {"ranks": [_solve(g, case["iters"], "l1", case["tol"])
                          for g in _batch_graphs(case, seed)]}
    if op == "data_driven" or case.get("kind", "f32") != "f32":
        return None     # defined by thresholds and integer codes, not by a sum of real numbers
    if op == "spmv" and case["form"] in ("fixed", "push_fixed"):
        return None
    g = _graph(case, seed)
    if op == "spmv":
        _weights(case, g, seed)
        x = torch.from_numpy(_vector(case, g, seed)).cuda().double()
        p = _Pull(g)
        if case["weighted"]:
            return {"y": p(x, _on_gpu(g.inv_weight, torch.float64))}
        return {"y": p(x) * float(np.float32(0.0001))}
    if op == "push":
        return {"ranks": _solve(g, case["iters"], "none", 0.0)}
    if op == "pagerank":
        if case["storage"] != "f32":    # 16-bit storage converges to the solution its own way
            return {"ranks": _solve(g, 400, "l1", 1e-12)}
        return {"ranks": _solve(g, case["iters"], case["stop"], case["tol"])}
    # personalised columns: the solution itself, which every storage converges to
    p = _Pull(g)
    restart = torch.zeros(g.n, case["k"], dtype=torch.float64, device="cuda")
    for c, s in enumerate(_seeds(case, g.n, seed)):
        if s == ag.PPR_UNIFORM:
            restart[:, c] = 1.0 - DAMP
        else:
            restart[int(s), c] = (1.0 - DAMP) * g.n
    rank = torch.ones_like(restart)
    for _ in range(170):
        rank = p.iterate(rank, restart)
    return {"ranks": rank / g.n}
