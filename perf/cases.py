"""The work that this library is measured on, through its public Python entry points.

A case is a dict of plain values.  `path` names what a program does:

  bfs     one BFS from one root on a graph resident on the device, its levels
          and parents on the host afterwards (DeviceGraph.bfs)
  many    a sequence of roots on one resident graph, as Graph500-style programs
          run it, and the last root's levels and parents (DeviceGraph.bfs_many,
          DeviceGraph.results)
  batch   many instances of uneven size in one launch, every instance's levels
          and parents (Batch.run, Batch.results)
  load    a .cbd file loaded, laid out and searched once: the reference's own
          program from its file to its answer (DeviceGraph.load, bfs)
  build   the same from a CSR that the program holds (DeviceGraph.build, bfs)
  compat  the reference's own BFS entry point on a host CSR
          (run_custom_bfs_test)
  train   the direction selector trained on samples of BFS levels
          (Selector.train)

Sizes are those of the repository's configurations, benchmark, tests and
training set, or generic ones between them.  The graphs are the library's
seeded RMAT, Erdos-Renyi and grid generators, with ids permuted.
"""
import math
import os
import tempfile

import numpy as np

import albba_amd as A
from albba_amd import workloads as W

_SELECTOR = os.path.join(os.path.dirname(os.path.abspath(A.__file__)), "selector.txt")
_POLICY = {"heuristic": A.SWITCH_HEURISTIC, "learned": A.SWITCH_LEARNED}
# layouts that the autotuner picks for the families of the batched mix
_BATCH_LAYOUT = {"rmat": (128, 256), "er": (128, 128), "grid": (32, 32)}
_LR = 3e-3
_context = None


def _ctx():
    """A program has one context per device."""
    global _context
    if _context is None:
        _context = A.Context(0)
    return _context


def listed():
    return [
        # the smallest call: a query on a graph of a thousand vertices
        dict(name="rmat10", path="bfs", kind="rmat", scale=10, edgefactor=16, C=64, sigma=1024, policy="heuristic"),
        # RMAT s16, the smallest configuration of the benchmark
        dict(name="rmat16", path="bfs", kind="rmat", scale=16, edgefactor=16, C=64, sigma=4096, policy="heuristic"),
        # an ordinary query on a graph without hubs, of no round size
        dict(name="er_odd", path="bfs", kind="er", n=500009, mean_degree=9.0, C=32, sigma=256, policy="learned"),
        # a ragged high-diameter graph: hundreds of levels of a few hundred vertices
        dict(name="grid_odd", path="bfs", kind="grid", rows=601, cols=1009, C=64, sigma=4096, policy="learned"),
        # the high-diameter configuration: thousands of levels
        dict(name="grid4096", path="bfs", kind="grid", rows=4096, cols=4096, C=64, sigma=4096, policy="heuristic"),
        # 64 roots with the reference's own direction switch (RMAT s22)
        dict(name="rmat22_heuristic", path="many", kind="rmat", scale=22, edgefactor=16, C=64, sigma=4096,
             policy="heuristic", roots=64),
        # the headline: 64 roots with the learned switch (RMAT s24)
        dict(name="rmat24_learned", path="many", kind="rmat", scale=24, edgefactor=16, C=64, sigma=4096,
             policy="learned", roots=64),
        # instances of the batched mix (RMAT, Erdos-Renyi and grids together)
        dict(name="batch24", path="batch", count=24, mix=6, policy="learned"),
        # the reference's program: from a .cbd file to levels and parents
        dict(name="load_rmat20", path="load", kind="rmat", scale=20, edgefactor=16, C=64, sigma=4096,
             policy="heuristic"),
        # a graph that a program made itself, built and searched once
        dict(name="build_rmat21", path="build", kind="rmat", scale=21, edgefactor=16, C=64, sigma=4096,
             policy="learned"),
        # a reference application linked against the library
        dict(name="compat_rmat18", path="compat", kind="rmat", scale=18, edgefactor=16),
        # training on the levels of a few graphs
        dict(name="train_9000", path="train", samples=9000, steps=200),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _graph_spec(rng, top):
    """A graph of at most about 2**top vertices (RMAT a scale of at most top)."""
    kind = rng.choice(("rmat", "rmat", "er", "grid"))
    if kind == "rmat":
        return dict(kind=kind, scale=rng.randint(8, top), edgefactor=rng.randint(4, 24))
    if kind == "er":
        return dict(kind=kind, n=_log_int(rng, 300, 1 << top), mean_degree=round(rng.uniform(2.0, 24.0), 2))
    side = 1 << (top // 2)
    return dict(kind=kind, rows=_log_int(rng, 8, side), cols=_log_int(rng, 8, side))


def draw(rng):
    path = rng.choice(("bfs", "bfs", "bfs", "many", "many", "batch", "load", "build", "compat", "train"))
    if path == "train":
        return dict(path=path, samples=_log_int(rng, 200, 33000), steps=rng.randint(20, 200))
    if path == "batch":
        return dict(path=path, count=rng.randint(2, 24), mix=rng.randint(1, 10000),
                    policy=rng.choice(("heuristic", "learned")))
    if path == "compat":
        return dict(path=path, **_graph_spec(rng, 18))
    C, sigma = rng.choice(((64, 4096), (64, 4096), (64, 1024), (32, 256), (128, 256), (16, 64)))
    case = dict(path=path, C=C, sigma=sigma, policy=rng.choice(("heuristic", "learned")))
    if path == "many":
        spec = _graph_spec(rng, 22)
        # a grid's BFS takes thousands of levels: fewer of them
        return dict(case, roots=rng.randint(2, 5) if spec["kind"] == "grid" else rng.randint(4, 64), **spec)
    return dict(case, **_graph_spec(rng, 22 if path == "bfs" else 20))


def _gen_args(case, seed):
    if case["kind"] == "rmat":
        return dict(scale=case["scale"], edgefactor=case["edgefactor"], seed=seed + 1, perm_seed=seed + 2)
    if case["kind"] == "er":
        return dict(n=case["n"], mean_degree=case["mean_degree"], seed=seed + 1, perm_seed=seed + 2)
    return dict(rows=case["rows"], cols=case["cols"], p_remove=0.1, seed=seed + 1, perm_seed=seed + 2)


def _roots(g, case, count, seed):
    # RMAT: any vertex with an edge; the others: the largest component
    r = g.pick_roots(count, seed + 3, largest_cc=case["kind"] != "rmat")
    return np.resize(r if r.size else np.zeros(1, np.int32), count).astype(np.int32)


def _host_graph(case, seed):
    """The case's graph on the host (generated on the device)."""
    dg, g = A.DeviceGraph.generate(_ctx(), case["kind"], 64, 4096, 1, **_gen_args(case, seed))
    dg.close()
    return g


def _selector():
    sel = A.Selector(_ctx())
    sel.load(_SELECTOR)
    return sel


def prepare(case, seed):
    ctx, path = _ctx(), case["path"]
    state = dict(case=case, path=path)
    if path == "train":
        # features lie in [0, 1]; targets are relative log times, around zero
        # in every sample, that depend on the features
        rng = np.random.default_rng(seed)
        x = rng.random((case["samples"], A.NUM_FEATURES), dtype=np.float32)
        mix = rng.normal(size=(A.NUM_FEATURES, 4))
        t = np.tanh(x @ mix) + 0.3 * rng.normal(size=(case["samples"], 4))
        state["x"], state["t"] = x, (t - t.mean(axis=1, keepdims=True)).astype(np.float32)
        state["selector"] = A.Selector(ctx, seed=seed + 1)
        state["params"] = state["selector"].params
        return state
    state["policy"] = _POLICY[case.get("policy", "heuristic")]
    state["selector"] = _selector() if case.get("policy") == "learned" else None
    if path == "batch":
        graphs, roots = [], []
        for i, (kind, p) in enumerate(W.batch_specs(case["count"], case["mix"])):
            C, sigma = _BATCH_LAYOUT[kind]
            p = dict(p, seed=p["seed"] + seed, perm_seed=p["perm_seed"] + seed)
            dg, g = A.DeviceGraph.generate(ctx, kind, C, sigma, 1, **W.gen_args(kind, p))
            graphs.append(dg)
            roots.append(W.root_of(kind, g, i))
        state["graphs"], state["roots"] = graphs, roots
        state["batch"] = A.Batch(ctx, graphs)
        return state
    if path in ("bfs", "many"):
        dg, g = A.DeviceGraph.generate(ctx, case["kind"], case["C"], case["sigma"], 1, **_gen_args(case, seed))
        state["graph"] = dg
        state["roots"] = _roots(g, case, case.get("roots", 1), seed)
        return state
    g = _host_graph(case, seed)
    state["roots"] = _roots(g, case, 1, seed)
    if path == "load":
        state["dir"] = tempfile.TemporaryDirectory()
        state["file"] = os.path.join(state["dir"].name, "graph.cbd")
        g.write_cbd(state["file"])
    elif path == "build":
        state["csr"] = g
    else:
        state["csr"] = (g.n, g.row_ptr.astype(np.int32), g.col.copy())
    return state


def _bfs(state, dg):
    o = dg.bfs(int(state["roots"][0]), policy=state["policy"], selector=state["selector"])
    return {k: o[k] for k in ("level", "parent", "num_levels", "reached", "edges_in_component")}


def run(state):
    path, case = state["path"], state["case"]
    if path == "bfs":
        return _bfs(state, state["graph"])
    if path == "many":
        o = state["graph"].bfs_many(state["roots"], policy=state["policy"], selector=state["selector"])
        level, parent = state["graph"].results()
        return dict(level=level, parent=parent, num_levels=o["num_levels"], reached=o["reached"],
                    edges_in_component=o["edges_in_component"])
    if path == "batch":
        b = state["batch"]
        o = b.run(state["roots"], policy=state["policy"], selector=state["selector"])
        return dict(results=[b.results(i) for i in range(case["count"])], num_levels=o["num_levels"],
                    reached=o["reached"], edges_in_component=o["edges_in_component"])
    if path in ("load", "build"):
        if path == "load":
            dg = A.DeviceGraph.load(_ctx(), state["file"], case["C"], case["sigma"], 1)
        else:
            dg = A.DeviceGraph.build(_ctx(), state["csr"], case["C"], case["sigma"], 1)
        out = _bfs(state, dg)
        dg.close()
        return out
    if path == "compat":
        o = A.run_custom_bfs_test(*state["csr"])
        # the frontier sizes as the caller's array holds them, one entry per
        # vertex of which the levels fill the first
        out = {k: o[k] for k in ("num_iter", "num_vex", "nnzx")}
        out["frontier"] = np.pad(o["frontier"], (0, state["csr"][0] - o["frontier"].size))
        return out
    sel = state["selector"]
    sel.params = state["params"]
    loss = sel.train(state["x"], state["t"], steps=case["steps"], lr=_LR)
    return dict(params=sel.params, loss=loss)


def _size(case):
    """Vertices and (nearly) stored entries of the case's graph."""
    if case["kind"] == "rmat":
        n = 1 << case["scale"]
        return n, 2 * case["edgefactor"] * n
    if case["kind"] == "er":
        return case["n"], int(case["n"] * case["mean_degree"])
    n = case["rows"] * case["cols"]
    return n, int(0.9 * 4 * n)


def work(case):
    """A search cannot do without a row pointer and one column entry of every
    vertex, nor without writing its level and parent (20 bytes a vertex); a
    build or load reads the matrix and writes its layout besides."""
    path = case["path"]
    if path == "train":
        per_sample = 12 * 32 + 32 * 32 + 32 * 4
        return {"bytes": case["samples"] * 64 + 4 * A.MLP_NPARAM * 2,
                "flops": 6.0 * per_sample * case["samples"] * case["steps"]}
    if path == "batch":
        n = sum(W.vertices(*s) for s in W.batch_specs(case["count"], case["mix"]))
        return {"bytes": 20 * n, "flops": 0}
    n, m = _size(case)
    if path in ("bfs", "many"):
        return {"bytes": 20 * n * case.get("roots", 1), "flops": 0}
    return {"bytes": 8 * m + 40 * n, "flops": 0}


def _train_exact(x, t, p, steps):
    """Full-batch Adam on the MLP 12 -> 32 -> 32 -> 4 in 64 bits."""
    x, t, p = x.astype(np.float64), t.astype(np.float64), p.astype(np.float64)
    shapes = [(32, 12), (32,), (32, 32), (32,), (4, 32), (4,)]
    m, v = np.zeros_like(p), np.zeros_like(p)
    for it in range(1, steps + 2):
        w, at = [], 0
        for s in shapes:
            w.append(p[at:at + math.prod(s)].reshape(s))
            at += math.prod(s)
        h1 = np.maximum(x @ w[0].T + w[1], 0.0)
        h2 = np.maximum(h1 @ w[2].T + w[3], 0.0)
        e = h2 @ w[4].T + w[5] - t
        if it > steps:
            return p, float(np.mean(e * e))
        d = 2.0 * e / e.size
        d2 = (d @ w[4]) * (h2 > 0)
        d1 = (d2 @ w[2]) * (h1 > 0)
        g = np.concatenate([(d1.T @ x).ravel(), d1.sum(0), (d2.T @ h1).ravel(), d2.sum(0),
                            (d.T @ h2).ravel(), d.sum(0)])
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - _LR * (m / (1 - 0.9 ** it)) / (np.sqrt(v / (1 - 0.999 ** it)) + 1e-8)


def exact(case, seed):
    # every other path answers in whole numbers, which stay equal
    if case["path"] != "train":
        return None
    s = prepare(case, seed)
    p, loss = _train_exact(s["x"], s["t"], s["params"], case["steps"])
    return dict(params=p, loss=loss)
