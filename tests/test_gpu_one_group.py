"""A small graph's BFS runs in one workgroup: levels and parents equal the
oracle's, and the statistics equal those of the level loop (which runs when
levels are timed), over the sizes where the kernel's arrays, row classes and
key fields end."""
import os

import numpy as np
import pytest

import albba_amd as A
from oracle import oracle as O

pytestmark = pytest.mark.gpu
SELECTOR = os.path.join(os.path.dirname(os.path.abspath(A.__file__)), "selector.txt")


def _csr(n, e, symmetric, seed):
    e = np.asarray(e, np.int64).reshape(-1, 2)
    e = np.random.default_rng(seed).permutation(n)[e]
    if symmetric:
        e = np.concatenate([e, e[:, ::-1]])
    e = np.unique(e, axis=0)
    rp = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(e[:, 0], minlength=n), out=rp[1:])
    return rp, e[:, 1].astype(np.int32), symmetric


def _random(n, m, symmetric, seed):
    e = np.random.default_rng(seed).integers(0, n, (m, 2))
    return _csr(n, e[e[:, 0] != e[:, 1]], symmetric, seed)


def _path(n):
    return _csr(n, np.stack([np.arange(n - 1), np.arange(1, n)], 1), True, n)


def _star(n, tail):
    """A hub with leaves at the end of a tail."""
    e = [(i, i + 1) for i in range(tail)] + [(tail, i) for i in range(tail + 1, n)]
    return _csr(n, e, True, n)


def _complete(n):
    return _csr(n, np.stack(np.triu_indices(n, 1), 1), True, n)


def _two_cliques(k, joint):
    """Two cliques of k joined by a path of `joint` vertices."""
    a = np.stack(np.triu_indices(k, 1), 1)
    p = np.arange(k - 1, k + joint + 1)
    return _csr(2 * k + joint, np.concatenate([a, a + k + joint, np.stack([p[:-1], p[1:]], 1)]), True, k)


def _grid(r, c):
    v = np.arange(r * c).reshape(r, c)
    e = np.concatenate([np.stack([v[:, :-1].ravel(), v[:, 1:].ravel()], 1),
                        np.stack([v[:-1].ravel(), v[1:].ravel()], 1)])
    return _csr(r * c, e, True, r * c)


CASES = {
    "one": lambda: _csr(1, [], True, 1),
    "isolated": lambda: _csr(64, [(0, 1)], True, 2),
    "pair": lambda: _csr(2, [(0, 1)], True, 3),
    "r63": lambda: _random(63, 300, True, 4),
    "r65_directed": lambda: _random(65, 300, False, 5),
    "r1023": lambda: _random(1023, 9000, True, 6),
    "r1025_directed": lambda: _random(1025, 20000, False, 7),
    "r8192": lambda: _random(8192, 100000, True, 8),
    "r8193": lambda: _random(8193, 100000, True, 9),  # one past: the level loop
    "sparse8192": lambda: _random(8192, 9000, True, 10),
    "path8192": lambda: _path(8192),
    "path4500": lambda: _path(4500),
    "star8192": lambda: _star(8192, 9),
    "complete512": lambda: _complete(512),  # rows past a lane's part, 261 632 entries
    "complete520": lambda: _complete(520),  # past the entries: the level loop
    "cliques": lambda: _two_cliques(200, 12),
    "grid": lambda: _grid(90, 91),
}


@pytest.mark.parametrize("name", list(CASES))
def test_small_graph(ctx, name):
    rp, col, symmetric = CASES[name]()
    g = A.Graph.from_arrays(rp, col, symmetric=symmetric)
    sel = A.Selector(ctx)
    sel.load(SELECTOR)
    rng = np.random.default_rng(len(name))
    for C_, sigma in ((64, 4096), (16, 64), (128, 256), (32, 32)):
        dg = A.DeviceGraph.build(ctx, g, C_, sigma, 1)
        for root in {0, g.n - 1, int(rng.integers(g.n))}:
            lv, pa = O.bfs_queue(rp, col, root)
            for kw in (dict(policy=A.SWITCH_HEURISTIC), dict(policy=A.SWITCH_LEARNED, selector=sel),
                       dict(policy=A.SWITCH_HEURISTIC, small_frontier_edges=0),
                       dict(policy=A.SWITCH_LEARNED, selector=sel, small_frontier_edges=100)):
                o = dg.bfs(root, **kw)
                np.testing.assert_array_equal(o["level"], lv)
                np.testing.assert_array_equal(o["parent"], pa)
                assert O.validate(rp, col, root, o["level"], o["parent"]) == 0
                w = dg.bfs(root, time_levels=True, results=False, **kw)
                for k in ("num_levels", "reached", "edges_in_component"):
                    assert o[k] == w[k], k
                for k in ("frontier", "choice", "features", "choice_ms"):
                    np.testing.assert_array_equal(o[k], w[k], err_msg=k)
                push = o["choice"] == A.CHOICE_PUSH
                for k in ("entries", "words", "bypassed", "col_bypassed"):
                    np.testing.assert_array_equal(o[k][push], w[k][push], err_msg=k)
                np.testing.assert_array_equal((o["bypassed"] + o["words"])[~push], (w["bypassed"] + w["words"])[~push])
                assert (o["col_bypassed"] <= o["entries"]).all()
                assert (o["col_bypassed"][o["choice"] != A.CHOICE_PULL_CB] == 0).all()
        roots = rng.integers(0, g.n, 5).astype(np.int32)
        m = dg.bfs_many(roots)
        for i, r in enumerate(roots):
            lv, pa = O.bfs_queue(rp, col, int(r))
            assert m["num_levels"][i] == lv.max() + 1 and m["reached"][i] == (lv >= 0).sum()
        level, parent = dg.results()
        np.testing.assert_array_equal(level, lv)
        np.testing.assert_array_equal(parent, pa)
        dg.close()
