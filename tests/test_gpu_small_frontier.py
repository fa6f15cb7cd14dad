"""The small-frontier kernel at the sizes where its lists and reservations
change: sources of 31 to 33 out-edges (a listed vertex has at most 32), of
more out-edges than a workgroup's list holds (1 024), levels of more found
vertices than one reservation (1 024), runs of more levels than one launch
takes (4 096), and the learned policy's own rule for entering it.  Levels and
parents equal the oracle's exactly."""
import os

import numpy as np
import pytest

import albba_amd as A
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def symmetric(edges, n):
    e = np.asarray(edges, np.int64).reshape(-1, 2)
    e = np.unique(np.concatenate([e, e[:, ::-1]]), axis=0)
    rp = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(e[:, 0], minlength=n), out=rp[1:])
    return rp, e[:, 1].astype(np.int32)


def caterpillar(legs):
    """A path whose spine vertex i carries legs[i] leaves; ids shuffled."""
    edges, nxt = [], len(legs)
    for i, k in enumerate(legs):
        if i + 1 < len(legs):
            edges.append((i, i + 1))
        edges += [(i, nxt + j) for j in range(k)]
        nxt += k
    perm = np.random.default_rng(7).permutation(nxt)
    return symmetric(perm[np.array(edges)], nxt), nxt, int(perm[0])


def run(ctx, rp, col, root, policy=A.SWITCH_HEURISTIC, blocks=0, **kw):
    g = A.Graph.from_arrays(rp, col, symmetric=True)
    dg = A.DeviceGraph.build(ctx, g, 64, 4096, 1)
    lv, pa = O.bfs_queue(rp, col, root)
    for _ in range(2):  # the second BFS finds the keys at rest
        o = dg.bfs(root, policy=policy, small_frontier_blocks=blocks, capacity=1 << 14, **kw)
        np.testing.assert_array_equal(o["level"], lv)
        np.testing.assert_array_equal(o["parent"], pa)
        # (per-level statistics hold as many levels as the caller's arrays)
        np.testing.assert_array_equal(o["frontier"], np.bincount(lv[lv >= 0])[:1 << 14])
        assert o["edges_in_component"] == int(np.diff(rp)[lv >= 0].sum())
    dg.close()
    return o


@pytest.mark.parametrize("blocks", [0, 1, 5])
@pytest.mark.parametrize("legs", [[0] * 6 + [29, 30, 31, 32, 33] * 8, [3] * 40 + [1030, 1, 0, 2100] + [2] * 400,
                                  [0] * 5000, [1] * 2047 + [30] * 300])
def test_listed_and_shared_vertices(ctx, legs, blocks):
    (rp, col), n, root = caterpillar(legs)
    # leaves around the spine keep the frontier under 0.04 n only on graphs
    # with more vertices: pad with a far part that one long edge row reaches
    far = np.arange(n, n + 64 * 1024)
    spine = np.stack([far[:-1], far[1:]], 1)
    rows = np.repeat(np.arange(n), np.diff(rp))
    edges = np.concatenate([np.stack([rows, col], 1), spine])
    rp, col = symmetric(edges, n + far.size)
    run(ctx, rp, col, root, blocks=blocks)


@pytest.mark.parametrize("blocks", [1, 2, 64])
def test_wide_levels(ctx, blocks):
    """A tree whose levels grow to 8 192 vertices, in front of a long path:
    with one workgroup every list and reservation overflows."""
    depth = 13
    edges = [(i, 2 * i + 1) for i in range(2 ** depth - 1)] + [(i, 2 * i + 2) for i in range(2 ** depth - 1)]
    n0 = 2 ** (depth + 1) - 1
    n = n0 + 250_000
    edges += [(i, i + 1) for i in range(n0, n - 1)] + [(n0 - 1, n0)]
    rp, col = symmetric(np.random.default_rng(3).permutation(n)[np.array(edges)], n)
    root = int(np.random.default_rng(3).permutation(n)[0])
    run(ctx, rp, col, root, blocks=blocks)


def test_learned_policy_enters_on_slow_levels(ctx):
    sel = A.Selector(ctx)
    sel.load(os.path.join(os.path.dirname(A.__file__), "selector.txt"))
    g = A.Graph.grid(300, 211, 0.1, seed=9, perm_seed=10)
    root = int(g.pick_roots(1, 4, largest_cc=True)[0])
    o = run(ctx, g.row_ptr.copy(), g.col.copy(), root, policy=A.SWITCH_LEARNED, selector=sel)
    # whatever the network ranks first, the long run of small levels is pushed
    assert (o["choice"] == A.CHOICE_PUSH).sum() > 0.9 * o["num_levels"]
    off = run(ctx, g.row_ptr.copy(), g.col.copy(), root, policy=A.SWITCH_LEARNED, selector=sel,
              small_frontier_edges=0)
    assert off["num_levels"] == o["num_levels"]
    sel.close()
