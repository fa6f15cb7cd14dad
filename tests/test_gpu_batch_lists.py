"""The batched BFS where its push lists, its turns between push and pull and
its barrier's tags change: levels wider than a list (1 024 edges), than a
window (2 048) and than a reservation (2 048 vertices), sources around the
listed degree (32), a graph that turns to pull and back twice, more barriers
than a tag counts (65 536), and teams of 1 to 64 workgroups.  Levels and
parents equal the oracle's exactly."""
import os

import numpy as np
import pytest

import albba_amd as A
from oracle import oracle as O

pytestmark = pytest.mark.gpu
SELECTOR = os.path.join(os.path.dirname(A.__file__), "selector.txt")


def csr(edges, n, seed):
    perm = np.random.default_rng(seed).permutation(n)
    e = perm[np.asarray(edges, np.int64)]
    e = np.unique(np.concatenate([e, e[:, ::-1]]), axis=0)
    rp = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(e[:, 0], minlength=n), out=rp[1:])
    return rp, e[:, 1].astype(np.int32), int(perm[0])


def beads(blobs, path, seed):
    """Random blobs of the given sizes in a row, joined by paths: the search
    pulls inside a blob and pushes along a path."""
    rng = np.random.default_rng(seed)
    edges, n, last = [], 1, 0
    for size in blobs:
        ids = np.arange(n, n + path)
        edges += list(zip(np.concatenate([[last], ids[:-1]]), ids))
        n += path
        ids = np.arange(n, n + size)
        edges += [(n - 1, n)] + list(zip(rng.integers(n, n + size, 6 * size), rng.integers(n, n + size, 6 * size)))
        edges += list(zip(ids[:-1], ids[1:]))
        n += size
        last = n - 1
    return csr([(a, b) for a, b in edges if a != b], n, seed)


def stars(degrees):
    edges, n = [], len(degrees)
    for i, d in enumerate(degrees):
        if i + 1 < len(degrees):
            edges.append((i, i + 1))
        edges += [(i, n + j) for j in range(d)]
        n += d
    return csr(edges, n, 5)


def tree(depth):
    m = 2 ** depth - 1
    return csr([(i, 2 * i + 1) for i in range(m)] + [(i, 2 * i + 2) for i in range(m)], 2 * m + 1, 6)


GRAPHS = {"beads": lambda: beads([900, 12000, 700, 30000], 60, 1), "stars": lambda: stars([30, 31, 32, 33, 2100, 1, 0] * 9),
          "tree": lambda: tree(14), "dense": lambda: beads([3000], 3, 2)}


@pytest.mark.parametrize("workgroups", [1, 2, 7, 64])
@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_lists_and_turns(ctx, name, workgroups):
    rp, col, root = GRAPHS[name]()
    dg = A.DeviceGraph.build(ctx, A.Graph.from_arrays(rp, col, symmetric=True), 64, 1024, 1)
    b = A.Batch(ctx, [dg])
    lv, pa = O.bfs_queue(rp, col, root)
    sel = A.Selector(ctx)
    sel.load(SELECTOR)
    for policy in (A.SWITCH_HEURISTIC, A.SWITCH_LEARNED):
        for mapping in (A.MAP_LANE_ROW, A.MAP_WAVE_ROW):
            for _ in range(2):  # the second run finds the keys at rest
                o = b.run([root], policy=policy, selector=sel, mapping=mapping, workgroups=workgroups)
                level, parent = b.results(0)
                np.testing.assert_array_equal(level, lv)
                np.testing.assert_array_equal(parent, pa)
                assert o["num_levels"][0] == lv.max() + 1 == o["push_levels"][0] + o["pull_levels"][0]
                assert o["reached"][0] == (lv >= 0).sum()
                assert o["edges_in_component"][0] == np.diff(rp)[lv >= 0].sum()
        if name == "beads" and policy == A.SWITCH_HEURISTIC:
            assert o["pull_levels"][0] >= 2
    for x in (sel, b, dg):
        x.close()


@pytest.mark.parametrize("workgroups", [1, 3])
def test_more_barriers_than_a_tag_counts(ctx, workgroups):
    n = 70_000
    rp, col, root = csr([(i, i + 1) for i in range(n - 1)], n, 8)
    dg = A.DeviceGraph.build(ctx, A.Graph.from_arrays(rp, col, symmetric=True), 64, 4096, 1)
    b = A.Batch(ctx, [dg])
    o = b.run([root], workgroups=workgroups)
    lv, pa = O.bfs_queue(rp, col, root)
    level, parent = b.results(0)
    np.testing.assert_array_equal(level, lv)
    np.testing.assert_array_equal(parent, pa)
    assert o["num_levels"][0] == n
    b.close()
    dg.close()
