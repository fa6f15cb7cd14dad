"""The queue and its degree prefix that a push level's finalize lists for the
next push, and the queue listed from a bitmap after a pull: every edge of the
frontier is expanded once (the reported entries are the frontier's out-edges),
and levels and parents equal the oracle's, at sizes around the words that a
wave and a block take and the bounds between them."""
import numpy as np
import pytest

import albba_amd as A
from oracle import oracle as O

pytestmark = pytest.mark.gpu

P, SB = A.CHOICE_PUSH, A.CHOICE_PULL_SB
SCRIPTS = [[P] * 64, [P, SB] * 32, [P, P, SB, SB] * 16, [SB, P, P, P] * 16]


def _check(dg, rp, col, root, **kw):
    lv, pa = O.bfs_queue(rp, col, root)
    o = dg.bfs(root, **kw)
    np.testing.assert_array_equal(o["level"], lv)
    np.testing.assert_array_equal(o["parent"], pa)
    deg = np.diff(rp)
    push = np.flatnonzero(o["choice"] == P)
    want = np.bincount(lv[lv >= 0], weights=deg[lv >= 0], minlength=o["num_levels"])
    np.testing.assert_array_equal(o["entries"][push], want[push])


@pytest.mark.parametrize("n,degree", [(40, 3.0), (4096, 5.0), (4097, 40.0), (16384 - 63, 8.0), (70001, 12.0),
                                      ((1 << 20) - 64, 4.0), ((1 << 20) + 1, 7.0), ((1 << 23) + 65, 2.5)])
def test_scripted_pushes_and_pulls(ctx, n, degree):
    dg, g = A.DeviceGraph.generate(ctx, "er", 64, 4096, 1, n=n, mean_degree=degree, seed=n, perm_seed=n + 1)
    rp, col = g.row_ptr.copy(), g.col.copy()
    root = int(g.pick_roots(1, 9, largest_cc=True)[0])
    for s in SCRIPTS if n < 1 << 22 else SCRIPTS[:2]:
        _check(dg, rp, col, root, policy=A.SWITCH_SCRIPT, script=s)
    for pol in (A.SWITCH_HEURISTIC, A.SWITCH_BEST) if n < 1 << 22 else (A.SWITCH_HEURISTIC,):
        _check(dg, rp, col, root, policy=pol)
    _check(dg, rp, col, root, policy=A.SWITCH_FIXED, fixed_choice=P)
    dg.close()


@pytest.mark.parametrize("leaves", [1, 63, 8191, 8192, 8193, 70000])
def test_wide_level_after_a_narrow_one(ctx, leaves):
    """A hub's leaves, each with a tail of its own: a frontier of any width is
    pushed by the kernels queued ahead."""
    n = 2 + 2 * leaves
    a = np.arange(2, 2 + leaves)
    e = np.concatenate([[[0, 1]], np.stack([np.ones(leaves, np.int64), a], 1), np.stack([a, a + leaves], 1)])
    e = np.concatenate([e, e[:, ::-1]])
    e = e[np.lexsort((e[:, 1], e[:, 0]))]
    rp = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(e[:, 0], minlength=n), out=rp[1:])
    col = e[:, 1].astype(np.int32)
    dg = A.DeviceGraph.build(ctx, A.Graph.from_arrays(rp, col, symmetric=True), 64, 4096, 1)
    for root in (0, 1, n - 1):
        for s in (SCRIPTS[0], SCRIPTS[1]):
            _check(dg, rp, col, root, policy=A.SWITCH_SCRIPT, script=s)
        _check(dg, rp, col, root, policy=A.SWITCH_HEURISTIC)
    dg.close()
