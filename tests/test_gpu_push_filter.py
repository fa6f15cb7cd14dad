"""The push expansion's filter and its search for a wave's first row: many
edges into one target (the parent is still the smallest id, whichever edge
comes first), queues around the search's 64 probes, and rows that span
chunks.  Levels and parents equal the oracle's exactly."""
import numpy as np
import pytest

import albba_amd as A
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mids,leaves", [(1, 70), (2, 64), (63, 3), (64, 200), (65, 129), (127, 64), (128, 1),
                                         (700, 90), (4097, 3), (9000, 2)])
def test_every_target_hit_by_every_row(ctx, mids, leaves):
    """root -> mids -> leaves, complete between the two: mids edges into every
    leaf, from a queue of mids rows."""
    n = 1 + mids + leaves
    perm = np.random.default_rng(mids + leaves).permutation(n)
    m = np.arange(1, 1 + mids)
    e = np.concatenate([np.stack([np.zeros(mids, np.int64), m], 1),
                        np.stack([np.repeat(m, leaves), np.tile(np.arange(1 + mids, n), mids)], 1)])
    e = perm[e]
    e = np.concatenate([e, e[:, ::-1]])
    e = e[np.lexsort((e[:, 1], e[:, 0]))]
    rp = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(e[:, 0], minlength=n), out=rp[1:])
    col = e[:, 1].astype(np.int32)
    dg = A.DeviceGraph.build(ctx, A.Graph.from_arrays(rp, col, symmetric=True), 64, 4096, 1)
    root = int(perm[0])
    lv, pa = O.bfs_queue(rp, col, root)
    for _ in range(2):
        o = dg.bfs(root, policy=A.SWITCH_FIXED, fixed_choice=A.CHOICE_PUSH)
        np.testing.assert_array_equal(o["level"], lv)
        np.testing.assert_array_equal(o["parent"], pa)
        np.testing.assert_array_equal(o["entries"], [mids, mids * (leaves + 1), mids * leaves])
    dg.close()
