"""Batches of small graphs, whose found lists hold no more reservations than
their largest team makes: graphs at the sizes where that team grows (4 096
positions a workgroup), from a few instances to more than workgroups, under
the split by shares and the one by the first run's times.  Levels and parents
equal the oracle's exactly."""
import numpy as np
import pytest

import albba_amd as A
from oracle import oracle as O

pytestmark = pytest.mark.gpu

GRAPHS = [("grid", dict(rows=3, cols=1365)), ("grid", dict(rows=64, cols=64)), ("grid", dict(rows=91, cols=90)),
          ("er", dict(n=8193, mean_degree=6.0)), ("rmat", dict(scale=10, edgefactor=8)),
          ("rmat", dict(scale=15, edgefactor=4)), ("grid", dict(rows=2, cols=3))]


@pytest.mark.parametrize("count", [1, 2, 40, 1200])
def test_small_graphs(ctx, count):
    made = []
    for k, (kind, p) in enumerate(GRAPHS[:count]):
        dg, g = A.DeviceGraph.generate(ctx, kind, 64, 1024, 1, seed=30 + k, perm_seed=60 + k,
                                       **(dict(p, p_remove=0.02) if kind == "grid" else p))
        root = int(g.pick_roots(1, 5 + k, largest_cc=True)[0])
        made.append((dg, root, O.bfs_queue(g.row_ptr, g.col, root)))
    pick = [made[i % len(made)] for i in range(count)]
    b = A.Batch(ctx, [m[0] for m in pick])
    for _ in range(3):  # by shares, then by the times of the first run
        o = b.run([m[1] for m in pick])
        teams = {int(t): int(s) for t, s in zip(o["team"], o["team_size"])}
        assert min(teams.values()) >= 1 and max(teams.values()) <= 64
        for i in sorted({0, count // 2, count - 1, *range(min(count, 2 * len(GRAPHS)))}):
            level, parent = b.results(i)
            np.testing.assert_array_equal(level, pick[i][2][0])
            np.testing.assert_array_equal(parent, pick[i][2][1])
        np.testing.assert_array_equal(o["reached"], [(m[2][0] >= 0).sum() for m in pick])
    b.close()
    for m in made:
        m[0].close()
