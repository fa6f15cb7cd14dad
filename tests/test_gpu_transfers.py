"""Copies to and from ordinary memory at the sizes where their path changes
(one stage a piece below 3 MB an array, several threads and stages above it;
pieces of 256 KB to 4 MB), a .cbd that cannot seek, and device memory used
again by graphs of other sizes."""
import os
import threading

import numpy as np
import pytest

import albba_amd as A
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65535, 65537, 786431, 786432, 786433, 1048577, 4194303, 4194305])
def test_results_and_upload(ctx, n):
    # a path over permuted ids, cut short: most vertices are unreached
    perm = np.random.default_rng(n).permutation(n).astype(np.int64)
    a, b = perm[:700], perm[1:701]
    rows, cols = np.concatenate([a, b]), np.concatenate([b, a])
    at = np.lexsort((cols, rows))
    rp = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(rows, minlength=n), out=rp[1:])
    col = cols[at].astype(np.int32)
    dg = A.DeviceGraph.build(ctx, A.Graph.from_arrays(rp, col, symmetric=True), 64, 4096, 1)
    o = dg.bfs(int(perm[0]))
    lv, pa = O.bfs_queue(rp, col, int(perm[0]))
    np.testing.assert_array_equal(o["level"], lv)
    np.testing.assert_array_equal(o["parent"], pa)
    dg.close()


def test_load_from_a_pipe_equals_the_file(ctx, tmp_path):
    g = A.Graph.rmat(15, 16, seed=31, perm_seed=32)
    path, fifo = str(tmp_path / "g.cbd"), str(tmp_path / "p.cbd")
    g.write_cbd(path)
    os.mkfifo(fifo)
    data = open(path, "rb").read()

    def feed():
        try:
            with open(fifo, "wb") as f:
                f.write(data)
        except BrokenPipeError:
            pass  # the values at the file's end are not read

    t = threading.Thread(target=feed)
    t.start()
    dp = A.DeviceGraph.load(ctx, fifo, 64, 4096, 1)
    t.join()
    df = A.DeviceGraph.load(ctx, path, 64, 4096, 1)
    x, y = dp.layout().arrays(), df.layout().arrays()
    for k in x:
        if x[k] is not None:
            np.testing.assert_array_equal(x[k], y[k])
    dp.close()
    df.close()


def test_memory_used_again_by_other_graphs(ctx):
    """Graphs of changing sizes built, searched and closed in turn get each
    other's blocks; every search equals the oracle's."""
    for k, scale in enumerate((14, 16, 13, 16, 15, 14, 17, 12)):
        g = A.Graph.rmat(scale, 8 + k, seed=60 + k, perm_seed=70 + k)
        rp, col = g.row_ptr.copy(), g.col.copy()
        dg = A.DeviceGraph.build(ctx, g, 64, 1024, 1)
        for root in g.pick_roots(2, k):
            o = dg.bfs(int(root))
            lv, pa = O.bfs_queue(rp, col, int(root))
            np.testing.assert_array_equal(o["level"], lv)
            np.testing.assert_array_equal(o["parent"], pa)
        dg.close()
