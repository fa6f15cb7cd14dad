"""The transpose of the device build (the push rows of a directed graph) and
of the file loader (W = A^T): equal to the host's, over entry counts around a
block's chunk, hub rows that span chunks, runs of empty rows longer than a
chunk, and a column that holds everything."""
import numpy as np
import pytest

import albba_amd as A

pytestmark = pytest.mark.gpu


def _rows(name):
    rng = np.random.default_rng(len(name))
    if name.startswith("uniform"):
        m = int(name[7:])
        n = 1 + m // 3
        return n, rng.integers(0, n, m)
    if name == "hubs":  # neighbours in id and in position
        n = 9000
        return n, np.concatenate([np.repeat(np.arange(7), 8000), rng.integers(0, n, 20000)])
    if name == "empty_runs":
        n = 40000
        return n, np.repeat([0, 1, 12000, 12001, 39998], [3, 2050, 1, 5000, 9])
    if name == "one_row":
        return 5000, np.full(4999, 4321)
    assert name == "large"
    n = 300000
    return n, (rng.random(2500000) ** 3 * n).astype(np.int64)


@pytest.mark.parametrize("name", ["uniform1", "uniform2047", "uniform2048", "uniform2049", "uniform4097",
                                  "uniform70000", "hubs", "empty_runs", "one_row", "large"])
def test_transpose(ctx, tmp_path, name):
    n, rows = _rows(name)
    rng = np.random.default_rng(3)
    cols = rng.integers(0, n, rows.size)
    if name == "uniform4097":
        cols[:] = 17
    order = np.lexsort((cols, rows))
    rows, cols = rows[order], cols[order].astype(np.int32)
    rp = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(rows, minlength=n), out=rp[1:])
    g = A.Graph.from_arrays(rp, cols, symmetric=False)
    for C_, sigma in ((64, 4096), (32, 64)):
        host = g.sellcs(C_, sigma, 1).arrays()
        dg = A.DeviceGraph.build(ctx, g, C_, sigma, 1)
        dev = dg.layout().arrays()
        for k, v in host.items():
            np.testing.assert_array_equal(dev[k], v, err_msg=k)
        dg.close()
    # from a file: the layout of the transpose
    path = str(tmp_path / "a.cbd")
    g.write_cbd(path)
    tp, tc = A.convert_csr_to_csc(n, rp.astype(np.int32), cols)
    want = A.Graph.from_arrays(tp.astype(np.int64), tc, symmetric=False).sellcs(64, 4096, 1).arrays()
    dg = A.DeviceGraph.load(ctx, path, 64, 4096, 1)
    dev = dg.layout().arrays()
    for k, v in want.items():
        np.testing.assert_array_equal(dev[k], v, err_msg=k)
    dg.close()
