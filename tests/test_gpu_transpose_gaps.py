"""The transpose of a loaded file (W = A^T) where one block's entries lie on
both sides of a run of empty rows: equal to the host's around the run length
at which the rows are searched instead of walked, and in about the time of the
same entries without the run."""
import numpy as np
import pytest

import albba_amd as A

pytestmark = pytest.mark.gpu
SPAN = 8 * 2048  # rows of a block's entries beyond which they are searched


def _graph(n, rows, seed):
    rng = np.random.default_rng(seed)
    cols = rng.integers(0, n, rows.size)
    order = np.lexsort((cols, rows))
    rp = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(rows, minlength=n), out=rp[1:])
    return rp, cols[order].astype(np.int32)


# entries of the rows on either side; the run starts inside a block of 2 048
@pytest.mark.parametrize("counts", [(1, 1), (777, 1271), (2047, 5000), (5000, 3)])
@pytest.mark.parametrize("run", [SPAN - 1, SPAN, SPAN + 1, 3 * SPAN + 17])
def test_runs(ctx, tmp_path, run, counts):
    # rows 0 and `run` hold most entries, a few rows behind them the rest
    n = run + 40
    rng = np.random.default_rng(run)
    rows = np.concatenate([np.zeros(counts[0], np.int64), np.full(counts[1], run), rng.integers(run, n, 100)])
    rp, cols = _graph(n, np.sort(rows), 1)
    path = str(tmp_path / "a.cbd")
    A.Graph.from_arrays(rp, cols).write_cbd(path)
    tp, tc = A.convert_csr_to_csc(n, rp.astype(np.int32), cols)
    want = A.Graph.from_arrays(tp.astype(np.int64), tc, symmetric=False).sellcs(64, 4096, 1).arrays()
    dg = A.DeviceGraph.load(ctx, path, 64, 4096, 1)
    dev = dg.layout().arrays()
    for k, v in want.items():
        np.testing.assert_array_equal(dev[k], v, err_msg=k)
    dg.close()


def test_a_long_run_costs_no_more_than_its_rows(ctx, tmp_path):
    """2^24 rows, 2^21 entries, once spread evenly and once on either side of
    one run: the transposes read the same bytes, so that the run may cost a few
    times the even one but not a walk of the whole run by one block (49 times)."""
    n, m = 1 << 24, 1 << 21
    rng = np.random.default_rng(2)
    ms = {}
    for name, rows in (("even", rng.integers(0, n, m)),
                       ("run", np.concatenate([rng.integers(0, 1000, m // 2 + 777), rng.integers(n - 1000, n, m // 2)]))):
        rp, cols = _graph(n, np.sort(rows), 3)
        path = str(tmp_path / (name + ".cbd"))
        A.Graph.from_arrays(rp, cols).write_cbd(path)
        t = []
        for _ in range(4):
            dg = A.DeviceGraph.load(ctx, path, 64, 4096, 1)
            t.append(dg.build_report["prep_ms"])
            dg.close()
        ms[name] = min(t)
    assert ms["run"] <= 6 * ms["even"], ms
