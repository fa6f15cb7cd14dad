"""run_custom_bfs_test builds its layout on the device, or on the host where
the row pointers do not run from 0 to nnz: frontier sizes over the forms that
a caller's CSR may take equal the oracle's."""
import numpy as np
import pytest

import albba_amd as A
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _csr(n, m, seed, order):
    rng = np.random.default_rng(seed)
    rows, cols = rng.integers(0, n, m), rng.integers(0, n, m)
    k = np.lexsort((cols, rows)) if order == "ascending" else np.argsort(rows, kind="stable")
    rp = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(rows, minlength=n), out=rp[1:])
    return rp, cols[k].astype(np.int32)


@pytest.mark.parametrize("sort_flag", [False, True])
@pytest.mark.parametrize("order", ["ascending", "as drawn"])
@pytest.mark.parametrize("n,m,spare", [(1, 0, 0), (1, 3, 0), (63, 200, 0), (1000, 3000, 0), (20011, 130000, 0),
                                       (1000, 3000, 7), (20011, 130000, 1)])
def test_frontiers_over_matrix_forms(n, m, spare, order, sort_flag):
    """Directed, with duplicates and self loops; `spare` entries past the last
    row (the matrix's nnz is larger than its last row pointer)."""
    rp, col = _csr(n, m, n + m, order)
    out = A.run_custom_bfs_test(n, rp, np.concatenate([col, np.zeros(spare, np.int32)]), sort_flag=sort_flag)
    # the oracle wants ascending rows
    row = np.repeat(np.arange(n), np.diff(rp))
    lv, _ = O.bfs_queue(rp.astype(np.int64), col[np.lexsort((col, row))], 0)
    reached = np.bincount(lv[lv >= 0])
    np.testing.assert_array_equal(out["frontier"], reached)
    assert out["num_vex"] == reached.sum()
