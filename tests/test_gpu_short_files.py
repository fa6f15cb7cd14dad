"""A .cbd file that ends early: the threads that read it all leave together,
whichever of them finds the end first."""
import pytest

import albba_amd as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("keep", [0.0, 0.3, 0.999])
def test_short_files_again_and_again(ctx, tmp_path, keep):
    g = A.Graph.rmat(12, 16, seed=5, perm_seed=6)
    path = tmp_path / "g.cbd"
    g.write_cbd(str(path))
    raw = path.read_bytes()
    cols = 12 + 4 * (g.n + 1)
    path.write_bytes(raw[:cols + int(4 * g.nnz * keep)])
    for _ in range(200):
        with pytest.raises(A.AlbbaError, match="short read"):
            A.DeviceGraph.load(ctx, str(path))
    path.write_bytes(raw)
    dg = A.DeviceGraph.load(ctx, str(path))
    assert dg.bfs(int(g.pick_roots(1, 1)[0]))["reached"] > 1
    dg.close()
