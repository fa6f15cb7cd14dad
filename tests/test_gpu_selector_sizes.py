"""The selector's gradient where its passes' splits change: one sample, the
ends of a 64-sample chunk, and the ends of the 256-chunk tile of the sums
(16 384 samples), against the float64 restatement; and a training step's
update against Adam on that gradient."""
import numpy as np
import pytest

import albba_amd as A
from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu

# float32 sums of n terms against float64: n * 2^-24 relative to the sum of
# magnitudes, n <= 64 + 257 terms in the two passes and 32 in a layer (2.1e-5),
# with a factor of ten for layers on layers
TOL = 2e-4


def samples(ns, seed):
    rng = np.random.default_rng(seed)
    return rng.random((ns, 12), dtype=np.float32), rng.normal(size=(ns, 4)).astype(np.float32)


@pytest.mark.parametrize("ns", [1, 63, 64, 65, 127, 129, 16383, 16384, 16385, 33000])
def test_gradient_at_chunk_and_tile_ends(ctx, ns):
    x, t = samples(ns, ns)
    s = A.Selector(ctx, seed=5)
    loss, g = s.loss_grad(x, t)
    rl, rg = M.loss_grad(s.params, x, t)
    assert abs(loss - rl) <= TOL * rl
    assert np.linalg.norm(g - rg) <= TOL * np.linalg.norm(rg)
    s.close()


def test_one_step_is_adam_on_the_gradient(ctx):
    x, t = samples(1000, 3)
    s = A.Selector(ctx, seed=6)
    p0 = s.params.astype(np.float64)
    _, g = s.loss_grad(x, t)
    s.train(x, t, steps=1, lr=1e-2)
    g = g.astype(np.float64)
    # first step: the moments' bias corrections cancel
    want = p0 - 1e-2 * g / (np.abs(g) + 1e-8)
    # every term is rounded to float32 a handful of times
    np.testing.assert_allclose(s.params, want, rtol=1e-5, atol=1e-7)
    s.close()
