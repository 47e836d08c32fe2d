"""GPU test of the training kernels' matrix tiles at their edges: rows around
the 32-row tile, the 32-step K stage and the 256-row split of the weight
gradients, against the FP64 oracle to the tolerances of the forward and
gradient tests (1e-4 of the output scale, of each block and of the largest
gradient)."""
import numpy as np
import pytest

from haseongpu_amd import _native
from oracle import mlp as M
from tests.test_gpu_proposal import _random_net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 31, 32, 33, 255, 257, 289, 16384 + 5])
def test_rows_around_the_tiles(n):
    rng = np.random.default_rng(n)
    p = _random_net(6, 0.8)
    x = rng.normal(size=(n, 10)).astype(np.float32)
    t = rng.normal(size=n).astype(np.float32)
    y = _native.mlp_forward(p, x)
    ref = M.forward(p.astype(np.float64), x.astype(np.float64))
    np.testing.assert_allclose(y, ref, rtol=1e-4, atol=1e-4 * np.abs(ref).max())
    w = np.ones(n, np.float32)
    _, g = _native.mlp_loss_gradient(p, x, t, w)
    _, gref = M.loss_gradient(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64), w.astype(np.float64))
    gb, rb = M.unpack(g.astype(np.float64)), M.unpack(gref)
    for name in M.NAMES:
        assert np.linalg.norm(gb[name] - rb[name]) <= 1e-4 * np.linalg.norm(rb[name]) + 1e-9, name
    assert np.max(np.abs(g - gref)) <= 1e-4 * np.abs(gref).max()
