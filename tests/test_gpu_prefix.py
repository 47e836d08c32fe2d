"""GPU test of the proposal's prefix and buckets (mixture_prefix) at the sizes
where its rows and runs end: fewer triangles than a row holds, one more row
than full ones, fewer rows than wavefronts, one layer, and each work-group
size.  On identical streams the estimate follows the CPU oracle's own FP64
prefix: a ray moves to a neighbouring entry only where its target lies within
the FP32 error of the importance (2e-5 in the median, as in the estimator
tests), and one ray of N moves a sample by about 1 / N, so every sample is
held to 8 / N."""
import numpy as np
import pytest

from haseongpu_amd.workloads import production_disk
from oracle import oracle as O
from tests.test_gpu_parity import _context, _oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("points,levels,orders,rays,rows", [
    (4, 2, 0, 8192, 1),          # 7 triangles, one layer: one row; all cladding, so nothing emits
    (12, 2, 0, 8192, 1),         # 21 triangles, one layer
    (20, 3, 0, 8192, 2),         # 37 triangles
    (20, 10, 1, 8192, 27),       # 37 triangles, more rows than 16 wavefronts
    (38, 3, 1, 8192, 12),        # 70 triangles: a full row and six entries
    (38, 20, 0, 2048, 38),       # 760 samples: 256 threads
    (60, 28, 2, 512, 270),       # 1680 samples of 270 rows: 512 threads
])
def test_estimate_from_the_prefix_of_small_and_ragged_meshes(points, levels, orders, rays, rows):
    w = production_disk(levels=levels, n_points=points, wavelengths=2)
    T = w.topology.numberOfTriangles
    assert (1 + 2 * orders) * (levels - 1) * ((T + 63) // 64) == rows
    kw = dict(use_reflections=orders > 0, max_reflections=max(1, orders))
    ctx, spectra = _context(w, min_rays=rays, rng_seed=3, **kw)
    om, op = _oracle(w, spectra, min_rays=rays, seed=3, **kw)
    with ctx:
        res = ctx.evaluate()
    ref = O.calc_phi_ase(om, op)
    assert np.array_equal(res.totalRays, ref["totalRays"]) and res.droppedRays.sum() == 0
    lit = ref["phiAse"] > 0.0
    assert np.all(res.phiAse[~lit] == 0.0) and (lit.all() or points == 4)
    if points == 4:
        return
    rel = np.abs(res.phiAse.astype(np.float64) / ref["phiAse"] - 1.0)
    assert np.median(rel) <= 2e-5 and rel.max() <= 8.0 / rays, np.sort(rel)[-5:]
