"""The importance map's path replay (column_path, path_ray_* of
importance_walk.h) compiled for the host: each entry equals the whole column
walk's bit for bit, with the same count of prisms visited - importance and
transfer factors, without and with reflections (orders 0-2, total internal
reflection), cladding, one layer and many, and a path storage too short for
the longer paths (those are reported full and take the column walk)."""
import ctypes as C
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

from haseongpu_amd.workloads import plain_small, production_disk
from tests.test_walk_host import _f32_exact, _records

HERE = Path(__file__).resolve().parent / "walk_host"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
pytestmark = pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc is needed to build the host walk")
U32, F32, U64 = C.c_uint32, C.c_float, C.c_ulonglong


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = tmp_path_factory.mktemp("path") / "column_path_host.so"
    subprocess.run([HIPCC, "-O2", "-fPIC", "-shared", "--cuda-host-only", "-x", "hip",
                    str(HERE / "column_path_host.cpp"), "-o", str(out)], check=True, capture_output=True)
    return C.CDLL(str(out))


CASES = {
    "slab": (lambda: plain_small(), 1, None),
    "one_layer": (lambda: production_disk(levels=2, n_points=120, wavelengths=1), 3, None),
    "disk_2_orders": (lambda: production_disk(levels=6, n_points=300, wavelengths=5), 5, [1.83, 1.0, 1.83, 1.0]),
    "deep_disk": (lambda: production_disk(levels=24, n_points=150, wavelengths=3), 3, [1.0, 1.0, 1.0, 1.0]),
}


@pytest.mark.parametrize("transfer", [0, 1])
@pytest.mark.parametrize("cap", [4096, 12])
@pytest.mark.parametrize("name", list(CASES))
def test_replay_equals_the_column_walks(lib, name, cap, transfer):
    make, R, nidx = CASES[name]
    w = _f32_exact(make())
    topo, med = w.topology, w.medium
    T, L, Np = topo.numberOfTriangles, int(topo.levels), topo.numberOfPoints
    rec, _, beta = _records(w)
    h = float(topo.thickness)
    bv = np.maximum(med.value("betaVolume"), 0.0).astype(np.float32) * np.float32(1e-3)
    sa, se, _, _ = w.spectra.spectralPairs(False)
    nt = float(med.value("nTot"))
    c1, c2 = (nt * (np.asarray(se) + sa) * 1.4427).astype(np.float32), (nt * np.asarray(sa) * 1.4427).astype(np.float32)
    refl = np.ascontiguousarray(med.value("reflectivities"), np.float32) if R > 1 else None
    ni = None if nidx is None else np.array(nidx, np.float32)
    pts = topo.points.astype(np.float32)
    ptr = lambda a, t: None if a is None else np.ascontiguousarray(a).ctypes.data_as(C.POINTER(t))   # noqa: E731
    fulls = 0
    for s in np.random.default_rng(2).integers(0, w.samples, 6):
        p, lv = int(s) % Np, int(s) // Np
        replay, columns = np.full(R * T * (L - 1), -1.0, np.float32), np.zeros(R * T * (L - 1), np.float32)
        n1, n2, full = U64(0), U64(0), U32(0)
        assert 0 == lib.column_path_host(U32(T), U32(L - 1), F32(h), ptr(rec, U32), ptr(pts, F32), U32(Np), ptr(beta, F32), ptr(bv, F32), ptr(refl, F32),
                             ptr(ni, F32), F32(float(med.value("claddingAbsorption"))), ptr(c1, F32), ptr(c2, F32),
                             U32(len(c1)), F32(pts[p, 0]), F32(pts[p, 1]), C.c_int(lv), U32(R), C.c_int(transfer),
                             U32(cap), ptr(replay, F32), ptr(columns, F32), C.byref(n1), C.byref(n2), C.byref(full))
        fulls += full.value
        done = replay >= 0.0
        assert int((~done).sum()) == full.value * R * (L - 1)
        assert np.array_equal(replay[done], columns[done])
        if full.value == 0:
            assert n1.value == n2.value and done.all()
    assert (fulls == 0) if cap == 4096 else (fulls > 0)
