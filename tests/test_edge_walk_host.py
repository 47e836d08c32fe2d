"""The walk over edge records (walk_edges of prism_walk.h, packed by
edge_records.h) compiled for the host: the same results, bit for bit, and the
same prism counts as the walk over the 48-byte records, in the global format
and each of the three staged ones - with and without cladding, reflections
(orders 0-2, total internal reflection), one layer and many, rays that start
at a vertex or end above the start; and the format chosen by mesh size."""
import ctypes as C
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

from haseongpu_amd.workloads import plain_small, production_disk
from oracle import oracle as O
from tests.test_walk_host import _case, _f32_exact, _rays, _records

HERE = Path(__file__).resolve().parent / "walk_host"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
pytestmark = pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc is needed to build the host walk")
U32, F32 = C.c_uint32, C.c_float
KINDS = {"global": 0, "edges": 4, "indexed": 5, "twins": 6}


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = tmp_path_factory.mktemp("edges") / "edge_walk_host.so"
    subprocess.run([HIPCC, "-O2", "-fPIC", "-shared", "--cuda-host-only", "-x", "hip",
                    str(HERE / "edge_walk_host.cpp"), "-o", str(out)], check=True, capture_output=True)
    return C.CDLL(str(out))


def _walks(lib, w, kind, starts, prisms, ends, nr, fp):
    topo, med = w.topology, w.medium
    T, L, Np = topo.numberOfTriangles, int(topo.levels), topo.numberOfPoints
    rec, _, beta = _records(w)
    h = float(topo.thickness)
    n = len(prisms)
    a, e = np.float32(starts), np.float32(ends)
    a[:, 2] = np.float32(starts[:, 2] / h)
    e[:, 2] = np.rint(ends[:, 2] / h)          # end points lie on level planes
    hold = []

    def ptr(v, kind_of, dtype):
        hold.append(np.ascontiguousarray(v, dtype))
        return hold[-1].ctypes.data_as(C.POINTER(kind_of))

    outs = [(np.zeros((n, 5), np.float32), np.zeros(n, np.uint32), np.zeros(n, np.int32)) for _ in range(2)]
    at = [(o.ctypes.data_as(C.POINTER(F32)), s.ctypes.data_as(C.POINTER(U32)), t.ctypes.data_as(C.POINTER(C.c_int32)))
          for o, s, t in outs]
    lib.edge_walk_host(U32(T), U32(L - 1), F32(h), ptr(rec, U32, np.uint32), ptr(topo.points, F32, np.float32), U32(Np),
                       U32(KINDS[kind]), ptr(beta, F32, np.float32), ptr(med.value("reflectivities"), F32, np.float32),
                       ptr(med.value("refractiveIndices"), F32, np.float32), U32(n), ptr(a, F32, np.float32),
                       ptr(prisms, U32, np.uint32), ptr(e, F32, np.float32), ptr(nr, U32, np.uint32),
                       ptr(fp, U32, np.uint32), *at[0], *at[1])
    return outs


MESHES = {
    "plain_small": lambda: (plain_small(), 0),
    "true_cladding": lambda: _case("true_cladding"),
    "disk_reflect": lambda: _case("disk_reflect"),
    "one_layer": lambda: (production_disk(levels=2, n_points=120, wavelengths=1), 2),
}


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("name", list(MESHES))
def test_edge_walk_equals_the_record_walk(lib, name, kind):
    w, orders = MESHES[name]()
    w = _f32_exact(w)
    om = O.OracleMesh(w.topology, w.medium)
    starts, prisms, ends, nr, fp = _rays(w, om, 2000, seed=8, reflections=orders)
    topo = w.topology
    tri = topo.trianglePointIndices[prisms % topo.numberOfTriangles]
    starts[:200, :2] = np.float32(topo.points[tri[:200, 1]])     # from a vertex of the start triangle
    ends[100:300, :2] = starts[100:300, :2]                      # straight up or down
    edge, ref = _walks(lib, w, kind, starts, prisms, ends, nr, fp)
    for got, want in zip(edge, ref):
        assert np.array_equal(got, want)
    assert orders == 0 or (nr > 0).any()


@pytest.mark.parametrize("T,points,kind", [
    (2, 4, 4), (4522, 2300, 4), (4523, 2300, 5), (7904, 2567, 5), (7905, 2567, 6), (7400, 3700, 5), (10100, 5050, 6),
    (10200, 5052, 6), (10200, 5053, 0), (10922, 3969, 6), (10922, 100, 6), (10923, 100, 0), (4000, 65536, 4),
    (4000, 65537, 0), (9000, 6852, 6), (9000, 6853, 0)])
def test_format_by_mesh_size(lib, T, points, kind):
    """The widest format whose arrays fit in 10,176 16-byte words (162,816 B):
    36 B a triangle, else 18 B a triangle and 8 B a point, else 12 and 8;
    record numbers stay below 0x7FFF and point numbers within 16 bits."""
    assert lib.edge_kind_host(U32(T), U32(points)) == kind


@pytest.mark.parametrize("d", [1, 2, 3, 5, 90, 4023, 65536, 2**24 - 1, 76_437, 2**31 - 1, 2**31, 2**32 - 1])
def test_division_by_a_mesh_count(lib, d):
    near = {x for k in (0, 1, 2, 7, (2**32 - 1) // d) for x in (k * d - 1, k * d, k * d + 1)} | {2**32 - 1, 2**31}
    for n in (n for n in near if 0 <= n < 2**32):
        assert C.c_uint32(lib.fast_div_host(U32(d), U32(n))).value == n // d
