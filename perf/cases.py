"""Performance cases of the library: what a program that uses it has it do.

Every case goes through the entry points such a program calls (``PhiASE.run``,
a resident ``Context``, ``Batch``, ``Simulation``, ``ForwardContext``, the
network training and the transfer maps it is trained on).  The sizes are those
of the repository's own workloads: the plain slab, the production disk, the
batching configuration's disks (200-8000 triangles, 5-40 levels), the combined
configuration's large mesh (128 wavelengths, records beyond LDS), the
time-stepped loop and the tetrahedral forward estimator.

``exact`` restates each of them in 64-bit torch (walks by edge intersections
and layer sums, the same counter-based random streams), without the library.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from haseongpu_amd import (FrozenPhiAseRungeKutta4, GainMedium, Grid, LocalPump, MeshTopology, PhiASE, Simulation,
                           _native)
from haseongpu_amd.proposal import LearnedProposal
from haseongpu_amd.tet_mesh import TetMesh
from haseongpu_amd.workloads import disk_points, gaussian_spectra

N_TOT, TAU = 2.76e20, 9.5e-4
CLADDING_ALPHA = 5.5
FIELDS = ("phiAse", "mse", "totalRays", "dndtAse", "standardError", "droppedRays")
WHOLE = ("totalRays", "droppedRays")


# ------------------------------------------------------------------- the cases

def _estimate(name, mesh, points, levels, wavelengths, *, samples, min_rays, reflections=0, cladding=False,
              proposal="walked", entry="resident"):
    c = {"kind": "estimate", "mesh": mesh, "points": points, "levels": levels, "wavelengths": wavelengths,
         "samples": samples, "min_rays": min_rays, "reflections": reflections, "cladding": cladding,
         "proposal": proposal, "entry": entry}
    return c if name is None else {"name": name, **c}


def listed():
    return [
        # one front-end call on the plain slab, one level of sample points, few rays: context set-up, launches and
        # latency (a parameter scan or an interactive session calls it like this)
        _estimate("slab-run", "slab", 10, 10, 1, samples=121, min_rays=4096, entry="run"),
        # the plain slab at its full ray count on a resident context whose beta is refreshed before each evaluation
        # (a user's own time loop)
        _estimate("slab-resident", "slab", 10, 10, 1, samples=1210, min_rays=100_000),
        # a share of the production disk's sample points with the walked importance map: reflections, cladding, 64
        # wavelengths, adaptive rays (the plain form of the headline workload)
        _estimate("disk-walked", "disk", 2060, 20, 64, samples=3000, min_rays=100_000, reflections=1, cladding=True),
        # the same disk with the learned proposal (the headline form)
        _estimate("disk-learned", "disk", 2060, 20, 64, samples=5000, min_rays=100_000, reflections=1, cladding=True,
                  proposal="learned"),
        # one of the batching configuration's larger disks (beyond 4800 triangles, no reflections), walked
        _estimate("wide-disk-walked", "disk", 3301, 27, 9, samples=3000, min_rays=10_000),
        # and with the learned proposal
        _estimate("wide-disk-learned", "disk", 3301, 27, 9, samples=6000, min_rays=10_000, proposal="learned"),
        # a share of a mesh beyond both LDS record formats with the combined configuration's options (30 levels, 128
        # wavelengths, reflections, cladding), learned proposal
        _estimate("large-learned", "disk", 5000, 30, 128, samples=700, min_rays=100_000, reflections=1, cladding=True,
                  proposal="learned"),
        # many small independent problems in one batch (shared work queue)
        {"name": "batch-small", "kind": "batch", "problems": 32, "points": 150, "levels": 8, "wavelengths": 8,
         "min_rays": 10_000},
        # one step of the time-stepped loop (frozen-flux Runge-Kutta 4, local pump) on a small disk
        {"name": "time-step", "kind": "loop", "points": 300, "levels": 10, "wavelengths": 16, "min_rays": 10_000,
         "reflections": 1},
        # the forward estimator on a disk of tetrahedra with cladding, beta refreshed before the evaluation
        {"name": "forward", "kind": "forward", "points": 2060, "levels": 20, "wavelengths": 64, "rays": 4_000_000},
        # training of the proposal network: AdamW steps over one batch of rows
        {"name": "train", "kind": "train", "rows": 16_384, "epochs": 12},
        # transfer maps, the rows the network is trained on, for a run of sample points
        {"name": "transfer-map", "kind": "transfer", "points": 2060, "levels": 20, "wavelengths": 64, "samples": 16,
         "reflections": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# estimated work (walked proposal entries x path length + traced rays x path length) a drawn estimate may take
_WORK_CAP = 4.5e10


def draw(rng):
    kind = rng.choice(["slab", "disk", "disk", "disk", "disk", "batch", "loop", "forward", "train", "transfer"])
    if kind == "slab":
        n, levels = rng.randint(5, 16), rng.randint(4, 14)
        entry = rng.choice(["run", "resident"])
        total = (n + 1) ** 2 * levels
        return _estimate(None, "slab", n, levels, 1, samples=rng.randint(max(1, total // 12), total),
                         min_rays=_log(rng, 1000, 60_000), entry=entry)
    if kind == "disk":
        points, levels = _log(rng, 120, 4700), rng.randint(5, 32)
        proposal = rng.choice(["walked", "learned"])
        reflections = rng.choice([0, 1])
        min_rays = _log(rng, 8000, 100_000)
        path = 1.1 * math.sqrt(2 * points)
        entries = (1 + 2 * reflections) * 2 * points * (levels - 1) if proposal == "walked" else 0
        most = int(_WORK_CAP / (path * (entries + min_rays)))
        total = points * levels
        hi = max(320, min(total - 1, most, 6000))
        return _estimate(None, "disk", points, levels, _log(rng, 1, 128), samples=_log(rng, 300, hi),
                         min_rays=min_rays, reflections=reflections, cladding=bool(rng.getrandbits(1)),
                         proposal=proposal, entry="resident")
    if kind == "batch":
        return {"kind": "batch", "problems": rng.randint(6, 32), "points": rng.randint(90, 200),
                "levels": rng.randint(5, 10), "wavelengths": rng.randint(1, 16), "min_rays": _log(rng, 3000, 10_000)}
    if kind == "loop":
        return {"kind": "loop", "points": _log(rng, 120, 300), "levels": rng.randint(5, 10),
                "wavelengths": rng.randint(1, 16), "min_rays": _log(rng, 2000, 10_000),
                "reflections": rng.choice([0, 1])}
    if kind == "forward":
        return {"kind": "forward", "points": _log(rng, 200, 2060), "levels": rng.randint(4, 20),
                "wavelengths": rng.randint(1, 64), "rays": _log(rng, 200_000, 4_000_000)}
    if kind == "train":
        return {"kind": "train", "rows": _log(rng, 1500, 16_384), "epochs": rng.randint(4, 12)}
    return {"kind": "transfer", "points": _log(rng, 200, 2060), "levels": rng.randint(5, 20),
            "wavelengths": rng.randint(1, 64), "samples": rng.randint(2, 16), "reflections": rng.choice([0, 1])}


# ------------------------------------------------------------------- inputs

@functools.lru_cache(maxsize=64)
def _topology(mesh, points, levels, mesh_seed=0):
    """Meshes depend on the case alone (a program keeps its mesh); beta, reflectivities and streams on the seed."""
    if mesh == "slab":
        return MeshTopology.fromGrid(Grid(x=1.0, y=1.0, z=0.7, tileSizeX=1.0 / points, tileSizeZ=0.7 / (levels - 1)))
    radius = 3.0 * math.sqrt(max(points, 500) / 2060.0)
    return MeshTopology.fromPoints(disk_points(radius, points, 2 + mesh_seed), numberOfLevels=levels,
                                   thickness=0.7 / (levels - 1))


def _beta(topo, rng, clad):
    """A pumped spot with noise per prism, no inversion in the cladding ring; a random field on the slab."""
    if topo.metadata.get("source") == "grid":
        return rng.uniform(0.0, 0.3, size=topo.numberOfPrisms)
    cent = topo.prismCentroids()
    extent = float(np.hypot(topo.points[:, 0], topo.points[:, 1]).max())
    cx, cy = rng.uniform(-0.15, 0.15, size=2) * extent
    r2 = (cent[:, 0] - cx) ** 2 + (cent[:, 1] - cy) ** 2
    width = 0.4 * extent
    beta = rng.uniform(0.25, 0.32) * np.exp(-r2 / (2 * width * width)) + rng.normal(0.0, 0.01, size=r2.size)
    beta = np.clip(beta, 0.0, 1.0)
    beta[np.tile(clad, int(topo.levels) - 1)] = 0.0
    return beta


class _Problem:
    """Mesh, medium, spectra and run controls of an estimate, as numpy arrays and front-end objects."""

    def __init__(self, c, seed, mesh_seed=0):
        self.topo = topo = _topology(c.get("mesh", "disk"), c["points"], c["levels"], mesh_seed)
        rng = np.random.default_rng([seed, mesh_seed])
        slab = c.get("mesh") == "slab"
        clad = np.zeros(topo.numberOfTriangles, bool) if not c.get("cladding", not slab) else topo.boundaryTriangles()
        self.clad = clad
        self.beta = _beta(topo, rng, clad)
        self.refl = rng.uniform(0.0, 0.1, size=2 * topo.numberOfTriangles).astype(np.float32)
        pr2 = (topo.points ** 2).sum(axis=1)
        self.beta_cells = np.tile(0.3 * np.exp(-pr2 / (0.32 * pr2.max())), int(topo.levels))
        self.alpha = CLADDING_ALPHA if clad.any() else 0.0
        self.K = int(c.get("reflections", 0))
        self.medium = GainMedium(topo).withPhysicalProperties(
            betaVolume=self.beta, betaCells=self.beta_cells, claddingCellTypes=clad.astype(np.uint32),
            claddingNumber=1, claddingAbsorption=self.alpha, nTot=N_TOT, crystalTFluo=TAU, reflectivities=self.refl,
            refractiveIndices=[1.0, 1.0, 1.0, 1.0])
        self.spectra = gaussian_spectra(c["wavelengths"])
        self.sa, self.se, self.msa, self.mse = self.spectra.spectralPairs(False)
        S = topo.numberOfSamples
        # a share starts inside the range, as the shares of several processes do
        n = min(int(c.get("samples", S)), S)
        self.first = 0 if n == S or c.get("entry") == "run" else (S - n) // 3
        self.last = self.first + n - 1
        self.min_rays, self.max_rays, self.steps = c["min_rays"], c["min_rays"] * 100, 4
        self.seed = int(seed) & 0x7FFFFFFF
        self.threshold, self.eps = 0.005, 0.05

    def phi_ase(self, **more):
        return PhiASE(crossSections=self.spectra, minRaysPerSample=self.min_rays, maxRaysPerSample=self.max_rays,
                      mseThreshold=self.threshold, adaptiveSteps=self.steps, useReflections=self.K > 0,
                      maxReflections=max(1, self.K), rngSeed=self.seed, minSampleRange=self.first,
                      maxSampleRange=self.last, defensiveFraction=self.eps, **more)

    def context(self):
        return _native.Context(*self.phi_ase().nativeArguments(self.medium, self.spectra))


def _inputs_of(sx, sy, sz, cx, cy, level, beta, h, log_sigma):
    cz = (level + 0.5) * h
    dist = np.sqrt((sx - cx) ** 2 + (sy - cy) ** 2 + (sz - cz) ** 2)
    return np.stack([sx, sy, sz, cx, cy, cz, level, beta, dist, np.full(sx.shape, log_sigma)], axis=-1)


def _rows(problem, n, rng):
    """(inputs, log transfer) rows like those of the transfer maps: positions in the mesh, gain over the distance,
    weak mirror images."""
    topo, h = problem.topo, float(problem.topo.thickness)
    layers = int(topo.levels) - 1
    pts = topo.points
    s, t = rng.integers(0, len(pts), n), rng.integers(0, topo.numberOfTriangles, n)
    l = rng.integers(0, layers, n)
    plane = rng.integers(0, layers + 1, n) + (rng.integers(-1, 2, n) * layers if problem.K else 0)
    cent = pts[topo.trianglePointIndices].mean(axis=1)[t]
    beta = problem.beta[t + l * topo.numberOfTriangles]
    X = _inputs_of(pts[s, 0], pts[s, 1], plane * h, cent[:, 0], cent[:, 1], l.astype(float), beta, h,
                   math.log(problem.mse / problem.msa))
    mirrored = (plane < 0) | (plane > layers)
    Y = 0.25 * X[:, 8] * (0.3 + 2.0 * beta) - 3.0 * mirrored + rng.normal(0.0, 0.2, n)
    return X, Y


def _initial_params(rng):
    parts = []
    for shape in ((128, 10), (128, 128), (128, 128), (128, 128), (1, 128)):
        lim = math.sqrt(6.0 / shape[1])
        parts += [rng.uniform(-lim, lim, shape).reshape(-1), np.zeros(shape[0])]
    return np.concatenate(parts).astype(np.float32)


_SHAPES = ((128, 10), (128, 128), (128, 128), (128, 128), (1, 128))


def _split_params(p):
    out, at = [], 0
    for o, i in _SHAPES:
        out.append((p[at:at + o * i].reshape(o, i), p[at + o * i:at + o * i + o]))
        at += o * i + o
    return out


def _network(problem):
    """A network for the problem's mesh: random hidden layers, the output layer fitted to transfer rows (rounded, so
    that it is the same for everybody)."""
    rng = np.random.default_rng(11)
    X, Y = _rows(problem, 6000, rng)
    shift, scale = X.mean(axis=0), 1.0 / np.maximum(X.std(axis=0), 1e-3)
    params = _initial_params(rng)
    a = (X - shift) * scale
    layers = _split_params(params.astype(np.float64))
    for w, b in layers[:4]:
        z = a @ w.T + b
        a = z / (1.0 + np.exp(-z))
    A = np.column_stack([a, np.ones(len(a))])
    w5 = np.linalg.solve(A.T @ A + 2.0 * np.eye(129), A.T @ Y)
    params[-129:] = np.round(w5 * 1024.0) / 1024.0
    T, lay = problem.topo.numberOfTriangles, int(problem.topo.levels) - 1
    ct, cl = max(1, T // 64), max(1, -(-lay // 3))   # about 150-200 clusters per reflection slice
    return LearnedProposal(params, shift.astype(np.float32), scale.astype(np.float32), ct, cl, True)


def _tet_mesh(c, seed):
    p = _Problem({**c, "cladding": True, "min_rays": 1}, seed)
    mesh = TetMesh.fromPrisms(p.topo, p.beta, cladding_types=p.clad.astype(np.uint32), cladding_number=1,
                              cladding_absorption=CLADDING_ALPHA, n_tot=N_TOT, tau=TAU)
    return p, mesh


def prepare(case, seed):
    kind = case["kind"]
    if kind == "estimate":
        p = _Problem(case, seed)
        if case["entry"] == "run":
            return {"do": "run", "phi": p.phi_ase(), "medium": p.medium}
        ctx = p.context()
        if case["proposal"] == "learned":
            ctx.set_proposal(_network(p))
        return {"do": "resident", "ctx": ctx, "beta": p.beta, "beta_cells": p.beta_cells}
    if kind == "batch":
        ctxs = [_Problem({**case, "cladding": False}, seed, i).context() for i in range(case["problems"])]
        return {"do": "batch", "ctxs": ctxs, "batch": _native.Batch(ctxs)}
    if kind == "loop":
        p = _Problem(case, seed)
        rate = _pump_rate(p.topo)
        sim = Simulation(gain_medium=p.medium, phi_ase=p.phi_ase(ase_steps=1 << 30),
                         time_integrator=FrozenPhiAseRungeKutta4(), time_step_size=2e-5, cross_sections=p.spectra)
        sim.add_pump(LocalPump(rate=rate, saturation=1.21 * rate, pump_steps=1 << 30))
        return {"do": "loop", "sim": sim}
    if kind == "forward":
        p, mesh = _tet_mesh(case, seed)
        exp = _native.NativeExperiment(sigma_a=p.sa, sigma_e=p.se, min_rays=case["rays"], max_rays=case["rays"])
        comp = _native.make_compute(n_samples=1, adaptive_steps=0, rng_seed=p.seed)
        return {"do": "forward", "ctx": _native.ForwardContext(mesh, exp, comp), "beta": mesh.beta}
    if kind == "train":
        X, Y, params = _training_set(case, seed)
        return {"do": "train", "X": X, "Y": Y, "params": params, "epochs": case["epochs"]}
    p = _Problem({**case, "cladding": True, "min_rays": 1000}, seed)
    return {"do": "transfer", "ctx": p.context(), "beta": p.beta, "first": p.first, "count": p.last - p.first + 1}


def _pump_rate(topo):
    cent = topo.prismCentroids()
    return 1500.0 * np.exp(-(cent[:, 0] ** 2 + cent[:, 1] ** 2) / 2.88) * np.exp(-1.5 * cent[:, 2])


def _training_set(case, seed):
    rng = np.random.default_rng(seed)
    p = _Problem({"points": 300, "levels": 10, "wavelengths": 1, "min_rays": 1, "reflections": 1}, seed)
    X, Y = _rows(p, case["rows"], rng)
    Xn = ((X - X.mean(axis=0)) / np.maximum(X.std(axis=0), 1e-3)).astype(np.float32)
    return Xn, Y.astype(np.float32), _initial_params(rng)


def _result(r):
    return {name: getattr(r, name) for name in FIELDS}


def run(state):
    do = state["do"]
    if do == "run":
        return _result(state["phi"].run(state["medium"]))
    if do == "resident":
        state["ctx"].update_beta(state["beta"], state["beta_cells"])
        return _result(state["ctx"].evaluate())
    if do == "batch":
        results = state["batch"].evaluate()
        return {name: np.concatenate([getattr(r, name) for r in results]) for name in FIELDS}
    if do == "loop":
        st = state["sim"].step(1).getLastState()
        return {"betaVolume": st.betaVolume, "phiAse": st.phiAse, "dndtAse": st.dndtAse, "dndtPump": st.dndtPump,
                "phiSamples": st.aseResult.phiAse, "mse": st.aseResult.mse, "totalRays": st.aseResult.totalRays,
                "standardError": st.aseResult.standardError}
    if do == "forward":
        state["ctx"].update_beta(state["beta"])
        r = state["ctx"].evaluate()
        return {name: getattr(r, name) for name in ("phiAse", "standardError", "relativeStandardError", "dndtAse",
                                                    "rayVisits", "droppedRays", "convergenceRays")}
    if do == "train":
        params, history = _native.mlp_train(state["params"], state["X"], state["Y"], epochs=state["epochs"],
                                            batch=state["X"].shape[0], learning_rate=2e-3, weight_decay=1e-5)
        return {"params": params, "history": history}
    state["ctx"].update_beta(state["beta"])
    return state["ctx"].transfer_map(state["first"], state["count"])


def work(case):
    """What a pass cannot do without.  A walked entry or a ray is one path: its triangle crossings (2 side products,
    a crossing parameter and the beta sum, ~24 operations each) and the gain of every wavelength (5 each); bytes are
    the mesh and beta read and the results written."""
    kind = case["kind"]
    if kind == "train":
        n, per = case["rows"], 2 * (10 * 128 + 3 * 128 * 128 + 128)
        return {"bytes": n * 44.0 + 8 * 51_073.0, "flops": 3.0 * per * n * case["epochs"]}
    slab = case.get("mesh") == "slab"
    Np = (case["points"] + 1) ** 2 if slab else case["points"]
    T = 2 * case["points"] ** 2 if slab else 2 * case["points"]
    layers = case["levels"] - 1
    P, W = T * layers, case["wavelengths"]
    crossings = 0.55 * math.sqrt(T)
    if kind == "forward":
        segments = case["rays"] * 2.2 * layers
        return {"bytes": 3 * P * (16.0 + 9.0 + 36.0) + Np * case["levels"] * 24.0, "flops": 120.0 * segments}
    R = 1 + 2 * case.get("reflections", 0)
    mesh_bytes = T * 24.0 + Np * 16.0 + P * 8.0
    walk = crossings * 24.0 + 5.0 * W
    if kind == "transfer":
        n = case["samples"] * R * P
        return {"bytes": mesh_bytes + 4.0 * n, "flops": n * walk}
    samples = case.get("samples", Np * case["levels"]) * case.get("problems", 1)
    # a ray aimed by the proposal crosses about a quarter of a uniform path's triangles
    flops = samples * case["min_rays"] * (0.25 * crossings * 24.0 + 12.0 * R + 5.0 * W + 60.0)
    flops += samples * R * P * (walk if case.get("proposal", "walked") == "walked" else 12.0)
    return {"bytes": case.get("problems", 1) * mesh_bytes + 36.0 * samples, "flops": flops}


# ------------------------------------------------------------------- the same in 64 bits

_M32 = 0xFFFFFFFF


def _philox(c0, c1, c2, c3, k0, k1):
    """Philox4x32-10 on int64 tensors (or numbers) holding 32-bit words."""
    for _ in range(10):
        p0, p1 = 0xD2511F53 * c0, 0xCD9E8D57 * c2
        c0, c1, c2, c3 = (((p1 >> 32) & _M32) ^ c1 ^ k0), p1 & _M32, (((p0 >> 32) & _M32) ^ c3 ^ k1), p0 & _M32
        k0, k1 = (k0 + 0x9E3779B9) & _M32, (k1 + 0xBB67AE85) & _M32
    return c0, c1, c2, c3


def _unit(x):
    return (((x >> 9) << 1) | 1).to(torch.float64) * 2.0 ** -24


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _hilbert(x, y):
    d = np.zeros_like(x)
    s = 1 << 15
    while s:
        rx, ry = ((x & s) > 0).astype(np.int64), ((y & s) > 0).astype(np.int64)
        d += s * s * ((3 * rx) ^ ry)
        flip = (ry == 0) & (rx == 1)
        x, y = np.where(flip, 65535 - x, x), np.where(flip, 65535 - y, y)
        x, y = np.where(ry == 0, y, x), np.where(ry == 0, x, y)
        s >>= 1
    return d


class _Geometry:
    """Mesh and beta of a problem in 64 bits, triangles in the order the proposal runs over (Hilbert order of their
    centroids)."""

    def __init__(self, p):
        dev = _device()
        topo = p.topo
        tri = np.asarray(topo.trianglePointIndices, np.int64)
        pts = topo.points
        T, self.layers, self.np_, self.h = len(tri), int(topo.levels) - 1, len(pts), float(topo.thickness)
        c = (pts[tri[:, 0]] + pts[tri[:, 1]] + pts[tri[:, 2]]) / 3.0
        lo, hi = c.min(axis=0), c.max(axis=0)
        q = np.clip(np.floor((c - lo) / np.where(hi > lo, hi - lo, 1.0) * 65535.0), 0, 65535).astype(np.int64)
        order = np.argsort(_hilbert(q[:, 0], q[:, 1]), kind="stable")
        back = np.empty(T, np.int64)
        back[order] = np.arange(T)
        nb = np.asarray(topo.topology()["triangleNeighbors"], np.int64).reshape(3, T).T
        nb = np.where(nb >= 0, back[np.maximum(nb, 0)], -1)[order]
        v = pts[tri[order]]
        area = 0.5 * ((v[:, 1, 0] - v[:, 0, 0]) * (v[:, 2, 1] - v[:, 0, 1])
                      - (v[:, 1, 1] - v[:, 0, 1]) * (v[:, 2, 0] - v[:, 0, 0]))
        beta = p.beta.reshape(self.layers, T)[:, order]
        walk = np.where(p.clad[order][None, :], 0.0, beta)
        K, n = p.K, self.layers
        u = np.arange(-K * n, (K + 1) * n)
        copy, r = np.floor_divide(u, n), np.mod(u, n)
        level = np.where(copy % 2 != 0, n - 1 - r, r)
        unfolded = walk[level].T                                         # (T, planes)
        self.low, self.planes = -K * n, len(u)
        prefix = np.concatenate([np.zeros((T, 1)), np.cumsum(unfolded, axis=1)], axis=1)[:, :-1]
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)  # noqa: E731
        self.T, self.order, self.back = T, order, back
        self.v, self.nb, self.prefix, self.unfolded = t(v), t(nb), t(prefix), t(unfolded)
        self.clad = t(p.clad[order].astype(np.float64))
        self.refl = t(p.refl.reshape(T, 2)[order].astype(np.float64))
        self.bv = t(np.maximum(beta, 0.0) * area[None, :] * self.h).reshape(-1)   # level-major
        self.cent = self.v.mean(dim=1)
        self.pts = t(pts)
        self.beta_level, self.area = beta, area
        # per wavelength: exponent = a * sum(beta l) - b * sum(l), in gain prisms
        self.wa, self.wb = t(N_TOT * (p.se + p.sa)), t(N_TOT * p.sa)
        self.alpha, self.R = p.alpha, 1 + 2 * K

    def gain(self, bl, gl, cl):
        g = torch.zeros_like(bl)
        for a, b in zip(self.wa.tolist(), self.wb.tolist()):
            g += torch.exp(a * bl - b * gl - self.alpha * cl)
        return g / len(self.wa)

    def image(self, lv, k):
        """Unfolded plane of the mirror image of level lv for reflection slice k (tensors or numbers)."""
        n = self.layers
        m = (k + 1) // 2
        top = torch.where(m % 2 == 1, m * n + (n - lv), m * n + lv)
        bottom = torch.where(m % 2 == 1, -(m - 1) * n - lv, -m * n + lv)
        return torch.where(m == 0, lv, torch.where(k % 2 == 1, top, bottom))


def _walk(g, t, ax, ay, ex, ey, za, ze, k):
    """Paths from (ax, ay) in triangle t to (ex, ey), [n]; heights za to ze with reflection slice k, [n, m] or
    broadcast.  Returns sum(beta l), sum(l) in gain and cladding prisms, surface factors and length, [n, m]."""
    n, m = ax.shape[0], torch.broadcast_shapes(za.shape, ze.shape)[-1]
    dev = ax.device
    za, ze, k = (x.expand(n, m) for x in (za, ze, k))
    dx, dy = ex - ax, ey - ay
    dz = ze - za
    D = torch.sqrt((dx * dx + dy * dy)[:, None] + (dz * g.h) ** 2)
    bsum, rf = torch.zeros(n, m, dtype=torch.float64, device=dev), torch.ones(n, m, dtype=torch.float64, device=dev)
    clad = torch.zeros(n, dtype=torch.float64, device=dev)
    ok = torch.ones(n, dtype=torch.bool, device=dev)
    nref, first = (k + 1) // 2, k % 2
    bounds = []
    for b in range(1, (g.R - 1) // 2 + 1):
        zb = torch.where(first == 1, torch.full_like(dz, b * g.layers), torch.full_like(dz, -(b - 1) * g.layers))
        sb = torch.where(nref >= b, torch.clamp((zb - za) / dz, max=1.0), torch.full_like(dz, 9.0))
        plane = first if b % 2 == 1 else 1 - first
        bounds.append((sb, plane))
    at = torch.arange(n, device=dev)
    s0 = torch.zeros(n, dtype=torch.float64, device=dev)
    f0 = torch.floor(za)
    z0 = za
    live = dict(t=t, ax=ax, ay=ay, dx=dx, dy=dy, za=za, dz=dz, s0=s0, z0=z0, at=at, b=bsum.clone(), c=clad.clone(),
                r=rf.clone())
    for i, (sb, plane) in enumerate(bounds):
        live["sb%d" % i], live["pl%d" % i] = sb, plane
    for _ in range(10_000):
        L = live
        V = g.v[L["t"]]
        best, edge = None, None
        for e in range(3):
            p, q = V[:, e], V[:, (e + 1) % 3]
            nx, ny = q[:, 1] - p[:, 1], p[:, 0] - q[:, 0]
            den = L["dx"] * nx + L["dy"] * ny
            num = (p[:, 0] - L["ax"]) * nx + (p[:, 1] - L["ay"]) * ny
            s = torch.where(den > 0, num / torch.where(den > 0, den, torch.ones_like(den)),
                            torch.full_like(den, math.inf))
            if best is None:
                best, edge = s, torch.zeros_like(L["t"])
            else:
                less = s < best
                best, edge = torch.where(less, s, best), torch.where(less, torch.full_like(edge, e), edge)
        nxt = g.nb[L["t"], edge]
        end = best >= 1.0 - 1e-11
        left = ~end & (nxt < 0)
        s1 = torch.where(end, torch.ones_like(best), torch.maximum(best, L["s0"]))
        z1 = L["za"] + s1[:, None] * L["dz"]
        lo, hi = g.low, g.low + g.planes - 1
        f0 = torch.clamp(torch.floor(L["z0"]), lo, hi)
        f1 = torch.clamp(torch.floor(z1), lo, hi)
        base = (L["t"] * g.planes)[:, None] - lo
        i0, i1 = base + f0.to(torch.int64), base + f1.to(torch.int64)
        b0, b1 = g.unfolded.view(-1)[i0], g.unfolded.view(-1)[i1]
        c = (g.prefix.view(-1)[i1] + b1 * (z1 - f1)) - (g.prefix.view(-1)[i0] + b0 * (L["z0"] - f0))
        ds = s1 - L["s0"]
        L["b"] += torch.where(f0 == f1, b0 * ds[:, None], c / torch.where(L["dz"] == 0, torch.ones_like(c), L["dz"]))
        L["c"] += g.clad[L["t"]] * ds
        for i in range(len(bounds)):
            hit = (L["sb%d" % i] > L["s0"][:, None]) & (L["sb%d" % i] <= s1[:, None])
            if bool(hit.any()):
                fac = torch.gather(g.refl[L["t"]], 1, L["pl%d" % i])
                L["r"] = torch.where(hit, L["r"] * fac, L["r"])
        done = end | left
        if bool(done.any()):
            w = L["at"][done]
            bsum[w], clad[w], rf[w] = L["b"][done], L["c"][done], L["r"][done]
            ok[w] = ~(left & ((1.0 - s1) > 1e-5))[done]
            keep = ~done
            if not bool(keep.any()):
                break
            L["s0"], L["z0"], L["t"] = s1, z1, nxt
            live = {name: x[keep] for name, x in L.items()}
        else:
            L["s0"], L["z0"], L["t"] = s1, z1, nxt
    cl = clad[:, None] * D
    return bsum * D, (1.0 - clad)[:, None] * D, cl, rf, D, ok


def _map(g, samples, transfer=False):
    """Walked importance (or transfer factors) of the samples, [samples, R, layers, T]."""
    S, n, T, R = len(samples), g.layers, g.T, g.R
    dev = g.v.device
    out = torch.empty(S, R, n, T, dtype=torch.float64, device=dev)
    k = torch.arange(R, device=dev).repeat_interleave(n)[None, :]
    za = (torch.arange(n, device=dev).repeat(R) + 0.5)[None, :].to(torch.float64)
    step = max(1, int(3e7 / (T * n * R)))
    for i in range(0, S, step):
        s = samples[i:i + step]
        lv, pt = torch.div(s, g.np_, rounding_mode="floor"), s % g.np_
        N = len(s) * T
        t = torch.arange(T, device=dev).repeat(len(s))
        e = g.pts[pt].repeat_interleave(T, dim=0)
        ze = g.image(lv.repeat_interleave(T)[:, None], k).to(torch.float64)
        bl, gl, cl, rf, D, ok = _walk(g, t, g.cent[t, 0], g.cent[t, 1], e[:, 0], e[:, 1], za, ze, k.expand(N, -1))
        v = g.gain(bl, gl, cl) * rf
        if not transfer:
            v = v / (4.0 * math.pi * D * D)
        v = torch.where(ok[:, None] & torch.isfinite(v), v, torch.zeros_like(v))
        v = v.view(len(s), T, R, n).permute(0, 2, 3, 1)
        out[i:i + step] = v if transfer else v * g.bv.view(1, 1, n, T)
    return out


def _bf16(x):
    return x.to(torch.bfloat16).to(torch.float64)


def _learned_map(g, net, samples, log_sigma):
    """The learned proposal: the network (BF16 weights and activations) once per cluster and slice, its exponential
    times beta V / (4 pi d^2) of each prism."""
    dev = g.v.device
    n, T, R = g.layers, g.T, g.R
    ct, cl = min(net.cluster_triangles, T), min(net.cluster_levels, n)
    tg, lg = np.arange(T) // ct, np.arange(n) // cl
    TG, LG = int(tg[-1]) + 1, int(lg[-1]) + 1
    a = np.bincount(tg, g.area)
    cent = g.cent.cpu().numpy()
    x, y = np.bincount(tg, g.area * cent[:, 0]) / a, np.bincount(tg, g.area * cent[:, 1]) / a
    lev = np.bincount(lg, np.arange(n)) / np.bincount(lg)
    bsum = np.zeros((LG, TG))
    np.add.at(bsum, (lg[:, None], tg[None, :]), g.beta_level * g.area[None, :])
    b = bsum / (a[None, :] * np.bincount(lg)[:, None])
    t_ = lambda v: torch.as_tensor(np.ascontiguousarray(v), dtype=torch.float64, device=dev)  # noqa: E731
    x, y, lev, b = (t_(v).reshape(-1) for v in np.broadcast_arrays(x[None, :], y[None, :], lev[:, None], b))
    weights = [(_bf16(t_(w)), t_(bias)) for w, bias in _split_params(net.params)]
    w5 = t_(_split_params(net.params)[4][0])
    shift, scale = t_(net.shift), t_(net.scale)
    k = torch.arange(R, device=dev)
    S = len(samples)
    lv, pt = torch.div(samples, g.np_, rounding_mode="floor"), samples % g.np_
    plane = g.image(lv[:, None], k[None, :]).to(torch.float64)                 # (S, R)
    shape = (S, R, len(x))
    sx, sy = g.pts[pt, 0].view(S, 1, 1).expand(shape), g.pts[pt, 1].view(S, 1, 1).expand(shape)
    sz = (plane * g.h)[:, :, None].expand(shape)
    cx, cy, lv_, be = (v.expand(shape) for v in (x, y, lev, b))
    cz = (lv_ + 0.5) * g.h
    d = torch.sqrt((sx - cx) ** 2 + (sy - cy) ** 2 + (sz - cz) ** 2)
    f = torch.stack([sx, sy, sz, cx, cy, cz, lv_, be, d, torch.full_like(d, log_sigma)], dim=-1).reshape(-1, 10)
    h = _bf16((f.float().double() - shift) * scale)
    for i, (w, bias) in enumerate(weights[:4]):
        z = h @ w.T + bias
        h = z * torch.sigmoid(z)
        if i < 3:
            h = _bf16(h)
    logit = (h @ w5.T + weights[4][1]).view(S, R, LG, TG)
    logit = torch.clamp(logit, max=80.0)[:, :, torch.as_tensor(lg, device=dev)][:, :, :, torch.as_tensor(tg, device=dev)]
    dxy = ((g.cent[None] - g.pts[pt][:, None]) ** 2).sum(dim=2)                 # (S, T)
    dz = (torch.arange(n, device=dev) + 0.5)[None, None, :] - plane[:, :, None]
    d2 = dxy[:, None, None, :] + (dz * g.h)[:, :, :, None] ** 2
    return g.bv.view(1, 1, n, T) * torch.exp(logit) / (4.0 * math.pi * d2)


def _target(p, k):
    if p.max_rays <= p.min_rays or p.steps == 0:
        return p.min_rays
    if k >= p.steps:
        return p.max_rays
    growth = (p.max_rays / p.min_rays) ** (1.0 / p.steps)
    return int(min(max(math.ceil(p.min_rays * growth ** k), p.min_rays), p.max_rays))


def _trace(g, p, sample, pre, launch, n):
    """Sums of X and X^2 and the dropped rays of one launch of n rays for one sample with proposal prefix `pre`."""
    dev = g.v.device
    r0, r1, _, _ = _philox(_M32, sample, launch, 1, p.seed, 0x48415345)
    offset = ((r0 >> 5) * 67108864.0 + (r1 >> 6)) / 9007199254740992.0
    Q = float(pre[-1])
    s1 = s2 = drop = 0
    T, P = g.T, g.T * g.layers
    for i in range(0, n, 4_000_000):
        ray = torch.arange(i, min(n, i + 4_000_000), device=dev)
        e = torch.searchsorted(pre, (ray.to(torch.float64) + offset) * (Q / n), right=True).clamp_(max=len(pre) - 1)
        q = pre[e] - torch.where(e > 0, pre[(e - 1).clamp(min=0)], torch.zeros_like(pre[e]))
        X, good = _trace_rays(g, p, torch.full_like(ray, sample), launch, Q, T, P, ray, e, q)
        s1, s2, drop = s1 + float(X.sum()), s2 + float((X * X).sum()), drop + int((~good).sum())
    return s1, s2, drop


def _trace_rays(g, p, smp, launch, Q, T, P, ray, e, q):
    k, j = torch.div(e, P, rounding_mode="floor"), e % P
    t, l = j % T, torch.div(j, T, rounding_mode="floor")
    o = _philox(ray, smp, torch.full_like(ray, launch), torch.zeros_like(ray), p.seed, 0x48415345)
    u1, u2, u3 = _unit(o[0]), _unit(o[1]), _unit(o[2])
    fold = u1 + u2 > 1.0
    u1, u2 = torch.where(fold, 1.0 - u1, u1), torch.where(fold, 1.0 - u2, u2)
    v = g.v[t]
    a = v[:, 0] + u1[:, None] * (v[:, 1] - v[:, 0]) + u2[:, None] * (v[:, 2] - v[:, 0])
    lv, pt = torch.div(smp, g.np_, rounding_mode="floor"), smp % g.np_
    end = g.pts[pt]
    ze = g.image(lv, k).to(torch.float64)[:, None]
    bl, gl, cl, rf, D, ok = _walk(g, t, a[:, 0], a[:, 1], end[:, 0], end[:, 1], (l + u3)[:, None], ze, k[:, None])
    X = (g.gain(bl, gl, cl) * rf / (4.0 * math.pi * D * D))[:, 0] * g.bv[j] * (Q / q)
    good = ok & torch.isfinite(X)
    return torch.where(good, X, torch.zeros_like(X)), good


def _chunk_trace(g, p, samples, pre, launch, n):
    """The same for several samples at once (n rays each): [samples] sums."""
    dev = g.v.device
    S = len(samples)
    r = _philox(torch.full_like(samples, _M32), samples, torch.full_like(samples, launch), torch.ones_like(samples),
                p.seed, 0x48415345)
    offset = ((r[0] >> 5).to(torch.float64) * 67108864.0 + (r[1] >> 6).to(torch.float64)) / 9007199254740992.0
    Q = pre[:, -1]
    ray = torch.arange(n, device=dev)
    target = (ray.to(torch.float64)[None, :] + offset[:, None]) * (Q / n)[:, None]
    e = torch.searchsorted(pre, target.contiguous(), right=True).clamp_(max=pre.shape[1] - 1)
    low = torch.gather(pre, 1, (e - 1).clamp(min=0))
    q = torch.gather(pre, 1, e) - torch.where(e > 0, low, torch.zeros_like(low))
    X, good = _trace_rays(g, p, samples[:, None].expand(S, n).reshape(-1), launch, Q.repeat_interleave(n), g.T,
                          g.T * g.layers, ray.repeat(S), e.view(-1), q.view(-1))
    X, good = X.view(S, n), good.view(S, n)
    return X.sum(dim=1), (X * X).sum(dim=1), (~good).sum(dim=1)


def _mse(s1, s2, n):
    return max((n * s2 / (s1 * s1) - 1.0) / n, 0.0) if s1 else math.nan


def _prefix(g, p, imp):
    imp = imp.reshape(imp.shape[0], -1)
    bv = g.bv.repeat(g.R)
    q = (1.0 - p.eps) * imp / imp.sum(dim=1, keepdim=True) + p.eps * bv / (g.R * g.bv.sum())
    return torch.cumsum(q, dim=1)


def _estimate_exact(p, net=None):
    g = _Geometry(p)
    dev = g.v.device
    S = p.topo.numberOfSamples
    phi, mse, se = np.zeros(S), np.zeros(S), np.zeros(S)
    entries = g.R * g.T * g.layers
    log_sigma = float(np.float32(math.log(p.mse / p.msa)))
    todo = list(range(p.first, p.last + 1))
    forms = ["learned", "walked"] if net is not None else ["walked"]
    for form in forms:
        missed = []
        step = max(1, min(int(3e7 / entries), int(1.2e7 / p.min_rays)))
        for i in range(0, len(todo), step):
            s = torch.as_tensor(todo[i:i + step], device=dev)
            pre = _prefix(g, p, _learned_map(g, net, s, log_sigma) if form == "learned" else _map(g, s))
            launch = 1 if form == "walked" and net is not None else 0
            n = _target(p, 0)
            s1, s2, drop = _chunk_trace(g, p, s, pre, launch, n)
            for x in range(len(s)):
                a1, a2, d, N, k, la = float(s1[x]), float(s2[x]), int(drop[x]), n, 1, launch
                while not (d == 0 and _mse(a1, a2, N) <= p.threshold):
                    if form == "learned" or N >= p.max_rays:
                        break
                    la += 1
                    more = _target(p, k) - N
                    k += 1
                    b1, b2, bd = _trace(g, p, int(s[x]), pre[x], la, more)
                    a1, a2, d, N = a1 + b1, a2 + b2, d + bd, N + more
                m = _mse(a1, a2, N)
                if form == "learned" and not (d == 0 and m <= p.threshold):
                    missed.append(int(s[x]))
                    continue
                at = int(s[x])
                phi[at], mse[at] = N_TOT / TAU * a1 / N, m
                se[at] = math.sqrt(m) * abs(phi[at])
        todo = missed
    dndt = (p.beta_cells * (p.mse + p.msa) - p.msa) * phi
    return {"phiAse": phi, "mse": mse, "totalRays": None, "dndtAse": dndt, "standardError": se, "droppedRays": None}


def _loop_exact(case, seed):
    p = _Problem(case, seed)
    r = _estimate_exact(p)
    topo = p.topo
    tri, L, Np = np.asarray(topo.trianglePointIndices, np.int64), int(topo.levels), topo.numberOfPoints
    phi = r["phiAse"].reshape(L, Np)
    flux = ((phi[:-1][:, tri] + phi[1:][:, tri]).sum(axis=2) / 6.0).reshape(-1)
    clad = np.tile(p.clad, L - 1)
    sa = float(p.sa[int(np.argmax(p.se))])
    rate, h = _pump_rate(topo), 2e-5

    def parts(b):
        pump, ase = rate - 1.21 * rate * b, (b * (p.mse + sa) - sa) * flux
        return [np.where(clad, 0.0, x) for x in (pump, ase, pump - ase - b / TAU)]

    b = p.beta
    k1 = parts(b)[2]
    k2 = parts(b + 0.5 * h * k1)[2]
    k3 = parts(b + 0.5 * h * k2)[2]
    pump, ase, k4 = parts(b + h * k3)
    b = np.clip(b + h / 6.0 * (k1 + 2 * k2 + 2 * k3 + k4), 0.0, 1.0)
    shape = lambda a: a.reshape(topo.numberOfTriangles, L - 1, order="F")   # noqa: E731
    return {"betaVolume": shape(b), "phiAse": shape(flux), "dndtAse": shape(ase), "dndtPump": shape(pump),
            "phiSamples": r["phiAse"], "mse": r["mse"], "totalRays": None, "standardError": r["standardError"]}


def _forward_exact(case, seed):
    p, mesh = _tet_mesh(case, seed)
    dev = _device()
    f64 = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=dev)   # noqa: E731
    cells_np = mesh.cells.astype(np.int64)
    n = len(cells_np)
    faces = np.stack([np.sort(np.delete(cells_np, k, axis=1), axis=1) for k in range(4)], axis=1)   # (n, 4, 3)
    key = faces.reshape(-1, 3)
    order = np.lexsort((key[:, 2], key[:, 1], key[:, 0]))
    same = (key[order[1:]] == key[order[:-1]]).all(axis=1)
    link = np.full(4 * n, -1, np.int64)
    a, b = order[:-1][same], order[1:][same]
    link[a], link[b] = b, a
    pts = mesh.points
    fa, fb, fc = (pts[faces[:, :, i]] for i in range(3))
    nrm = np.cross(fb - fa, fc - fa)
    den = (nrm * (pts[cells_np] - fa)).sum(axis=2)
    nrm = nrm / den[:, :, None]
    planes = np.concatenate([nrm, -(nrm * fa).sum(axis=2)[:, :, None]], axis=2)                     # (n, 4, 4)
    v = pts[cells_np]
    vol = np.abs(np.einsum("ij,ij->i", np.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]), v[:, 3] - v[:, 0])) / 6.0
    clad = mesh.cladding_mask()
    Np = len(pts)
    copies = cells_np + np.where(clad, Np, 0)[:, None]
    lumped = np.bincount(copies.reshape(-1), np.repeat(vol / 4.0, 4), minlength=2 * Np)
    cells, link, planes, copies_t = (torch.as_tensor(x, device=dev) for x in (cells_np, link, planes, copies))
    P3 = f64(pts)
    prefix_np = np.cumsum(mesh.beta * vol)
    prefix, total, beta, clad_t = f64(prefix_np), float(prefix_np[-1]), f64(mesh.beta), f64(clad.astype(float))
    sa, se = f64(p.sa), f64(p.se)
    rays, W = case["rays"], len(p.sa)
    scores = torch.zeros(8, 2 * Np, dtype=torch.float64, device=dev)
    tag, counts, first = 0x46574431, [], 0
    for bt in range(8):
        count = rays // 8 + (1 if bt < rays % 8 else 0)
        o = _philox(_M32, bt, 0, 2, p.seed, tag)
        shift, phase = float(((o[0] >> 9) << 1) | 1) * 2.0 ** -24, o[1] % W
        i = torch.arange(count, device=dev)
        r = i + first
        cell = torch.searchsorted(prefix, (i.to(torch.float64) + shift) / count * total, right=True).clamp_(max=n - 1)
        zero = torch.zeros_like(r)
        o = _philox(r, zero, zero, zero, p.seed, tag)
        s, t, w = _unit(o[0]), _unit(o[1]), _unit(o[2])
        f = s + t > 1.0
        s, t = torch.where(f, 1.0 - s, s), torch.where(f, 1.0 - t, t)
        f1 = t + w > 1.0
        f2 = ~f1 & (s + t + w > 1.0)
        s, t, w = (torch.where(f2, 1.0 - t - w, s), torch.where(f1, 1.0 - w, t),
                   torch.where(f1, 1.0 - s - t, torch.where(f2, s + t + w - 1.0, w)))
        w0 = 1.0 - s - t - w
        c4 = cells[cell]
        x = (w0[:, None] * P3[c4[:, 0]] + s[:, None] * P3[c4[:, 1]] + t[:, None] * P3[c4[:, 2]]
             + w[:, None] * P3[c4[:, 3]])
        u = torch.zeros(count, 3, dtype=torch.float64, device=dev)
        u[:, 2] = 1.0
        open_ = torch.ones(count, dtype=torch.bool, device=dev)
        for call in range(32):
            o = _philox(r, zero, zero + (call + 1), zero, p.seed, tag)
            for pair in range(2):
                x1, x2 = 2.0 * _unit(o[2 * pair]) - 1.0, 2.0 * _unit(o[2 * pair + 1]) - 1.0
                q = x1 * x1 + x2 * x2
                take = open_ & (q < 1.0)
                rr = torch.sqrt(torch.clamp(1.0 - q, min=0.0))
                u = torch.where(take[:, None], torch.stack([2 * x1 * rr, 2 * x2 * rr, 1 - 2 * q], dim=1), u)
                open_ = open_ & ~take
            if not bool(open_.any()):
                break
        lam = (torch.div(i * W, count, rounding_mode="floor") + phase) % W
        la, le = sa[lam], se[lam]
        gain, forbid = torch.ones_like(la), torch.full_like(cell, -1)
        for _ in range(10_000):
            pl = planes[cell]
            c = (pl[:, :, :3] * x[:, None, :]).sum(dim=2) + pl[:, :, 3]
            d = (pl[:, :, :3] * u[:, None, :]).sum(dim=2)
            use = (d < 0) & (torch.arange(4, device=dev)[None, :] != forbid[:, None])
            lens = torch.where(use, -c / torch.where(use, d, torch.ones_like(d)), torch.full_like(c, math.inf))
            lens = torch.where(lens > 0, lens, torch.full_like(c, math.inf))
            length, face = lens.min(dim=1)
            good = torch.isfinite(length)
            length = torch.where(good, length, torch.zeros_like(length))
            gl = torch.where(clad_t[cell] > 0, torch.full_like(length, -CLADDING_ALPHA),
                             N_TOT * (beta[cell] * (le + la) - la))
            em1 = torch.expm1(gl * length)
            contribution = gain * torch.where(gl * length == 0, length, em1 / gl)
            wt = torch.clamp(c + 0.5 * length[:, None] * d, min=0.0)
            wt = wt / wt.sum(dim=1, keepdim=True)
            scores[bt].index_add_(0, copies_t[cell].view(-1), (contribution[:, None] * wt).view(-1))
            gain = gain * (1.0 + em1)
            x = x + u * length[:, None]
            nxt = link[cell * 4 + face]
            keep = good & (nxt >= 0)
            if not bool(keep.any()):
                break
            x, u, gain, la, le, nxt = x[keep], u[keep], gain[keep], la[keep], le[keep], nxt[keep]
            cell, forbid = torch.div(nxt, 4, rounding_mode="floor"), nxt % 4
        counts.append(count)
        first += count
    scores = scores.cpu().numpy()
    dens = np.where(lumped > 0, scores / np.where(lumped > 0, lumped, 1.0), 0.0)[:, copies].mean(axis=2) * vol   # (8, n)
    est = dens.sum(axis=0) * total / (rays * vol)
    mean = dens / np.asarray(counts)[:, None]
    m = mean.mean(axis=0)
    var = np.maximum(0.0, (mean ** 2).sum(axis=0) - mean.sum(axis=0) ** 2 / 8.0) / 7.0
    with np.errstate(divide="ignore", invalid="ignore"):
        rse = np.sqrt(var / 8.0) / np.abs(m)
    phi = est * N_TOT / TAU
    dndt = (mesh.beta * (p.se.max() + p.sa.max()) - p.sa.max()) * phi
    return {"phiAse": phi, "standardError": np.where(m == 0, 0.0, rse * np.abs(phi)),
            "relativeStandardError": np.where(m == 0, np.nan, rse), "dndtAse": dndt, "rayVisits": None,
            "droppedRays": None, "convergenceRays": None}


def _train_exact(case, seed):
    X, Y, params = _training_set(case, seed)
    dev = _device()
    X, Y = (torch.as_tensor(v, dtype=torch.float64, device=dev) for v in (X, Y))
    p = torch.as_tensor(params, dtype=torch.float64, device=dev).requires_grad_(True)
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    history = []
    # the run's hyperparameters are 32-bit numbers
    lr, b1, b2, eps, wd = (float(np.float32(x)) for x in (2e-3, 0.9, 0.999, 1e-8, 1e-5))
    for step in range(1, case["epochs"] + 1):
        h = X
        for i, (w, bias) in enumerate(_split_params(p)):
            z = h @ w.T + bias
            h = z * torch.sigmoid(z) if i < 4 else z
        loss = ((h[:, 0] - Y) ** 2).mean()
        history.append(float(loss.detach()))
        g, = torch.autograd.grad(loss, p)
        with torch.no_grad():
            m, v = b1 * m + (1 - b1) * g, b2 * v + (1 - b2) * g * g
            p -= lr * (m / (1 - b1 ** step) / (torch.sqrt(v / (1 - b2 ** step)) + eps) + wd * p)
    return {"params": p.detach(), "history": np.asarray(history)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "estimate":
        p = _Problem(case, seed)
        return _estimate_exact(p, _network(p) if case["proposal"] == "learned" else None)
    if kind == "batch":
        rs = [_estimate_exact(_Problem({**case, "cladding": False}, seed, i)) for i in range(case["problems"])]
        return {n: None if n in WHOLE else np.concatenate([r[n] for r in rs]) for n in FIELDS}
    if kind == "loop":
        return _loop_exact(case, seed)
    if kind == "forward":
        return _forward_exact(case, seed)
    if kind == "train":
        return _train_exact(case, seed)
    p = _Problem({**case, "cladding": True, "min_rays": 1000}, seed)
    g = _Geometry(p)
    samples = torch.arange(p.first, p.last + 1, device=g.v.device)
    tm = _map(g, samples, transfer=True)[:, :, :, torch.as_tensor(g.back, device=g.v.device)]
    return tm.reshape(len(samples), g.R, g.layers * g.T)
