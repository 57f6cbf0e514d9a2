"""Workloads of the FEM time-stepping backend, as a program that uses it runs them.

``listed()`` names the workloads, ``draw(rng)`` gives others of the same
ranges, ``prepare`` makes what a program has in hand before the call (mesh,
context, solver, fields), ``run`` is one pass through the public interface,
``work`` the bytes and operations that a pass cannot do without, and ``exact``
the same results from 64-bit arithmetic in plain torch.

Kinds:
  steps    a simulation: the initial fields are set, ``steps`` steps run in
           one call, the fields are read back (float surface values; in FP64
           the unknowns themselves)
  frames   the visualiser's loop: every frame hands the surface values in,
           advances one step, reads them back and asks for the normals of the
           extruded surface
  batch    many meshes of uneven size, several right-hand sides each, advanced
           together; the fields of all are read back
  rollout  a training step through torch.autograd: rollout, loss, gradients
           with respect to the initial field and the per-element diffusivity,
           descent step on the diffusivity
  apply    a sparse product on device tensors
  solve    one linear solve of a caller's system on host arrays
  open     a surface is loaded: numbering, CSR pattern and matrices
"""
from __future__ import annotations

import functools
import importlib
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "fea-visualizer_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)


def _fem():
    return importlib.import_module("femhip")


# --------------------------------------------------------------------- cases

def listed():
    return [
        # the reference's plain setting: heat on the structured unit square,
        # FP64, the smallest mesh its examples use for a simulation
        {"name": "heat_square64_f64", "kind": "steps", "eq": "heat", "mesh": "square", "nx": 64, "ny": 64,
         "dirichlet": True, "precision": "f64", "engine": "persistent", "steps": 20, "dt": 1e-3, "c": 1.0},
        # the application's default equation with its default parameters on a
        # small closed surface, frame by frame
        {"name": "frames_wave_sphere4", "kind": "frames", "eq": "wave", "mesh": "sphere", "level": 4, "frames": 8,
         "dt": 0.05, "c": 0.05},
        # Gray-Scott on the icosphere, frame by frame, as it is watched
        {"name": "frames_grayscott_sphere6", "kind": "frames", "eq": "grayscott", "mesh": "sphere", "level": 6,
         "frames": 4, "dt": 0.5, "c": 2e-4},
        # the same simulation run without watching every step
        {"name": "grayscott_sphere6", "kind": "steps", "eq": "grayscott", "mesh": "sphere", "level": 6,
         "dirichlet": False, "precision": "f32", "engine": "persistent", "steps": 100, "dt": 0.5, "c": 2e-4},
        # an ordinary planar simulation with the default options
        {"name": "heat_500x520", "kind": "steps", "eq": "heat", "mesh": "lattice", "nx": 500, "ny": 520,
         "dirichlet": True, "precision": "f32", "engine": "persistent", "steps": 20, "dt": 1e-3, "c": 0.05},
        # a million unknowns: Newmark wave on the engine for large meshes
        {"name": "newmark_1024", "kind": "steps", "eq": "newmark", "mesh": "lattice", "nx": 1024, "ny": 1024,
         "dirichlet": True, "precision": "f32", "engine": "stream", "steps": 10, "dt": 2e-4, "c": 1.0},
        # a parameter study: 16 meshes of uneven size, 16 initial fields each
        {"name": "batch_advdiff_16x16", "kind": "batch", "count": 16, "lo": 32, "hi": 512, "nrhs": 16, "steps": 20,
         "dt": 1e-3},
        # fitting a diffusivity: one gradient step through a rollout
        {"name": "rollout_advdiff_512", "kind": "rollout", "nx": 512, "ny": 512, "steps": 20, "every": 10, "dt": 2e-3},
        # the sparse product alone, one column, a matrix larger than the caches
        {"name": "apply_f32_2048", "kind": "apply", "nx": 2048, "ny": 2048, "precision": "f32", "nrhs": 1},
        # the sparse product on a block of columns
        {"name": "apply_f32_1000x1100_16", "kind": "apply", "nx": 1000, "ny": 1100, "precision": "f32", "nrhs": 16},
        # one implicit solve of the caller's own matrix combination
        {"name": "solve_512", "kind": "solve", "nx": 512, "ny": 512, "precision": "f32", "nrhs": 1, "k": 1e-4},
        # opening a surface in the application
        {"name": "open_lattice_300x310", "kind": "open", "nx": 300, "ny": 310, "dirichlet": True},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "frames", "batch", "rollout", "apply", "apply", "solve", "open"])
    if kind == "steps":
        eq = rng.choice(["heat", "heat", "advdiff", "grayscott", "newmark", "wave"])
        case = {"kind": kind, "eq": eq, "steps": rng.randint(1, 40),
                "precision": rng.choice(["f32", "f32", "f64"])}
        if eq == "grayscott":
            case |= {"mesh": "sphere", "level": rng.randint(2, 6), "dirichlet": False, "engine": "persistent",
                     "dt": round(rng.uniform(0.1, 0.5), 4), "c": round(rng.uniform(1e-4, 3e-4), 7)}
            return case
        side = _logint(rng, 24, 800)
        case |= {"mesh": "lattice", "nx": side, "ny": max(8, side + rng.randint(-side // 4, side // 4)),
                 "dirichlet": rng.random() < 0.7, "engine": "stream" if side > 450 else "persistent"}
        case |= {"heat": {"dt": 1e-3, "c": round(rng.uniform(0.02, 0.3), 4)},
                 "advdiff": {"dt": 1e-3, "c": round(rng.uniform(0.005, 0.1), 4)},
                 "newmark": {"dt": 2e-4, "c": 1.0},
                 "wave": {"dt": 0.01, "c": 0.05}}[eq]
        return case
    if kind == "frames":
        eq = rng.choice(["wave", "heat", "grayscott"])
        return {"kind": kind, "eq": eq, "mesh": "sphere", "level": rng.randint(2, 6), "frames": rng.randint(1, 8),
                "dt": {"wave": 0.05, "heat": 0.01, "grayscott": round(rng.uniform(0.1, 0.5), 4)}[eq],
                "c": {"wave": 0.05, "heat": 0.05, "grayscott": 2e-4}[eq]}
    if kind == "batch":
        nrhs = rng.choice([1, 4, 16])
        return {"kind": kind, "count": rng.randint(2, 16), "lo": 24, "hi": rng.randint(60, 400), "nrhs": nrhs,
                "steps": rng.randint(2, 20), "dt": 1e-3}
    if kind == "rollout":
        side = _logint(rng, 40, 480)
        return {"kind": kind, "nx": side, "ny": max(8, side + rng.randint(-side // 5, side // 5)),
                "steps": rng.randint(4, 20), "every": rng.randint(2, 10), "dt": 2e-3}
    if kind == "apply":
        k = rng.choice([1, 1, 2, 4, 16])
        side = _logint(rng, 64, 1500 if k == 1 else 1100 if k < 16 else 700)
        return {"kind": kind, "nx": side, "ny": max(8, side + rng.randint(-side // 4, side // 4)),
                "precision": rng.choice(["f32", "f64"]), "nrhs": k}
    if kind == "solve":
        side = _logint(rng, 32, 512)
        return {"kind": kind, "nx": side, "ny": max(8, side + rng.randint(-side // 4, side // 4)),
                "precision": rng.choice(["f32", "f32", "f64"]), "nrhs": rng.choice([1, 1, 4]),
                "k": round(math.exp(rng.uniform(math.log(1e-5), math.log(2e-4))), 9)}
    side = _logint(rng, 32, 600)
    return {"kind": kind, "nx": side, "ny": max(8, side + rng.randint(-side // 4, side // 4)),
            "dirichlet": rng.random() < 0.5}


# -------------------------------------------------------------------- meshes

@functools.lru_cache(maxsize=32)
def _lattice(nx, ny, jitter, seed):
    """(nx+1) x (ny+1) vertices on a rectangle with unit short side, interior
    ones moved by up to jitter cells, each cell split along one of its
    diagonals (a hash of the cell decides)."""
    h = 1.0 / min(nx, ny)
    rng = np.random.Generator(np.random.PCG64(seed))
    i, j = np.meshgrid(np.arange(nx + 1), np.arange(ny + 1), indexing="xy")
    x, y = i.ravel() * h, j.ravel() * h
    edge = ((i == 0) | (i == nx) | (j == 0) | (j == ny)).ravel()
    if jitter:
        d = rng.uniform(-jitter * h, jitter * h, size=(2, x.size))
        x = np.where(edge, x, x + d[0])
        y = np.where(edge, y, y + d[1])
    ci, cj = np.meshgrid(np.arange(nx), np.arange(ny), indexing="xy")
    a = (cj * (nx + 1) + ci).ravel()
    b, c, d4 = a + 1, a + nx + 1, a + nx + 2
    flip = (rng.random(a.size) < 0.5)[:, None] if jitter else np.zeros((a.size, 1), bool)
    t1 = np.where(flip, np.stack([a, b, c], 1), np.stack([a, b, d4], 1))
    t2 = np.where(flip, np.stack([b, d4, c], 1), np.stack([a, d4, c], 1))
    return {"xyz": np.ascontiguousarray(np.stack([x, y, np.zeros_like(x)], 1), dtype=np.float32),
            "tri": np.ascontiguousarray(np.stack([t1, t2], 1).reshape(-1, 3), dtype=np.uint32),
            "on_boundary": edge.astype(np.uint8)}


@functools.lru_cache(maxsize=8)
def _sphere(level):
    m = _fem().icosphere(level)
    n = m["xyz"].astype(np.float64)
    m["normals"] = np.ascontiguousarray(n / np.linalg.norm(n, axis=1, keepdims=True), dtype=np.float32)
    return m


def _mesh(case):
    if case.get("mesh") == "sphere":
        return _sphere(case["level"])
    if case.get("mesh") == "square":
        return _lattice(case["nx"], case["ny"], 0.0, 0)
    return _lattice(case["nx"], case["ny"], 0.2, 2)


def _bumps(X, rng, count, sigma):
    out = np.zeros(len(X))
    lo, hi = X.min(0), X.max(0)
    for _ in range(count):
        c = lo + (hi - lo) * rng.uniform(0.2, 0.8, 3)
        if hi[2] > lo[2]:  # closed surfaces: on the sphere
            c = c / max(np.linalg.norm(c), 1e-9)
        out += rng.uniform(0.5, 1.0) * np.exp(-((X - c) ** 2).sum(1) / (2 * sigma ** 2))
    return out


def _patches(X, rng):
    """Gray-Scott's usual start: u = 1, v = 0, and 50 round patches of v."""
    u, v = np.ones(len(X)), np.zeros(len(X))
    for q in rng.integers(0, len(X), 50):
        near = ((X - X[q]) ** 2).sum(1) < 0.1 ** 2
        v[near] = 0.25 + rng.uniform(-0.05, 0.05, int(near.sum()))
    return u, v


def _fields(case, X, seed):
    """Initial surface values (float32), one array per state field."""
    rng = np.random.Generator(np.random.PCG64(seed))
    eq = case["eq"]
    if eq == "grayscott":
        f = _patches(X, rng)
    elif eq in ("wave", "newmark"):
        f = (_bumps(X, rng, 8, 0.08 if case["mesh"] == "sphere" else 0.03), np.zeros(len(X)))
    else:
        f = (_bumps(X, rng, 4, 0.1),)
    return [np.ascontiguousarray(a, dtype=np.float32) for a in f]


def _batch_specs(case, seed):
    shape = np.random.Generator(np.random.PCG64(4))  # the study's meshes
    rng = np.random.Generator(np.random.PCG64(seed))
    specs = []
    for i in range(case["count"]):
        side = int(round(math.exp(shape.uniform(math.log(case["lo"]), math.log(case["hi"])))))
        kap = float(math.exp(shape.uniform(math.log(1e-4), math.log(1e-1))))
        sp, th = shape.uniform(0, 1), shape.uniform(0, 2 * math.pi)
        m = _lattice(side, side, 0.2, 100 + i)
        X = m["xyz"].astype(np.float64)[m["on_boundary"] == 0]
        cols = [_bumps(X, rng, 1, rng.uniform(0.02, 0.1)) for _ in range(case["nrhs"])]
        specs.append((m, kap, (sp * math.cos(th), sp * math.sin(th), 0.0), np.ascontiguousarray(np.stack(cols, 1))))
    return specs


def _rollout_inputs(case, seed):
    m = _mesh(case)
    X = m["xyz"].astype(np.float64)
    cen = X[m["tri"]].mean(axis=1)
    ve = np.stack([-(cen[:, 1] - 0.5), cen[:, 0] - 0.5, np.zeros(len(cen))], axis=1)
    rng = np.random.Generator(np.random.PCG64(seed))
    kappa = 1e-3 * np.exp(0.3 * rng.standard_normal(len(m["tri"])))
    Xi = X[m["on_boundary"] == 0]
    f32 = [a.astype(np.float32) for a in (kappa, _bumps(Xi, rng, 2, 0.06), _bumps(Xi, rng, 2, 0.06))]
    return (m, ve, *f32)  # torch's default type, as a training program holds them


def _coef(case):
    return (1.0, case["k"], 0.0) if case["kind"] == "solve" else (1000.0, 1.0, 0.0)


# ------------------------------------------------------------------- prepare

def _params(F, case):
    eq, dt, c = case["eq"], case["dt"], case["c"]
    if eq == "heat":
        return F.Equation.Heat, F.HeatParameters(dt, c)
    if eq == "advdiff":
        return F.Equation.Advection_Diffusion, F.AdvectionDiffusionParameters(dt, c)
    if eq == "wave":
        return F.Equation.Wave, F.WaveParameters(dt, c)
    if eq == "newmark":
        return F.Equation.Wave_Newmark, F.NewmarkParameters(dt, c, 0.25, 0.5)
    return F.Equation.Reaction_Diffusion, F.ReactionDiffusionParameters(
        dt, c, 0.5 * c, 0.037, 0.06, F._lib.FEM_REACTION_LUMPED)


def _precision(F, case):
    return F._lib.FEM_PREC_FP64 if case["precision"] == "f64" else F._lib.FEM_PREC_FP32_IR


def _context(F, case, m, dirichlet, **kw):
    c = F.FEMContext(m, F.BoundaryCondition.Dirichlet if dirichlet else F.BoundaryCondition.Neumann, **kw)
    if "eq" in case:
        c.equation, prm = _params(F, case)
        c.parameters[c.equation] = prm
    return c


def prepare(case, seed):
    F = _fem()
    L = F._lib
    kind = case["kind"]
    st = {"case": case}
    if kind in ("steps", "frames"):
        m = _mesh(case)
        st["mesh"] = m
        st["ctx"] = _context(F, case, m, case.get("dirichlet", False))
        opts = {}
        if kind == "steps":
            opts = {"precision": _precision(F, case),
                    "engine": L.FEM_ENGINE_STREAM if case["engine"] == "stream" else L.FEM_ENGINE_PERSISTENT}
            if case["engine"] == "stream":
                opts["inner_tol"] = 1e-6
        st["solver"] = F.HIPSolver(st["ctx"], F.SolverOptions(**opts))
        st["fields"] = _fields(case, m["xyz"].astype(np.float64), seed)
        st["f64"] = case.get("precision") == "f64"
        if st["f64"]:
            keep = st["ctx"].idx_map >= 0
            st["fields"] = [np.ascontiguousarray(f[keep], dtype=np.float64) for f in st["fields"]]
    elif kind == "batch":
        specs = _batch_specs(case, seed)
        st["ctxs"] = [F.FEMContext(m, 0, velocity=v, normalize_velocity=False) for m, _, v, _ in specs]
        b = F.Batch(st["ctxs"], F.SolverOptions(nrhs=case["nrhs"], engine=L.FEM_ENGINE_STREAM, inner_tol=1e-6))
        for i, (_, kap, _, f) in enumerate(specs):
            b.set_equation(i, F.AdvectionDiffusionParameters(case["dt"], kap))
            b.set_state_unknowns(i, L.FEM_FIELD_U, f)
        st["batch"] = b
    elif kind == "rollout":
        A = importlib.import_module("femhip.autograd")
        m, ve, kappa, u0, target = _rollout_inputs(case, seed)
        st["model"] = A.Rollout(m, F.AdvectionDiffusionParameters(case["dt"], 1.0), case["steps"], case["every"],
                                velocity_e=ve, normalize_velocity=False)
        dev = "cuda"
        st["kappa"] = torch.tensor(kappa, device=dev, requires_grad=True)
        st["u0"] = torch.tensor(u0, device=dev, requires_grad=True)
        st["target"] = torch.tensor(target, device=dev)
    elif kind == "apply":
        m = _mesh(case)
        st["ctx"] = F.FEMContext(m, 0)
        st["op"] = F.Operator(st["ctx"], _coef(case), _precision(F, case))
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        dt = torch.float64 if case["precision"] == "f64" else torch.float32
        st["x"] = torch.randn((st["op"].n, case["nrhs"]), generator=g, device="cuda", dtype=dt)
        st["y"] = torch.empty_like(st["x"])
        torch.cuda.synchronize()
    elif kind == "solve":
        m = _mesh(case)
        st["ctx"] = F.FEMContext(m, 0)
        st["opts"] = F.SolverOptions(precision=_precision(F, case))
        st["b"] = _solve_rhs(case, m, seed)
    else:
        st["mesh"] = _moved(case, seed)
    return st


def _solve_rhs(case, m, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    X = m["xyz"].astype(np.float64)[m["on_boundary"] == 0]
    cols = [_bumps(X, rng, 3, 0.1) for _ in range(case["nrhs"])]
    h2 = 1.0 / min(case["nx"], case["ny"]) ** 2
    return np.ascontiguousarray(h2 * (cols[0] if case["nrhs"] == 1 else np.stack(cols, 1)))


def _moved(case, seed):
    """The surface to open: the lattice, lifted by a smooth height field."""
    m = dict(_mesh(case))
    rng = np.random.Generator(np.random.PCG64(seed))
    xyz = m["xyz"].astype(np.float64)
    xyz[:, 2] = 0.2 * np.sin(xyz[:, 0] * rng.uniform(2, 6)) * np.cos(xyz[:, 1] * rng.uniform(2, 6))
    m["xyz"] = xyz.astype(np.float32)
    return m


# ----------------------------------------------------------------------- run

def run(st):
    F = _fem()
    L = F._lib
    case = st["case"]
    kind = case["kind"]
    if kind == "steps":
        s = st["solver"]
        put, get = (s.set_state_unknowns, s.get_state_unknowns) if st["f64"] else (s.set_state, s.get_state)
        for q, f in enumerate(st["fields"]):
            put(q, f)
        if case["eq"] == "newmark":
            put(L.FEM_FIELD_A, st["fields"][1])  # at rest: zero, as the velocity
        s.advance_time(case["steps"])
        return [get(q) for q in range(len(st["fields"]))]
    if kind == "frames":
        s, m = st["solver"], st["mesh"]
        shown = L.FEM_FIELD_V if case["eq"] == "grayscott" else L.FEM_FIELD_U
        for q, f in enumerate(st["fields"]):
            s.set_state(q, f)
        vals = st["fields"][shown]
        normals = None
        for _ in range(case["frames"]):
            s.set_state(shown, vals)
            s.advance_time()
            vals = s.get_state(shown)
            normals = s.smooth_normals(m["normals"], 0.25)
        return {"values": vals, "normals": normals}
    if kind == "batch":
        b = st["batch"]
        b.advance(case["steps"])
        return [b.get_state_unknowns(i) for i in range(case["count"])]
    if kind == "rollout":
        uT = st["model"](st["u0"], st["kappa"])
        loss = ((uT - st["target"]) ** 2).mean()
        gu, gk = torch.autograd.grad(loss, (st["u0"], st["kappa"]))
        with torch.no_grad():
            st["kappa"].sub_(gk, alpha=1e-2)
        return {"uT": uT.detach(), "grad_u0": gu, "grad_kappa": gk}
    if kind == "apply":
        st["op"].apply_device(case["nrhs"], st["x"].data_ptr(), st["y"].data_ptr())
        st["op"].sync()
        return st["y"]
    if kind == "solve":
        return st["ctx"].solve(_coef(case), st["b"], st["opts"])
    c = F.FEMContext(st["mesh"], 0 if case["dirichlet"] else 1)
    rp, ci = c.pattern()
    out = {"row_ptr": rp, "col_idx": ci, "idx_map": c.idx_map, "K": c.matrix(L.FEM_MATRIX_K),
           "M": c.matrix(L.FEM_MATRIX_M)}
    c.close()
    return out


# ---------------------------------------------------------------------- work

def _size(case):
    """(vertices, unknowns, nonzeros) of a case's mesh, about (lattice)."""
    if case.get("mesh") == "sphere":
        nv = 10 * 4 ** case["level"] + 2
        return nv, nv, 7 * nv
    nv = (case["nx"] + 1) * (case["ny"] + 1)
    n = nv if not case.get("dirichlet", True) else (case["nx"] - 1) * (case["ny"] - 1)
    return nv, n, 7 * n


def _step_work(n, nnz, k, kv, fields):
    """One implicit step: the system and mass matrices and the pattern read
    once, the fields read and written once; one product with each matrix."""
    return nnz * (4 + 8 * kv + 8) + 16 * n * k * fields, 4 * nnz * k


def work(case):
    kind = case["kind"]
    if kind in ("steps", "frames"):
        nv, n, nnz = _size(case)
        gs = case["eq"] == "grayscott"
        k = 2 if gs else 1
        fields = {"wave": 2, "newmark": 3}.get(case["eq"], 1)
        by, fl = _step_work(n, nnz, k, k, fields)
        reps = case["steps"] if kind == "steps" else case["frames"]
        io = 8 * nv * (k if gs else fields)
        if kind == "frames":
            io = reps * (8 * nv + 24 * nv + 24 * nv)  # values in and out, normals in and out, triangles
            fl += 60 * nv
        return {"bytes": float(reps * by + io), "flops": float(reps * fl)}
    if kind == "batch":
        shape = np.random.Generator(np.random.PCG64(4))
        by = fl = 0.0
        for _ in range(case["count"]):
            side = int(round(math.exp(shape.uniform(math.log(case["lo"]), math.log(case["hi"])))))
            shape.uniform(size=3)
            n = (side - 1) ** 2
            b1, f1 = _step_work(n, 7 * n, case["nrhs"], 1, 1)
            by += case["steps"] * b1 + 8 * n * case["nrhs"]
            fl += case["steps"] * f1
        return {"bytes": by, "flops": fl}
    nv, n, nnz = _size(case)
    if kind == "rollout":
        by, fl = _step_work(n, nnz, 1, 1, 1)
        tri = 2 * case["nx"] * case["ny"]
        # forward steps, adjoint steps, and the gradient's pass over the states
        return {"bytes": float(2 * case["steps"] * by + tri * (12 + 16) + 16 * n * case["steps"]),
                "flops": float(2 * case["steps"] * fl + 30 * tri * case["steps"])}
    if kind == "apply":
        s = 8 if case["precision"] == "f64" else 4
        return {"bytes": float(nnz * (4 + s) + 4 * n + 2 * n * case["nrhs"] * s), "flops": 2.0 * nnz * case["nrhs"]}
    if kind == "solve":
        return {"bytes": float(nnz * 20 + 16 * n * case["nrhs"]), "flops": 2.0 * nnz * case["nrhs"]}
    tri = 2 * case["nx"] * case["ny"]
    return {"bytes": float(12 * nv + 12 * tri + nv + nnz * 20 + 8 * n), "flops": float(200 * tri)}


# --------------------------------------------------------------------- exact

class _System:
    """K, M, A of a mesh in 64-bit torch (sparse CSR), assembled from the
    linear element formulas."""

    def __init__(self, m, dirichlet, velocity=None, velocity_e=None, normalize=True, kappa=None):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        X = m["xyz"].astype(np.float64)
        T = m["tri"].astype(np.int64)
        onb = m["on_boundary"].astype(bool) & dirichlet
        self.keep = ~onb
        self.idx = np.where(onb, -1, np.cumsum(~onb) - 1)
        self.n = int((~onb).sum())
        a, b, c = X[T[:, 0]], X[T[:, 1]], X[T[:, 2]]
        cr = np.cross(b - a, c - a)
        two = np.linalg.norm(cr, axis=1)
        nrm = cr / two[:, None]
        # gradient of the hat at a vertex: normal x opposite edge / (2 area)
        g = np.stack([np.cross(nrm, c - b), np.cross(nrm, a - c), np.cross(nrm, b - a)], 1) / two[:, None, None]
        kab = 0.5 * two[:, None, None] * np.einsum("eai,ebi->eab", g, g)
        self.kab = kab if kappa is None else None
        self.k_unit = kab
        kk = kab if kappa is None else kab * kappa[:, None, None]
        mm = two[:, None, None] / 24.0 * (np.ones((3, 3)) + np.eye(3))
        if velocity_e is None:
            velocity_e = np.broadcast_to(np.asarray(velocity if velocity is not None else (1.0, 0, 0), float),
                                         nrm.shape)
        tv = velocity_e - (velocity_e * nrm).sum(1)[:, None] * nrm
        if normalize:
            ln = np.linalg.norm(tv, axis=1)
            tv = tv / np.where(ln > 0, ln, 1.0)[:, None]
        aa = np.broadcast_to((two / 6.0)[:, None, None] * np.einsum("ei,ebi->eb", tv, g)[:, None, :], kk.shape)
        I = self.idx[T]
        r = np.broadcast_to(I[:, :, None], kk.shape).ravel()
        s = np.broadcast_to(I[:, None, :], kk.shape).ravel()
        on = m["on_boundary"].astype(bool)[T]
        free = ~np.broadcast_to(on[:, :, None] | on[:, None, :], kk.shape).ravel()
        ok = (r >= 0) & (s >= 0)
        self.tri = T
        self.K, self.M = (self._csr(r[ok], s[ok], v.ravel()[ok]) for v in (kk, mm))
        self.A = self._csr(r[ok], s[ok], np.where(free, aa.ravel(), 0.0)[ok])

    def _csr(self, r, s, v):
        t = torch.sparse_coo_tensor(torch.from_numpy(np.stack([r, s])).to(self.dev), torch.from_numpy(v).to(self.dev),
                                    (self.n, self.n)).coalesce()
        return t.to_sparse_csr()

    def mix(self, cM, cK, cA=0.0):
        v = cM * self.M.values() + cK * self.K.values() + cA * self.A.values()
        return torch.sparse_csr_tensor(self.M.crow_indices(), self.M.col_indices(), v, (self.n, self.n))


def _diag(S):
    rows = torch.repeat_interleave(torch.arange(S.shape[0], device=S.device), S.crow_indices().diff())
    return S.values()[rows == S.col_indices()]


def _solve(S, b, x0=None, tol=1e-15, symmetric=True):
    """Jacobi-preconditioned CG or BiCGSTAB per column in 64 bits; b is [n, k]."""
    d = 1.0 / _diag(S)[:, None]
    x = torch.zeros_like(b) if x0 is None else x0.clone()
    bn = b.square().sum(0).sqrt().clamp_min(1e-300)
    for _ in range(3):  # the true residual is taken anew
        r = b - S @ x
        if float((r.square().sum(0).sqrt() / bn).max()) < tol:
            break
        if symmetric:
            z = d * r
            p, rz = z.clone(), (r * z).sum(0)
            for it in range(2000):
                q = S @ p
                al = rz / (p * q).sum(0).clamp_min(1e-300)
                x += al * p
                r -= al * q
                z = d * r
                new = (r * z).sum(0)
                p = z + (new / rz.clamp_min(1e-300)) * p
                rz = new
                if it % 5 == 4 and float((r.square().sum(0).sqrt() / bn).max()) < tol / 4:
                    break
        else:
            rh = r.clone()
            p, rho = r.clone(), (rh * r).sum(0)
            tiny = lambda t: torch.where(t.abs() < 1e-300, torch.full_like(t, 1e-300), t)  # noqa: E731
            for it in range(2000):
                v = S @ (d * p)
                al = rho / tiny((rh * v).sum(0))
                s = r - al * v
                t = S @ (d * s)
                om = (t * s).sum(0) / tiny((t * t).sum(0))
                x += d * (al * p + om * s)
                r = s - om * t
                new = (rh * r).sum(0)
                p = r + (new / tiny(rho)) * (al / tiny(om)) * (p - om * v)
                rho = new
                if it % 3 == 2 and float((r.square().sum(0).sqrt() / bn).max()) < tol / 4:
                    break
    return x


def _col(a, keep, dev):
    return torch.from_numpy(np.ascontiguousarray(a[keep], dtype=np.float64)).to(dev)[:, None]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("steps", "frames"):
        m = _mesh(case)
        dirichlet = bool(case.get("dirichlet", False))
        s = _System(m, dirichlet)
        f = [_col(a, s.keep, s.dev) for a in _fields(case, m["xyz"].astype(np.float64), seed)]
        out = _trajectory(s, case, f, case["steps"] if kind == "steps" else case["frames"])

        def surface(x):
            full = np.zeros(len(s.idx))
            full[s.keep] = x[:, 0].cpu().numpy()
            return full
        if kind == "steps":
            return [x[:, 0] if case["precision"] == "f64" else surface(x) for x in out]
        v = surface(out[1 if case["eq"] == "grayscott" else 0])
        return {"values": v, "normals": _normals(m, v, 0.25)}
    if kind == "batch":
        out = []
        for m, kap, vel, f in _batch_specs(case, seed):
            s = _System(m, True, velocity=vel, normalize=False)
            S, x = s.mix(1 / case["dt"], kap, -1.0), torch.from_numpy(f).to(s.dev)
            for _ in range(case["steps"]):
                x = _solve(S, s.M @ x / case["dt"], x, symmetric=False)
            out.append(x.reshape(-1))
        return out
    if kind == "rollout":
        m, ve, kappa, u0, target = _rollout_inputs(case, seed)
        s = _System(m, True, velocity_e=ve, normalize=False, kappa=kappa.astype(np.float64))
        u0, target = u0.astype(np.float64), target.astype(np.float64)
        dt = case["dt"]
        S = s.mix(1 / dt, 1.0, -1.0)
        St = S.to_sparse_coo().t().coalesce().to_sparse_csr()
        us = [torch.from_numpy(u0).to(s.dev)[:, None]]
        for _ in range(case["steps"]):
            us.append(_solve(S, s.M @ us[-1] / dt, us[-1], symmetric=False))
        g = 2.0 * (us[-1] - torch.from_numpy(target).to(s.dev)[:, None]) / s.n
        mu = _solve(St, g, symmetric=False)
        ke = torch.from_numpy(s.k_unit).to(s.dev)
        idx = torch.from_numpy(s.idx[s.tri]).to(s.dev)
        at = lambda x: torch.where(idx >= 0, x[:, 0][idx.clamp_min(0)], 0.0)  # noqa: E731
        gk = torch.zeros(len(s.tri), dtype=torch.float64, device=s.dev)
        for t in range(case["steps"], 0, -1):
            gk -= (at(mu)[:, :, None] * ke * at(us[t])[:, None, :]).sum((1, 2))
            if t > 1:
                mu = _solve(St, s.M @ mu / dt, mu, symmetric=False)
        return {"uT": us[-1][:, 0], "grad_u0": (s.M @ mu)[:, 0] / dt, "grad_kappa": gk}
    if kind == "apply":
        if case["nx"] * case["ny"] > 1500 * 1500:
            return None  # assembling it takes too long here
        s = _System(_mesh(case), True)
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        dt = torch.float64 if case["precision"] == "f64" else torch.float32
        return s.mix(1000.0, 1.0) @ torch.randn((s.n, case["nrhs"]), generator=g, device="cuda", dtype=dt).double()
    if kind == "solve":
        m = _mesh(case)
        s = _System(m, True)
        b = torch.from_numpy(_solve_rhs(case, m, seed)).to(s.dev)
        x = _solve(s.mix(1.0, case["k"]), b.reshape(s.n, -1))
        return x.reshape(b.shape)
    s = _System(_moved(case, seed), case["dirichlet"])
    return {"row_ptr": None, "col_idx": None, "idx_map": None, "K": s.K.values(), "M": s.M.values()}


def _trajectory(s, case, f, steps):
    eq, dt, c = case["eq"], case["dt"], case["c"]
    if eq in ("heat", "advdiff"):
        S = s.mix(1 / dt, c, -1.0 if eq == "advdiff" else 0.0)
        for _ in range(steps):
            f = [_solve(S, s.M @ f[0] / dt, f[0], symmetric=eq == "heat")]
        return f
    if eq == "wave":  # velocity-form backward Euler
        u, v = f
        S = s.mix(1 / dt, c * c * dt)
        for _ in range(steps):
            v = _solve(S, s.M @ v / dt - c * c * (s.K @ u), v)
            u = u + dt * v
        return [u, v]
    if eq == "newmark":
        u, v = f
        a = torch.zeros_like(u)
        S = s.mix(1.0, 0.25 * dt * dt * c * c)
        for _ in range(steps):
            ut = u + dt * v + 0.25 * dt * dt * a
            an = _solve(S, -c * c * (s.K @ ut), a)
            u, v, a = ut + 0.25 * dt * dt * an, v + 0.5 * dt * (a + an), an
        return [u, v]
    u, v = f
    Su, Sv = s.mix(1 / dt, c), s.mix(1 / dt, 0.5 * c)
    w = (s.M @ torch.ones_like(u))
    for _ in range(steps):
        uvv = u * v * v
        bu = s.M @ u / dt + w * (-uvv + 0.037 * (1 - u))
        bv = s.M @ v / dt + w * (uvv - (0.037 + 0.06) * v)
        u, v = _solve(Su, bu, u), _solve(Sv, bv, v)
    return [u, v]


def _normals(m, val, extrusion):
    X, T = m["xyz"].astype(np.float64), m["tri"].astype(np.int64)
    P = X + np.minimum(1.0, extrusion * np.maximum(0.0, val))[:, None] * m["normals"].astype(np.float64)
    fn = np.cross(P[T[:, 1]] - P[T[:, 0]], P[T[:, 2]] - P[T[:, 0]])
    out = np.zeros_like(X)
    for a in range(3):
        np.add.at(out, T[:, a], fn)
    return out
