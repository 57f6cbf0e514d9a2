"""Teams whose workgroups keep their rows in LDS and exchange products in
tagged words (krylov_pcg_rows, krylov_bicgstab_rows), at the edges of their
plan: team sizes around the reduction groups of 16, more workgroups than rows,
every column count, scattered numberings whose halo does and does not fit.

Tolerance: the solves stop at |r| <= 1e-12 |b|; the Jacobi-scaled systems here
have condition numbers below 10 and run 3 steps, so the states are within
3e-11 of the oracle's (tol 1e-14).  1e-10 leaves room for the oracle's own."""
import numpy as np
import pytest

import oracle
from femhip import (AdvectionDiffusionParameters, Batch, FEMContext, HeatParameters, SolverOptions, _lib,
                    meshes)

pytestmark = pytest.mark.gpu
TOL = 1e-10
VEL = (0.5, 0.3, 0.0)


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def scattered(m, seed):
    """The mesh with its vertices renumbered at random."""
    n = len(m["xyz"])
    p = np.random.default_rng(seed).permutation(n)
    q = np.empty(n, dtype=np.int64)
    q[p] = np.arange(n)
    return {"xyz": np.ascontiguousarray(m["xyz"][p]),
            "tri": np.ascontiguousarray(q[m["tri"].astype(np.int64)].astype(np.uint32)),
            "on_boundary": np.ascontiguousarray(m["on_boundary"][p])}


def check(m, advdiff, k, precision, steps=3, **opts):
    ctx = FEMContext(m, 0, velocity=VEL, normalize_velocity=False)
    s = oracle.System(m, bc=0, velocity=VEL, normalize=False)
    f = np.random.default_rng(5).standard_normal((s.n, k))
    b = Batch([ctx], SolverOptions(nrhs=k, precision=precision, tol=1e-12, **opts))
    b.set_equation(0, AdvectionDiffusionParameters(1e-3, 0.05) if advdiff else HeatParameters(1e-3, 0.05))
    b.set_state_unknowns(0, _lib.FEM_FIELD_U, f)
    info = b.plan_info()
    assert b.advance(steps) == _lib.FEM_OK
    got = b.get_state_unknowns(0).reshape(-1, k)
    for j in sorted({0, k - 1}):
        if advdiff:
            _, ref, _, _ = s.run(oracle.ADVDIFF, [1e-3, 0.05], steps, f[:, j].copy(), krylov=oracle.BICGSTAB, tol=1e-14)
        else:
            _, ref, _, _ = s.run(oracle.HEAT, [1e-3, 0.05], steps, f[:, j].copy(), tol=1e-14)
        assert rel(got[:, j], ref) <= TOL, j
    b.close()
    ctx.close()
    return info


@pytest.mark.parametrize("precision", [_lib.FEM_PREC_FP32_IR, _lib.FEM_PREC_FP64])
@pytest.mark.parametrize("advdiff", [False, True])
@pytest.mark.parametrize("k,team", [(1, 2), (1, 16), (1, 17), (1, 33), (1, 65), (2, 33), (4, 17), (16, 40), (16, 100)])
def test_team_sizes(gpu, k, team, advdiff, precision):
    print("case rows", k, team, advdiff, precision, flush=True)
    info = check(meshes.jittered_square(40, seed=3), advdiff, k, precision, team_size=team)
    assert info.grid == team


@pytest.mark.parametrize("exchange", [_lib.FEM_EXCHANGE_COHERENT, _lib.FEM_EXCHANGE_FENCED])
@pytest.mark.parametrize("advdiff", [False, True])
def test_more_workgroups_than_rows(gpu, advdiff, exchange):
    print("case few rows", advdiff, exchange, flush=True)
    check(meshes.jittered_square(6, seed=1), advdiff, 1, _lib.FEM_PREC_FP32_IR, team_size=40, exchange=exchange)


@pytest.mark.parametrize("precision", [_lib.FEM_PREC_FP32_IR, _lib.FEM_PREC_FP64])
@pytest.mark.parametrize("advdiff", [False, True])
@pytest.mark.parametrize("side,team", [(30, 4), (78, 6), (110, 12)])
def test_scattered_numbering(gpu, side, team, advdiff, precision):
    """About 1,000 rows per workgroup at the larger sizes: the halo fits in
    FP32 at 6 workgroups, not in FP64, and in neither at 12."""
    print("case scattered", side, team, advdiff, precision, flush=True)
    check(scattered(meshes.jittered_square(side, seed=4), 7), advdiff, 1, precision, team_size=team)


@pytest.mark.parametrize("precision", [_lib.FEM_PREC_FP32_IR, _lib.FEM_PREC_FP64])
def test_launch_plan_kept_over_new_matrices(gpu, precision):
    """New matrices of the same pattern run on the plan built before, halos
    included, and repeat bit for bit."""
    m = meshes.jittered_square(48, seed=2)
    ctx = FEMContext(m, 0)
    s = oracle.System(m, bc=0)
    f = np.random.default_rng(1).standard_normal(s.n)
    b = Batch([ctx], SolverOptions(precision=precision, tol=1e-12))
    seen = []
    for c in (0.05, 0.01, 0.05):
        b.set_equation(0, HeatParameters(1e-3, c))
        b.set_state_unknowns(0, _lib.FEM_FIELD_U, f)
        assert b.advance(3) == _lib.FEM_OK
        got = b.get_state_unknowns(0)
        _, ref, _, _ = s.run(oracle.HEAT, [1e-3, c], 3, f.copy(), tol=1e-14)
        assert rel(got, ref) <= TOL
        seen.append(got)
    assert np.array_equal(seen[0], seen[2])
    b.close()
    ctx.close()


@pytest.mark.parametrize("precision", [_lib.FEM_PREC_FP32_IR, _lib.FEM_PREC_FP64])
@pytest.mark.parametrize("advdiff", [False, True])
@pytest.mark.parametrize("k,team", [(1, 0), (1, 3), (4, 20)])
def test_vertices_without_triangles(gpu, k, team, advdiff, precision):
    """Rows without entries, the first and the last of the pattern among them:
    the phases that read a row's entries all at once leave them out.  The
    streaming engine, whose gathers take them one by one, is the reference."""
    print("case empty rows", k, team, advdiff, precision, flush=True)
    m = meshes.jittered_square(24, seed=5)
    alone = np.zeros((3, 3), np.float32)
    m = {"xyz": np.ascontiguousarray(np.concatenate([alone + 2, m["xyz"], alone + 3])),
         "tri": np.ascontiguousarray(m["tri"] + 3).astype(np.uint32),
         "on_boundary": np.concatenate([np.zeros(3, np.uint8), m["on_boundary"], np.zeros(3, np.uint8)])}
    ctx = FEMContext(m, 1, velocity=VEL, normalize_velocity=False)
    rp, _ = ctx.pattern()
    assert rp[3] == 0 and rp[-1] == rp[-4]
    f = np.random.default_rng(6).standard_normal((len(rp) - 1, k))
    got = []
    for opts in ({"team_size": team}, {"engine": _lib.FEM_ENGINE_STREAM}):
        b = Batch([ctx], SolverOptions(nrhs=k, precision=precision, tol=1e-12, **opts))
        b.set_equation(0, AdvectionDiffusionParameters(1e-3, 0.05) if advdiff else HeatParameters(1e-3, 0.05))
        b.set_state_unknowns(0, _lib.FEM_FIELD_U, f)
        assert b.advance(3) == _lib.FEM_OK
        got.append(b.get_state_unknowns(0).reshape(-1, k))
        b.close()
    assert rel(got[0], got[1]) <= TOL
    ctx.close()
