"""The plan rules of the persistent engine at the sizes where they change.

Tolerances as in test_gpu_team_rows: solves to 1e-12 of Jacobi-scaled systems,
here with condition numbers up to 16, and 3 steps, so the states are within 5e-11
of the oracle's."""
import numpy as np
import pytest

import oracle
from femhip import AdvectionDiffusionParameters, Batch, FEMContext, HeatParameters, SolverOptions, _lib, meshes
from test_gpu_team_rows import TOL, VEL, check, rel, scattered
from test_zz_no_alloc import solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,k,grid", [(3, 1, 1), (13, 1, 1), (17, 1, 1), (23, 1, 1), (24, 1, 5), (17, 2, 1), (18, 2, 5),
                                          (12, 4, 1), (6, 16, 1), (7, 16, 5)])
@pytest.mark.parametrize("krylov", [_lib.FEM_KRYLOV_CG, _lib.FEM_KRYLOV_BICGSTAB, _lib.FEM_KRYLOV_CG_CLASSIC])
def test_one_workgroup_up_to_two_rows_per_lane(gpu, cells, k, grid, krylov):
    """(cells - 1)^2 unknowns: up to 512 rows x columns one workgroup has no
    barrier across the chip, whatever the method; beyond, one per 128."""
    print("case one workgroup", cells, k, krylov, flush=True)
    info = check(meshes.jittered_square(cells, seed=6), False, k, _lib.FEM_PREC_FP32_IR, krylov=krylov, max_iters=1000)
    assert info.grid == grid and (info.exchange == 0) == (grid == 1)


def fan_square(cells, seed):
    """A jittered square whose vertex in the middle is joined to all vertices
    within four cells, which leaves rows past the 10 entries that stay in LDS."""
    m = meshes.jittered_square(cells, seed=seed)
    side, c, r = cells + 1, cells // 2, 4
    idx = np.arange(side * side).reshape(side, side)
    drop = idx[c - r + 1:c + r, c - r + 1:c + r].ravel()
    hub = idx[c, c]
    keep = m["tri"][~np.isin(m["tri"], drop).any(1)]
    ring = np.concatenate([idx[c - r, c - r:c + r], idx[c - r:c + r, c + r], idx[c + r, c + r:c - r:-1],
                           idx[c + r:c - r:-1, c - r]])
    tri = np.concatenate([keep, np.stack([np.full(len(ring), hub), ring, np.roll(ring, -1)], 1)])
    used = np.zeros(side * side, bool)
    used[tri] = True
    to = np.cumsum(used) - 1
    return {"xyz": np.ascontiguousarray(m["xyz"][used]), "tri": to[tri].astype(np.uint32),
            "on_boundary": np.ascontiguousarray(m["on_boundary"][used])}


@pytest.mark.parametrize("mesh,precision,krylov,grid", [
    ("lattice", _lib.FEM_PREC_FP32_IR, _lib.FEM_KRYLOV_CG, 64), ("lattice", _lib.FEM_PREC_FP64, _lib.FEM_KRYLOV_CG, 64),
    ("lattice", _lib.FEM_PREC_FP32_IR, _lib.FEM_KRYLOV_CG_CLASSIC, 256),
    ("long rows", _lib.FEM_PREC_FP32_IR, _lib.FEM_KRYLOV_CG, 256), ("long rows", _lib.FEM_PREC_FP64, _lib.FEM_KRYLOV_BICGSTAB, 256),
    ("scattered", _lib.FEM_PREC_FP32_IR, _lib.FEM_KRYLOV_CG, 64), ("scattered", _lib.FEM_PREC_FP64, _lib.FEM_KRYLOV_CG, 256)])
def test_team_of_rows_not_in_lds(gpu, mesh, precision, krylov, grid):
    """About 39,000 unknowns: a team of 64 keeps 620 rows a workgroup in LDS, but
    not with classic CG, rows of more than 10 entries, or, in FP64, the halo of a
    scattered numbering (about 3,500 rows, where 1,141 fit).  Such teams get one
    workgroup per 128 rows, and the solves without allocation the same plan."""
    print("case rows not in LDS", mesh, precision, krylov, flush=True)
    m = fan_square(200, 3) if mesh == "long rows" else meshes.jittered_square(198, seed=3)
    m = scattered(m, 5) if mesh == "scattered" else m
    info = check(m, False, 1, precision, krylov=krylov)
    assert (info.grid, info.exchange) == (grid, _lib.FEM_EXCHANGE_COHERENT)
    ctx = FEMContext(m, 0)
    b = np.random.default_rng(16).standard_normal(ctx.num_unknowns())
    got = [solve(gpu, ctx, fn, (1000.0, 0.05, 0.0), b, SolverOptions(precision=precision, krylov=krylov))
           for fn in ("fem_ctx_solve", "fem_ctx_solve_noalloc")]
    assert got[0][0] == got[1][0] == _lib.FEM_OK
    assert np.array_equal(got[0][1], got[1][1])
    ctx.close()


@pytest.mark.parametrize("precision", [_lib.FEM_PREC_FP32_IR, _lib.FEM_PREC_FP64])
@pytest.mark.parametrize("advdiff", [False, True])
@pytest.mark.parametrize("order", [(0, 1, 2), (1, 2, 0)])
def test_batch_of_fitting_and_other_halos(gpu, order, advdiff, precision):
    """A lattice, a scattered numbering whose halo fits in FP32 and not in FP64
    (about 1,000 rows per workgroup), and a mesh with a long row, in one plan."""
    print("case mixed halos", order, advdiff, precision, flush=True)
    mesh = [(meshes.jittered_square(30, seed=4)), scattered(meshes.jittered_square(78, seed=4), 7), fan_square(30, 4)]
    mesh = [mesh[i] for i in order]
    ctxs = [FEMContext(m, 0, velocity=VEL, normalize_velocity=False) for m in mesh]
    b = Batch(ctxs, SolverOptions(precision=precision, tol=1e-12, team_size=6))
    refs = []
    for i, m in enumerate(mesh):
        s = oracle.System(m, bc=0, velocity=VEL, normalize=False)
        f = np.random.default_rng(17 + i).standard_normal(s.n)
        b.set_equation(i, AdvectionDiffusionParameters(1e-3, 0.05) if advdiff else HeatParameters(1e-3, 0.05))
        b.set_state_unknowns(i, _lib.FEM_FIELD_U, f)
        kw = {"krylov": oracle.BICGSTAB} if advdiff else {}
        refs.append(s.run(oracle.ADVDIFF if advdiff else oracle.HEAT, [1e-3, 0.05], 3, f.copy(), tol=1e-14, **kw)[1])
    assert b.plan_info().grid == 18
    assert b.advance(3) == _lib.FEM_OK
    for i, ref in enumerate(refs):
        assert rel(b.get_state_unknowns(i), ref) <= TOL, i
    b.close()
    for c in ctxs:
        c.close()


@pytest.mark.parametrize("count,grid", [(256, 256), (257, 257), (300, 300), (512, 512), (513, 512)])
@pytest.mark.parametrize("advdiff", [False, True])
def test_more_instances_than_cus(gpu, advdiff, count, grid):
    """Equal instances, past one per CU: one-workgroup teams, two of which fit a CU."""
    print("case many instances", count, advdiff, flush=True)
    m = meshes.jittered_square(17, seed=4)
    ctx = FEMContext(m, 0, velocity=VEL, normalize_velocity=False)
    s = oracle.System(m, bc=0, velocity=VEL, normalize=False)
    b = Batch([ctx] * count, SolverOptions(tol=1e-12))
    f = np.random.default_rng(18).standard_normal((count, s.n))
    for i in range(count):
        b.set_equation(i, AdvectionDiffusionParameters(1e-3, 0.05) if advdiff else HeatParameters(1e-3, 0.05))
        b.set_state_unknowns(i, _lib.FEM_FIELD_U, f[i])
    info = b.plan_info()
    assert (info.grid, info.exchange) == (grid, 0)
    assert b.advance(3) == _lib.FEM_OK
    for i in (0, 255, count - 1):
        kw = {"krylov": oracle.BICGSTAB} if advdiff else {}
        ref = s.run(oracle.ADVDIFF if advdiff else oracle.HEAT, [1e-3, 0.05], 3, f[i].copy(), tol=1e-14, **kw)[1]
        assert rel(b.get_state_unknowns(i), ref) <= TOL, i
    b.close()
    ctx.close()


@pytest.mark.parametrize("precision", [_lib.FEM_PREC_FP32_IR, _lib.FEM_PREC_FP64])
@pytest.mark.parametrize("advdiff", [False, True])
@pytest.mark.parametrize("cells,exchange", [(513, _lib.FEM_EXCHANGE_COHERENT), (514, _lib.FEM_EXCHANGE_FENCED)])
def test_largest_mesh_in_lds_and_one_past_it(gpu, cells, exchange, advdiff, precision):
    """262,144 unknowns are two rows per lane of every CU, the most that stay in
    LDS; one lattice row more streams its phases.  Against the streaming engine:
    solves to 1e-12, condition numbers below 15, two steps of two engines."""
    print("case largest in LDS", cells, advdiff, precision, flush=True)
    ctx = FEMContext(meshes.jittered_square(cells, seed=7), 0, velocity=VEL, normalize_velocity=False)
    f = np.random.default_rng(19).standard_normal(ctx.num_unknowns())
    got = []
    for engine in (_lib.FEM_ENGINE_PERSISTENT, _lib.FEM_ENGINE_STREAM):
        b = Batch([ctx], SolverOptions(precision=precision, tol=1e-12, engine=engine))
        b.set_equation(0, AdvectionDiffusionParameters(1e-4, 0.05) if advdiff else HeatParameters(1e-4, 0.05))
        b.set_state_unknowns(0, _lib.FEM_FIELD_U, f)
        if engine == _lib.FEM_ENGINE_PERSISTENT:
            assert (b.plan_info().grid, b.plan_info().exchange) == (256, exchange)
        assert b.advance(2) == _lib.FEM_OK
        got.append(b.get_state_unknowns(0))
        b.close()
    assert rel(got[0], got[1]) <= TOL
    ctx.close()


def test_autotuner_tries_the_untuned_plan(gpu):
    """300 small instances: the plan of 300 one-workgroup teams is among the
    candidates.  Within one workgroup per CU a quarter of the teams walks two
    instances, twice the time; the limit leaves half of that for the clock."""
    print("case autotune many", flush=True)
    ctx = FEMContext(meshes.jittered_square(20, seed=4), 0)
    b = Batch([ctx] * 300, SolverOptions())
    f = np.random.default_rng(20).standard_normal(ctx.num_unknowns())
    ms = []
    for rep in range(4):
        for i in range(300):
            b.set_equation(i, HeatParameters(1e-3, 0.05))
            b.set_state_unknowns(i, _lib.FEM_FIELD_U, f)
        assert b.advance(10) == _lib.FEM_OK
        ms.append(b.last_stats.ms)
    for i in range(300):
        b.set_state_unknowns(i, _lib.FEM_FIELD_U, f)
    _, best = b.autotune(10)
    assert best <= 1.5 * min(ms), (best, ms)
    b.close()
    ctx.close()


@pytest.mark.parametrize("mesh,precision,krylov,grid", [
    ((20, False), _lib.FEM_PREC_FP32_IR, _lib.FEM_KRYLOV_CG, 16), ((20, False), _lib.FEM_PREC_FP64, _lib.FEM_KRYLOV_BICGSTAB, 16),
    ((33, False), _lib.FEM_PREC_FP64, _lib.FEM_KRYLOV_CG, 16), ((34, False), _lib.FEM_PREC_FP32_IR, _lib.FEM_KRYLOV_CG, 137),
    ((24, True), _lib.FEM_PREC_FP32_IR, _lib.FEM_KRYLOV_CG, 16), ((24, True), _lib.FEM_PREC_FP64, _lib.FEM_KRYLOV_CG, 24),
    ((33, True), _lib.FEM_PREC_FP64, _lib.FEM_KRYLOV_BICGSTAB, 128)])
def test_sixteen_column_teams(gpu, mesh, precision, krylov, grid):
    """(cells - 1)^2 unknowns x 16, scattered or not: 16 workgroups while two
    rows x columns per lane suffice, 24 (also summed in one level) where the halo
    does not fit those 16 in FP64, one per 128 rows x columns beyond."""
    cells, shuffled = mesh
    print("case sixteen columns", cells, shuffled, precision, krylov, flush=True)
    m = meshes.jittered_square(cells, seed=8)
    m = scattered(m, 6) if shuffled else m
    info = check(m, False, 16, precision, krylov=krylov)
    assert (info.grid, info.exchange) == (grid, _lib.FEM_EXCHANGE_COHERENT)
    ctx = FEMContext(m, 0)
    b = np.random.default_rng(21).standard_normal((ctx.num_unknowns(), 16))
    got = [solve(gpu, ctx, fn, (1000.0, 0.05, 0.0), b, SolverOptions(precision=precision, krylov=krylov))
           for fn in ("fem_ctx_solve", "fem_ctx_solve_noalloc")]
    assert got[0][0] == got[1][0] == _lib.FEM_OK
    assert np.array_equal(got[0][1], got[1][1])
    ctx.close()


@pytest.mark.parametrize("instances,team_size,grid", [(1, 256, 256), (1, 257, 64), (2, 128, 256), (2, 129, 256)])
def test_team_size_beyond_the_device_is_the_plans_own(gpu, instances, team_size, grid):
    """128 x 128 unknowns: a request that fits is taken; beyond one workgroup per
    CU the plan is that of team_size 0 (alone the 64 workgroups of the flat
    reduction, two share all by their work) and so are the results, bit for bit."""
    print("case team size", instances, team_size, flush=True)
    ctx = FEMContext(meshes.jittered_square(129, seed=2), 0)
    f = np.random.default_rng(21).standard_normal(ctx.num_unknowns())
    got = []
    for size in (team_size, 0):
        b = Batch([ctx] * instances, SolverOptions(team_size=size, tol=1e-12))
        for i in range(instances):
            b.set_equation(i, HeatParameters(1e-3, 0.05))
            b.set_state_unknowns(i, _lib.FEM_FIELD_U, f)
        info = b.plan_info()
        if size:
            assert (info.grid, info.coresident) == (grid, 256)
        elif team_size * instances > 256:
            assert info.grid == grid
        assert b.advance(2) == _lib.FEM_OK
        got.append(b.get_state_unknowns(instances - 1))
        b.close()
    assert rel(got[0], got[1]) <= TOL
    if team_size * instances > 256:
        assert np.array_equal(got[0], got[1])
    ctx.close()
