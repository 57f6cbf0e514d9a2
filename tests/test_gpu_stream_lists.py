"""The streaming engine's lists of the instances still iterating (one launch up
to 1,024 instances, three beyond) and its reductions (one workgroup per sum at
16 columns): instances of uneven size and stiffness leave the lists at
different iterations.

Tolerance: every column stops at |r| <= 1e-12 |b| and the Jacobi-scaled systems
here have condition numbers below 30 (dt c / h^2 up to 1.5), so two engines'
states after two steps are within 1.2e-10 of each other."""
import numpy as np
import pytest

from femhip import AdvectionDiffusionParameters, Batch, FEMContext, HeatParameters, SolverOptions, _lib, meshes

pytestmark = pytest.mark.gpu
TOL = 1.2e-10


@pytest.mark.parametrize("count,cells,k,advdiff", [
    (2, (5, 90), 16, True), (2, (5, 90), 16, False), (2, (5, 90), 4, True), (7, (3, 40, 66), 16, True),
    (256, (3, 6), 1, False), (257, (3, 6), 1, True), (1024, (3, 5), 1, False), (1025, (3, 5), 1, False)])
@pytest.mark.parametrize("precision", [_lib.FEM_PREC_FP32_IR, _lib.FEM_PREC_FP64])
def test_lists_and_reductions(gpu, count, cells, k, advdiff, precision):
    print("case stream lists", count, cells, k, advdiff, precision, flush=True)
    ctxs = {c: FEMContext(meshes.jittered_square(c, seed=c), 0, velocity=(0.5, 0.3, 0.0), normalize_velocity=False)
            for c in cells}
    use = [cells[i % len(cells)] for i in range(count)]
    prm = AdvectionDiffusionParameters if advdiff else HeatParameters
    got = []
    for eng in (_lib.FEM_ENGINE_STREAM, _lib.FEM_ENGINE_PERSISTENT):
        rng = np.random.default_rng(9)
        b = Batch([ctxs[c] for c in use], SolverOptions(nrhs=k, engine=eng, precision=precision, tol=1e-12,
                                                        max_iters=1000,  # the default, 2 n, is 8 for 4 unknowns
                                                        krylov=_lib.FEM_KRYLOV_BICGSTAB if advdiff else 0))
        for i, c in enumerate(use):
            b.set_equation(i, prm(1e-3, 1.5 / (1e-3 * c * c) * 10.0 ** -(i % 4)))
            b.set_state_unknowns(i, _lib.FEM_FIELD_U, rng.standard_normal(((c - 1) ** 2, k)))
        assert b.advance(2) == _lib.FEM_OK
        got.append([b.get_state_unknowns(i).reshape(-1, k) for i in range(count)])
        b.close()
    for i, (x, y) in enumerate(zip(*got)):
        assert np.linalg.norm(x - y) <= TOL * np.linalg.norm(y), i


def two_engines(m, bc, prm, k, n, **opts):
    """The state after two steps, on the streaming and on the persistent engine."""
    ctx = FEMContext(m, bc, velocity=(0.5, 0.3, 0.0), normalize_velocity=False)
    f = np.random.default_rng(10).standard_normal((n, k))
    got = []
    for eng in (_lib.FEM_ENGINE_STREAM, _lib.FEM_ENGINE_PERSISTENT):
        b = Batch([ctx], SolverOptions(nrhs=k, engine=eng, tol=1e-12, max_iters=1000, **opts))
        b.set_equation(0, prm)
        b.set_state_unknowns(0, _lib.FEM_FIELD_U, f)
        assert b.advance(2) == _lib.FEM_OK
        got.append(b.get_state_unknowns(0).reshape(-1, k))
        b.close()
    ctx.close()
    return got


@pytest.mark.parametrize("k,krylov", [(1, 1), (1, 2), (1, 3), (4, 1), (16, 2), (16, 3)])
@pytest.mark.parametrize("precision", [_lib.FEM_PREC_FP32_IR, _lib.FEM_PREC_FP64])
def test_stage_edges(gpu, k, krylov, precision):
    """Row blocks staged in 16-byte pieces from an aligned start: entry counts
    of every remainder by 4, one block and several."""
    rest = set()
    for cells, held in ((4, 0), (5, 0), (5, 1), (6, 2), (7, 1), (8, 3), (20, 1), (21, 0), (34, 2), (35, 1)):
        print("case stream stage", k, krylov, precision, cells, held, flush=True)
        m = meshes.jittered_square(cells, seed=cells)
        m["on_boundary"][np.flatnonzero(m["on_boundary"] == 0)[:held]] = 1  # held vertices change the remainder
        ctx = FEMContext(m, 0)
        n = ctx.info().num_unknowns
        rest.add(ctx.info().nnz % 4)
        ctx.close()
        c = 1.5 / (1e-3 * cells * cells)
        prm = AdvectionDiffusionParameters(1e-3, c) if krylov == _lib.FEM_KRYLOV_BICGSTAB else HeatParameters(1e-3, c)
        x, y = two_engines(m, 0, prm, k, n, krylov=krylov, precision=precision)
        assert np.linalg.norm(x - y) <= TOL * np.linalg.norm(y), cells
    assert rest == {0, 1, 2, 3}


def test_longest_row_that_fits(gpu):
    """A hub whose FP64 row of 5,074 entries fills the stage's limit (61,936
    bytes: 12 an entry and 1,040 for the block's rows) from an unaligned start,
    so the aligned one's slack comes on top; one entry more is refused."""
    def fan(d):
        t = 2 * np.pi * np.arange(d) / d
        xyz = np.concatenate([[[3, 0, 0], [4, 0, 0], [3, 1, 0], [0, 0, 0.5]],
                              np.stack([np.cos(t), np.sin(t), 0 * t], 1)]).astype(np.float32)
        tri = np.concatenate([[[0, 1, 2]], np.stack([np.full(d, 3), 4 + np.arange(d), 4 + (np.arange(d) + 1) % d], 1)])
        return {"xyz": xyz, "tri": tri.astype(np.uint32), "on_boundary": np.zeros(d + 4, np.uint8)}

    print("case stream longest row", flush=True)
    prm = HeatParameters(1e-3, 1e-3)
    x, y = two_engines(fan(5073), 1, prm, 1, 5077, precision=_lib.FEM_PREC_FP64)
    assert np.linalg.norm(x - y) <= TOL * np.linalg.norm(y)
    print("case stream row refused", flush=True)
    b = Batch([FEMContext(fan(5074), 1)], SolverOptions(engine=_lib.FEM_ENGINE_STREAM, precision=_lib.FEM_PREC_FP64))
    b.set_equation(0, prm)
    with pytest.raises(_lib.FemError, match="too many nonzeros"):
        b.advance(1)
    b.close()
