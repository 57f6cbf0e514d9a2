"""The column-scaled matrix is held by the streaming engine only."""
import numpy as np
import pytest

from femhip import Batch, FEMContext, HeatParameters, SolverOptions, _lib, meshes

pytestmark = pytest.mark.gpu


def test_persistent_solver_does_not_hold_it(gpu):
    """1401 x 1401 nodes: a solver that has its state and matrix holds the FP64
    and the inner matrix (12 bytes per entry) and, per row, both forms of the
    inverse diagonal (12 bytes), 5 FP64 and 11 inner vectors (84) and the surface
    values (4), in at most 14 allocations rounded to 2 MiB.  The column-scaled
    matrix would take 4 bytes for each of about 7 entries per row more."""
    import torch
    print("case solver memory", flush=True)
    ctx = FEMContext(meshes.jittered_square(1401, seed=1), 0)
    n, nnz = ctx.num_unknowns(), ctx.info().nnz
    assert 4 * nnz > 14 * 2**21 + 20e6
    solvers = []
    for _ in range(2):  # the first one has the context assembled
        free = torch.cuda.mem_get_info()[0]
        b = Batch([ctx], SolverOptions(predictor=_lib.FEM_PREDICTOR_LINEAR))  # keeps no history vectors
        b.set_equation(0, HeatParameters(1e-3, 1e-3))
        b.set_state_unknowns(0, _lib.FEM_FIELD_U, np.zeros((n, 1)))
        torch.cuda.synchronize()
        took = free - torch.cuda.mem_get_info()[0]
        solvers.append(b)
    assert took <= 12 * nnz + (12 + 84 + 4 + 1) * n + 14 * 2**21, (took, n, nnz)
    for b in solvers:
        b.close()
    ctx.close()


@pytest.mark.parametrize("k", [1, 4])
def test_streaming_after_new_values(gpu, k):
    """The streaming engine's matrix follows new coefficients, also after a first
    advance: the state equals that of a solver made with them."""
    print("case streaming values", k, flush=True)
    ctx = FEMContext(meshes.jittered_square(40, seed=2), 0)
    n = ctx.num_unknowns()
    u = np.cos(np.arange(n * k, dtype=float)).reshape(n, k)

    def made(first):
        b = Batch([ctx], SolverOptions(nrhs=k, engine=_lib.FEM_ENGINE_STREAM, predictor=_lib.FEM_PREDICTOR_PREVIOUS))
        if first:
            b.set_equation(0, HeatParameters(1e-3, 1e-3))
            b.set_state_unknowns(0, _lib.FEM_FIELD_U, u)
            assert b.advance(1) == _lib.FEM_OK
        b.set_equation(0, HeatParameters(2e-3, 5e-3))
        b.set_state_unknowns(0, _lib.FEM_FIELD_U, u)
        assert b.advance(2) == _lib.FEM_OK
        got = b.get_state_unknowns(0, _lib.FEM_FIELD_U)
        b.close()
        return got

    assert np.array_equal(made(True), made(False))
    ctx.close()
