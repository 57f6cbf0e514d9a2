"""Device memory that a launch plan takes."""
import numpy as np
import pytest

from femhip import Batch, FEMContext, HeatParameters, SolverOptions, _lib, meshes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,krylov,words", [(16, _lib.FEM_KRYLOV_CG, False), (1, _lib.FEM_KRYLOV_CG_CLASSIC, False),
                                            (1, _lib.FEM_KRYLOV_CG, True)])
def test_exchange_words_only_where_rows_stay_in_lds(gpu, k, krylov, words):
    """482 x 482 unknowns: the first advance takes the guess, the right-hand side
    and the history part (3 FP64 vectors), and 32 bytes per unknown and column of
    exchange words only if the teams use them.  At 16 columns the rows do not
    fit; classic CG has no form that keeps them.  Everything else (plan tables,
    halo tables of 10 entries at 2 bytes and at most 10 halo rows at 4 bytes per
    row, allocations rounded to 2 MiB) is below 24 MB at one column and 12 MB
    without halos."""
    import torch
    print("case plan memory", k, krylov, words, flush=True)
    warm = FEMContext(meshes.jittered_square(9, seed=1), 0)  # the code objects are loaded with the first plan
    w = Batch([warm], SolverOptions(nrhs=k, krylov=krylov, team_size=2))
    w.set_equation(0, HeatParameters(1e-3, 1e-3))
    assert w.advance(1) == _lib.FEM_OK
    w.close()
    warm.close()
    ctx = FEMContext(meshes.jittered_square(483, seed=1), 0)
    n = ctx.num_unknowns()
    b = Batch([ctx], SolverOptions(nrhs=k, krylov=krylov))
    b.set_equation(0, HeatParameters(1e-3, 1e-3))
    b.set_state_unknowns(0, _lib.FEM_FIELD_U, np.zeros((n, k)))
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    b.plan_info()
    took = free - torch.cuda.mem_get_info()[0]
    vectors, xch = 3 * 8 * n * k, 32 * n * k
    assert vectors <= took <= vectors + ((xch + 24e6) if words else 12e6), (took, vectors, xch)
    b.close()
    ctx.close()
