"""The plan rules of the persistent engine at the sizes where they change.

Tolerances as in test_gpu_team_rows (solves to 1e-12 of systems with condition
numbers below 10, 3 steps, against the oracle)."""
import pytest

from femhip import _lib, meshes
from test_gpu_team_rows import check

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
