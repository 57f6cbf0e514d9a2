"""A launch plan loads the stepping kernel's variant that it runs, not the others."""
import os
import subprocess
import sys

import pytest

from femhip import Batch, FEMContext, HeatParameters, SolverOptions, _lib, meshes
from test_gpu_team_plans import fan_square

pytestmark = pytest.mark.gpu

CHILD = """
import sys, time
sys.path[:0] = [{tests!r}]
import conftest
from femhip import Batch, FEMContext, HeatParameters, SolverOptions, _lib, meshes
ctx = {{c: FEMContext(meshes.jittered_square(c, seed=1), 0) for c in (20, 60)}}
for name, cells, exchange in (("coherent", 60, 1), ("fenced", 60, 2), ("alone", 20, 0)):
    ms = []
    for again in range(3):
        b = Batch([ctx[cells]], SolverOptions(exchange=exchange))
        b.set_equation(0, HeatParameters(1e-3, 0.05))
        t = time.perf_counter()
        assert b.plan_info().exchange == exchange
        ms.append(1e3 * (time.perf_counter() - t))
        b.close()
    print(name, *ms, flush=True)
"""


def test_first_plan_of_each_variant_loads_it(gpu):
    """In a process of its own: a variant's code object takes 2 ms and more to
    load, a plan without that 0.3 at most, so the first plan in each exchange
    mode takes three times as long as the next two.  With all variants loaded by
    the very first plan the others' first would take as long as the next."""
    print("case plan loads", flush=True)
    tests = os.path.dirname(os.path.abspath(__file__))
    r = subprocess.run([sys.executable, "-c", CHILD.format(tests=tests)], capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr[-2000:], flush=True)
    assert r.returncode == 0
    rows = [line.split() for line in r.stdout.splitlines()]
    assert [x[0] for x in rows] == ["coherent", "fenced", "alone"]
    for x in rows:
        first, *more = map(float, x[1:])
        assert first > 3 * min(more), x


@pytest.mark.parametrize("k", [1, 2, 4, 16])
@pytest.mark.parametrize("precision", [_lib.FEM_PREC_FP32_IR, _lib.FEM_PREC_FP64])
@pytest.mark.parametrize("krylov", [_lib.FEM_KRYLOV_CG, _lib.FEM_KRYLOV_BICGSTAB, _lib.FEM_KRYLOV_CG_CLASSIC])
def test_every_variant_holds_what_plans_are_sized_within(gpu, k, precision, krylov):
    """One workgroup per CU with teams of several and two of one-workgroup teams,
    with rows in LDS and without (a row of more than 10 entries)."""
    print("case variant holds", k, precision, krylov, flush=True)
    small, large = (FEMContext(meshes.jittered_square(c, seed=1), 0) for c in (4, 60))
    long_row = FEMContext(fan_square(20, 3), 0)
    for ctx, team, exchange, blocks in ((small, 1, 0, 512), (long_row, 1, 0, 512), (large, 256, 1, 256), (large, 256, 2, 256),
                                        (long_row, 2, 1, 256), (long_row, 2, 2, 256)):
        b = Batch([ctx], SolverOptions(nrhs=k, precision=precision, krylov=krylov, team_size=team, exchange=exchange))
        b.set_equation(0, HeatParameters(1e-3, 0.05))
        info = b.plan_info()
        assert (info.exchange, info.coresident) == (exchange, blocks)
        b.close()
    for c in (small, large, long_row):
        c.close()
