"""Element coefficients handed to fem_ctx_assemble in device memory: the matrices
of the same values in host memory, bit for bit (one kernel assembles both)."""
import ctypes as C

import numpy as np
import pytest

from femhip import FEMContext, _lib, meshes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kappa,velocity", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("bc", [0, 1])
def test_device_coefficients(gpu, bc, kappa, velocity):
    """The buffers are overwritten after the call: what it needs of them it has read."""
    import torch
    print("case device coefficients", bc, kappa, velocity, flush=True)
    m = meshes.jittered_square(33, seed=9)
    rng = np.random.default_rng(15)
    k, v = rng.uniform(0.5, 2.0, len(m["tri"])), rng.standard_normal((len(m["tri"]), 3))
    want = FEMContext(m, bc, velocity_e=v if velocity else None, normalize_velocity=False, kappa_e=k if kappa else None)
    got = FEMContext(m, bc)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        kd, vd = (2.0 * torch.from_numpy(0.5 * a).to("cuda") for a in (k, v))
    side.synchronize()  # the coefficients are complete
    p = _lib.fem_assembly_params()
    p.velocity[0], p.normalize_velocity = 1.0, 0
    if kappa:
        p.kappa_e = C.cast(C.c_void_p(kd.data_ptr()), C.POINTER(C.c_double))
    if velocity:
        p.velocity_e = C.cast(C.c_void_p(vd.data_ptr()), C.POINTER(C.c_double))
    _lib.check(gpu.fem_ctx_assemble(got.handle, C.byref(p)))
    kd.fill_(float("nan"))
    vd.fill_(float("nan"))
    torch.cuda.synchronize()
    for which in (_lib.FEM_MATRIX_M, _lib.FEM_MATRIX_K, _lib.FEM_MATRIX_A):
        assert np.array_equal(want.matrix(which), got.matrix(which))
    want.close()
    got.close()
