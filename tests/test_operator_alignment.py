"""Operator products on vectors aligned to their value type alone (an offset view
of a tensor): no access to x or y may assume more."""
import os
import re
import subprocess

import numpy as np
import pytest

from femhip import FEMContext, Operator, _lib, build, meshes


def test_vector_accesses_assume_the_type_alone(tmp_path):
    """Read from the compiler's IR of the variants whose matrix loads are marked
    non-temporal: every other vector load and every vector store is one of x or y."""
    out = tmp_path / "operator.ll"
    cmd = [build._hipcc(), *build.HIPCC_FLAGS, f"-I{build.INCLUDE}", f"-I{build.CSRC}", "--cuda-device-only", "-emit-llvm",
           "-S", os.path.join(build.CSRC, "operator.hip"), "-o", str(out)]
    subprocess.run(cmd, check=True, capture_output=True)
    bodies = {m[1]: m[2] for m in re.finditer(r"^define [^@\n]*@(\w+)\([^\n]*\n(.*?)^}", out.read_text(), re.M | re.S)}
    bodies = {n: b for n, b in bodies.items() if re.search(r"k_spmv_(stream|pipe)I[fd]Li\d+ELb1E", n)}
    assert len(bodies) == 16
    seen = 0
    for name, body in bodies.items():
        for op, ty, rest in re.findall(r"\b(load|store) <\d+ x (float|double)>([^\n]*ptr addrspace\(1\)[^\n]*)", body):
            if op == "load" and "nontemporal" in rest:
                continue  # the matrix
            seen += 1
            align = int(re.search(r"align (\d+)", rest)[1])
            assert align <= {"float": 4, "double": 8}[ty], (name, op, rest)
    assert seen


@pytest.mark.gpu
@pytest.mark.parametrize("schedule", [None, _lib.FEM_SPMV_STREAM, _lib.FEM_SPMV_STREAM_NT, _lib.FEM_SPMV_PIPE,
                                      _lib.FEM_SPMV_PIPE_NT])
@pytest.mark.parametrize("precision", [_lib.FEM_PREC_FP64, _lib.FEM_PREC_FP32_IR])
@pytest.mark.parametrize("k", [1, 2, 4, 16])
def test_shifted_vectors(gpu, k, precision, schedule):
    """x or y one to three values past an aligned address: the products of the
    aligned vectors, bit for bit."""
    import torch
    print("case operator shift", k, precision, schedule, flush=True)
    ctx = FEMContext(meshes.jittered_square(23, seed=8), 0)
    n = ctx.num_unknowns()
    dt = torch.float64 if precision == _lib.FEM_PREC_FP64 else torch.float32
    op = Operator(ctx, (500.0, 1.0, -1.0), precision)
    if schedule is not None:
        op.set_schedule(k, schedule)
    buf = torch.zeros(2, n * k + 4, dtype=dt, device="cuda")
    x = torch.from_numpy(np.random.default_rng(14).standard_normal(n * k)).to(dt)
    want = None
    for sx, sy in ((0, 0), (1, 0), (0, 1), (2, 3), (3, 2)):
        xd, yd = buf[0, sx:sx + n * k], buf[1, sy:sy + n * k]
        xd.copy_(x)
        yd.zero_()
        torch.cuda.synchronize()
        op.apply_device(k, xd.data_ptr(), yd.data_ptr())
        torch.cuda.synchronize()
        got = yd.cpu()
        want = got if want is None else want
        assert torch.equal(got, want), (sx, sy)
    op.close()
    ctx.close()
