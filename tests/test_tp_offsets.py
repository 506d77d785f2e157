"""Largest meshes of the tensor-product kernel: its 32-bit line offsets stay
below the buffer range (CPU, the header the kernel uses), and its results there
equal the cell kernel's (GPU)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "sum_factorization_kernels_amd", "csrc")


def test_line_offsets_in_range(tmp_path):
    exe = str(tmp_path / "tp_offsets_check")
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I" + CSRC,
                        os.path.join(ROOT, "tests", "cpp", "tp_offsets_check.cc"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("degree,nc", [(4, (1831, 1832, 2)), (8, (682, 683, 2))])
def test_largest_planes(cuda, degree, nc):
    """planes whose p + 1 hold just below 2^31 bytes, against the colored cell
    kernel (64-bit addresses): both are within TOL_FP64 of the operator"""
    import torch
    import sum_factorization_kernels_amd as sfk
    from helpers import TOL_FP64
    gx, gy = (c * degree + 1 for c in nc[:2])
    es = 8
    size = (degree + 1) * gx * gy * es
    assert 2 ** 31 - (degree - 1) * gx * es < size < 2 ** 31
    op = sfk.Operator(sfk.CONT_LAPLACE, degree, nc, inv_jac=(1.0, 0.9, 1.2))
    u = torch.rand(op.vector_size, dtype=torch.float64, device="cuda",
                   generator=torch.Generator("cuda").manual_seed(degree)) - 0.5
    got = op.apply(u, dst=torch.full_like(u, float("nan")))
    op.set_schedule(0, 1, 1)
    got -= op.apply(u)
    scale = float(op.apply(u).abs_().max())
    assert float(got.abs_().max()) <= 2 * TOL_FP64 * scale
