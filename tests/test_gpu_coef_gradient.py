"""Coefficient gradient of the continuous Laplacian at the degrees around which
the kernel loads the next pair ahead or not, one pair and several, against the
oracle at the tolerances of the other operator tests."""
import numpy as np
import pytest

import oracle_bindings as ob
import sum_factorization_kernels_amd as sfk
from helpers import TOL_FP32, TOL_FP64, rel_err, to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_rhs", [1, 3])
@pytest.mark.parametrize("degree,prec", [(10, "fp64"), (11, "fp64"), (12, "fp64"), (13, "fp64"), (14, "fp64"),
                                         (12, "fp32")])
def test_high_degree_gradient(cuda, degree, prec, n_rhs):
    import torch
    p, dtype, tol = (sfk.FP32, torch.float32, TOL_FP32) if prec == "fp32" else (sfk.FP64, torch.float64, TOL_FP64)
    real = np.float32 if prec == "fp32" else np.float64
    nc, ij = (3, 2, 2), (3.0, 5.0, 4.0)
    op = sfk.Operator(sfk.CONT_LAPLACE, degree, nc, inv_jac=ij, precision=p, flags=sfk.FLAG_VARIABLE_COEF, n_rhs=n_rhs)
    rng = np.random.default_rng(8600 + degree)
    u, lam = (rng.standard_normal(n_rhs * op.vector_size).astype(real).astype(np.float64) for _ in range(2))
    g = to_np(op.grad_coefficient(to_dev(u, dtype), to_dev(lam, dtype)))
    assert rel_err(g, ob.cont_laplacian_coef_grad(degree, nc, ij, u, lam, n_rhs=n_rhs)) < tol
