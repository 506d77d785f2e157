"""Variable-coefficient kernels of the continuous Laplacian where they can go
wrong: an odd right-hand side left over from a pair, meshes of one cell, odd
meshes (colours of unequal size, partial blocks), both scatters, every cells
per workgroup; apply, coefficient gradient and diagonal, the coefficient set
from the host and from the device."""
import numpy as np
import pytest

import dense_assembly as da
import oracle_bindings as ob
import sum_factorization_kernels_amd as sfk
from helpers import TOL_FP32, TOL_FP64, rel_err, to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("degree", range(1, 9))
def test_coefficient_kernels(cuda, degree, prec):
    import torch
    p, dtype, tol = (sfk.FP32, torch.float32, TOL_FP32) if prec == "fp32" else (sfk.FP64, torch.float64, TOL_FP64)
    real = np.float32 if prec == "fp32" else np.float64
    ij = (3.0, 5.0, 4.0)
    for nc, n_rhs in (((1, 1, 1), 1), ((2, 1, 3), 2), ((7, 3, 2), 3)):
        op = sfk.Operator(sfk.CONT_LAPLACE, degree, nc, inv_jac=ij, precision=p, flags=sfk.FLAG_VARIABLE_COEF,
                          n_rhs=n_rhs)
        n = op.vector_size
        rng = np.random.default_rng(7700 + degree)
        k = np.exp(0.5 * rng.standard_normal(op.n_cell_q)).astype(real).astype(np.float64)
        u, lam = (rng.standard_normal(n_rhs * n).astype(real).astype(np.float64) for _ in range(2))
        want = np.concatenate([ob.cont_laplacian(degree, nc, ij, u[r * n:(r + 1) * n].copy(), coef=k)
                               for r in range(n_rhs)])
        for host in (True, False):
            op.set_coefficient(k) if host else op.set_coefficient_device(to_dev(k, dtype))
            for scatter in (0, 1):
                for cb in sorted({1, 2, op.max_cells_per_block} & set(range(1, op.max_cells_per_block + 1))):
                    op.set_schedule(cb, 1, scatter)
                    out = torch.full((n_rhs * n,), float("nan"), dtype=dtype, device="cuda")
                    assert rel_err(to_np(op.apply(to_dev(u, dtype), dst=out)), want) < tol, (nc, host, scatter, cb)
        g = to_np(op.grad_coefficient(to_dev(u, dtype), to_dev(lam, dtype)))
        assert rel_err(g, ob.cont_laplacian_coef_grad(degree, nc, ij, u, lam, n_rhs=n_rhs)) < tol, nc
        if degree <= 3 and nc == (2, 1, 3):
            dense = da.cont_laplacian_dense(degree, nc, ij, coef=k)
            assert rel_err(to_np(op.diagonal()), np.diag(dense)) < tol, nc
