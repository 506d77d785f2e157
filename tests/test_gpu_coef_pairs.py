"""Variable-coefficient apply with two right-hand sides per workgroup (low
degrees, colours that fill the chip): even and odd numbers of right-hand sides,
partial row segments, against the oracle at the tolerances of the other operator
tests; every node written (outputs start as NaN)."""
import numpy as np
import pytest

import oracle_bindings as ob
import sum_factorization_kernels_amd as sfk
from helpers import TOL_FP32, TOL_FP64, rel_err, to_dev, to_np

pytestmark = pytest.mark.gpu

NC, IJ = (22, 21, 23), (3.0, 5.0, 4.0)


@pytest.mark.parametrize("cb,n_rhs", [(1, 2), (1, 3), (3, 5), (3, 6)])
@pytest.mark.parametrize("degree,prec", [(1, "fp64"), (1, "fp32"), (2, "fp32"), (3, "fp32"), (4, "fp32")])
def test_pairs(cuda, degree, prec, cb, n_rhs):
    import torch
    p, dtype, tol = (sfk.FP32, torch.float32, TOL_FP32) if prec == "fp32" else (sfk.FP64, torch.float64, TOL_FP64)
    real = np.float32 if prec == "fp32" else np.float64
    # pairs of a colour's launch: enough for the paired kernel
    assert -(-NC[0] // cb) // 2 * (-(-NC[1] // 2)) * (-(-NC[2] // 2)) * ((n_rhs + 1) // 2) >= 1300
    op = sfk.Operator(sfk.CONT_LAPLACE, degree, NC, inv_jac=IJ, precision=p, flags=sfk.FLAG_VARIABLE_COEF, n_rhs=n_rhs)
    op.set_schedule(cb, 1, 1)
    n = op.vector_size
    rng = np.random.default_rng(7750 + degree)
    k = np.exp(0.5 * rng.standard_normal(op.n_cell_q)).astype(real).astype(np.float64)
    u = rng.standard_normal(n_rhs * n).astype(real).astype(np.float64)
    op.set_coefficient(k)
    out = to_np(op.apply(to_dev(u, dtype), dst=torch.full((n_rhs * n,), float("nan"), dtype=dtype, device="cuda")))
    for r in range(n_rhs):
        want = ob.cont_laplacian(degree, NC, IJ, u[r * n:(r + 1) * n].copy(), coef=k)
        assert rel_err(out[r * n:(r + 1) * n], want) < tol, r
