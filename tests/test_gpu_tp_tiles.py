"""Tensor-product kernel at the edges of its tiles: meshes that end exactly at
a tile's last cell, one cell beyond it, and one before, in x and y, with z
ranges that start above the bottom (carried state), for every tile shape,
degree and precision, and on the schedule chosen for the mesh; matvec and the
fused Chebyshev step with values on the Dirichlet nodes.  Against the oracle's
quadrature-form operator at the tolerances of the other operator tests."""
import numpy as np
import pytest

import oracle_bindings as ob
import sum_factorization_kernels_amd as sfk
from helpers import TOL_FP32, TOL_FP64, rel_err, to_dev, to_np

pytestmark = pytest.mark.gpu


def _check(op, degree, nc, ij, seed, dtype, tol):
    import torch
    n = op.vector_size
    rng = np.random.default_rng(seed)
    real = np.float32 if dtype == torch.float32 else np.float64
    u, rhs, tm = (rng.uniform(-1, 1, n).astype(real).astype(np.float64) for _ in range(3))
    diag = rng.uniform(0.5, 1.5, n).astype(real).astype(np.float64)
    au = ob.cont_laplacian(degree, nc, ij, u)
    out = torch.full((n,), float("nan"), dtype=dtype, device="cuda")
    assert rel_err(to_np(op.apply(to_dev(u, dtype), dst=out)), au) < tol
    new, d_tm = torch.full_like(out, float("nan")), to_dev(tm, dtype)
    op.cheby_step(to_dev(rhs, dtype), to_dev(u, dtype), to_dev(diag, dtype), new, d_tm, 0.8, 0.37)
    r_tm = 0.37 * tm + 0.8 * diag * (au - rhs)
    assert rel_err(to_np(d_tm), r_tm) < tol
    assert rel_err(to_np(new), u - r_tm) < tol


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("degree", range(1, 9))
def test_tile_edges(cuda, degree, prec):
    import torch
    p, dtype, tol = (sfk.FP32, torch.float32, TOL_FP32) if prec == "fp32" else (sfk.FP64, torch.float64, TOL_FP64)
    probe = sfk.Operator(sfk.CONT_LAPLACE, degree, (4, 4, 4), precision=p)
    count = probe.tile_shape(0)[0]
    for shape in range(1, count):
        _, bx, by = probe.tile_shape(shape)
        for dx, dy, zc in ((0, 0, 2), (1, 1, 1), (-1, -1, 3)):
            nc = (max(1, bx + dx), max(1, by + dy), 4)
            ij = (float(nc[0]), 2.5, 4.5)
            op = sfk.Operator(sfk.CONT_LAPLACE, degree, nc, inv_jac=ij, precision=p)
            try:
                op.set_schedule(0, 1, 2, shape, zc)
            except sfk.SfkError as e:
                assert e.status == 2 and "LDS" in str(e) and prec == "fp64"
                continue
            _check(op, degree, nc, ij, 5100 + 10 * degree + shape, dtype, tol)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("degree,nc", [(1, (65, 9, 3)), (2, (31, 5, 4)), (3, (28, 7, 5)), (4, (15, 4, 7)),
                                       (5, (10, 3, 9)), (6, (14, 5, 6)), (7, (5, 9, 4)), (8, (7, 2, 6))])
def test_default_schedule(cuda, degree, nc, prec):
    """no schedule set: the tile and z range come from the cost model"""
    import torch
    p, dtype, tol = (sfk.FP32, torch.float32, TOL_FP32) if prec == "fp32" else (sfk.FP64, torch.float64, TOL_FP64)
    ij = (float(nc[0]), 3.0, 4.0)
    op = sfk.Operator(sfk.CONT_LAPLACE, degree, nc, inv_jac=ij, precision=p)
    _, bx, by = op.tile_shape(0)
    assert (bx, by) in [op.tile_shape(s)[1:] for s in range(1, op.tile_shape(0)[0])]
    _check(op, degree, nc, ij, 5300 + degree, dtype, tol)
