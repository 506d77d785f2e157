"""Precomputed-matrix DG kernel where its blocks are partial: meshes of one
cell, rows that a block crosses, blocks with idle threads, every cells per
block; matvec and Chebyshev step (with and without the previous tmp) against
the oracle at the tolerances of the other operator tests."""
import numpy as np
import pytest

import oracle_bindings as ob
import sum_factorization_kernels_amd as sfk
from helpers import TOL_FP32, TOL_FP64, rel_err, to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("degree", range(1, 9))
def test_partial_blocks(cuda, degree, prec):
    import torch
    p, dtype, tol = (sfk.FP32, torch.float32, TOL_FP32) if prec == "fp32" else (sfk.FP64, torch.float64, TOL_FP64)
    for nc in ((1, 1, 1), (2, 1, 3), (7, 3, 2)):
        ij = (3.0, 5.0, 4.0)
        op = sfk.Operator(sfk.DG_PRECOMP, degree, nc, inv_jac=ij, precision=p)
        n = op.vector_size
        rng = np.random.default_rng(7300 + degree)
        real = np.float32 if prec == "fp32" else np.float64
        u, rhs, tm = (rng.standard_normal(n).astype(real).astype(np.float64) for _ in range(3))
        diag = rng.uniform(0.5, 1.5, n).astype(real).astype(np.float64)
        au = ob.dg_precomputed(degree, nc, u, inv_jac=ij)
        m = op.max_cells_per_block
        for cb in sorted({1, 2, max(1, m // 2), m} & set(range(1, m + 1))):
            op.set_schedule(cb, 1, -1)
            out = torch.full((n,), float("nan"), dtype=dtype, device="cuda")
            assert rel_err(to_np(op.apply(to_dev(u, dtype), dst=out)), au) < tol, (nc, cb)
            for c_tm in (0.0, 0.37):
                new = torch.full_like(out, float("nan"))
                d_tm = to_dev(tm, dtype) if c_tm else torch.full_like(out, float("nan"))
                op.cheby_step(to_dev(rhs, dtype), to_dev(u, dtype), to_dev(diag, dtype), new, d_tm, 0.01, c_tm)
                r_tm = c_tm * tm + 0.01 * diag * (au - rhs)
                assert rel_err(to_np(d_tm), r_tm) < tol, (nc, cb, c_tm)
                assert rel_err(to_np(new), u - r_tm) < tol, (nc, cb, c_tm)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("degree", range(1, 10))
def test_cartesian_sipg(cuda, degree, prec):
    """the Cartesian SIPG operator as a sum of Kronecker products (up to degree
    8; degree 9 is the cell kernel's) against the oracle's quadrature form, on
    anisotropic cells, cells that are their own neighbours, and every order"""
    import torch
    p, dtype, tol = (sfk.FP32, torch.float32, TOL_FP32) if prec == "fp32" else (sfk.FP64, torch.float64, TOL_FP64)
    for nc in ((1, 2, 1), (5, 3, 6)):
        ij = (3.0, 5.0, 4.0)
        op = sfk.Operator(sfk.DG_SIPG, degree, nc, inv_jac=ij, precision=p)
        n = op.vector_size
        rng = np.random.default_rng(7500 + degree)
        real = np.float32 if prec == "fp32" else np.float64
        u, rhs, tm = (rng.standard_normal(n).astype(real).astype(np.float64) for _ in range(3))
        diag = rng.uniform(0.5, 1.5, n).astype(real).astype(np.float64)
        want = ob.dg_sipg(degree, nc, ij, u)
        w_new, w_tm = ob.dg_sipg_cheby(degree, nc, ij, rhs, u, diag, tm, 0.01, 0.37)
        for order in (0, 1, 2):
            op.set_schedule(0, order, -1)
            out = torch.full((n,), float("nan"), dtype=dtype, device="cuda")
            assert rel_err(to_np(op.apply(to_dev(u, dtype), dst=out)), want) < tol, (nc, order)
            new, d_tm = torch.full_like(out, float("nan")), to_dev(tm, dtype)
            op.cheby_step(to_dev(rhs, dtype), to_dev(u, dtype), to_dev(diag, dtype), new, d_tm, 0.01, 0.37)
            assert rel_err(to_np(d_tm), w_tm) < tol and rel_err(to_np(new), w_new) < tol, (nc, order)
