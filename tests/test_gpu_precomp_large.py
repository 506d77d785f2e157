"""Precomputed-matrix DG and Cartesian SIPG on vectors beyond the sizes at which
the kernels change how they read and write them: the field of a small periodic
mesh repeated over a large one (block and row ends anywhere, a partial last
block), whose result is the oracle's on the small mesh, repeated.  Tolerances
of the other operator tests."""
import numpy as np
import pytest

import oracle_bindings as ob
import sum_factorization_kernels_amd as sfk
from helpers import TOL_FP32, TOL_FP64, to_dev

pytestmark = pytest.mark.gpu

SMALL = (7, 3, 5)


def _repeat(v, n, times):
    """a canonical vector of SMALL, `times` meshes of it in x, y, z"""
    nx, ny, nz = SMALL
    return v.reshape(nz, ny, nx, n ** 3).repeat(times[2], times[1], times[0], 1).reshape(-1)


def _err(got, want):
    return float((got - want).abs().max() / want.abs().max())


@pytest.mark.parametrize("kind", ["precomp", "cart"])
@pytest.mark.parametrize("degree,prec,bytes_", [(1, "fp64", 104 << 20), (2, "fp64", 104 << 20), (2, "fp32", 104 << 20),
                                                (4, "fp32", 104 << 20), (5, "fp32", 104 << 20), (4, "fp64", 104 << 20)])
def test_large_vectors(cuda, kind, degree, prec, bytes_):
    import torch
    p, dtype, tol = (sfk.FP32, torch.float32, TOL_FP32) if prec == "fp32" else (sfk.FP64, torch.float64, TOL_FP64)
    real = np.float32 if prec == "fp32" else np.float64
    n, ij = degree + 1, (3.0, 5.0, 4.0)
    cells = bytes_ // (np.dtype(real).itemsize * n ** 3)
    times = [11, 23, 0]
    times[2] = cells // (np.prod(SMALL) * 11 * 23) + 1
    rng = np.random.default_rng(7900 + degree)
    size = int(np.prod(SMALL)) * n ** 3
    u, rhs, tm = (rng.standard_normal(size).astype(real).astype(np.float64) for _ in range(3))
    diag = rng.uniform(0.5, 1.5, size).astype(real).astype(np.float64)
    if kind == "precomp":
        au = ob.dg_precomputed(degree, SMALL, u, inv_jac=ij)
    else:
        au = ob.dg_sipg(degree, SMALL, ij, u)
    nc = tuple(a * b for a, b in zip(SMALL, times))
    op = sfk.Operator(sfk.DG_PRECOMP if kind == "precomp" else sfk.DG_SIPG, degree, nc, inv_jac=ij, precision=p)
    d_u = _repeat(to_dev(u, dtype), n, times)
    assert d_u.numel() * d_u.element_size() >= bytes_
    got = op.apply(d_u, dst=torch.full_like(d_u, float("nan")))
    assert _err(got, _repeat(to_dev(au, dtype), n, times)) < tol
    r_tm = 0.37 * tm + 0.01 * diag * (au - rhs)
    d_tm = _repeat(to_dev(tm, dtype), n, times)
    new = torch.full_like(d_u, float("nan"))
    op.cheby_step(_repeat(to_dev(rhs, dtype), n, times), d_u, _repeat(to_dev(diag, dtype), n, times), new, d_tm, 0.01,
                  0.37)
    assert _err(d_tm, _repeat(to_dev(r_tm, dtype), n, times)) < tol
    assert _err(new, _repeat(to_dev(u - r_tm, dtype), n, times)) < tol
