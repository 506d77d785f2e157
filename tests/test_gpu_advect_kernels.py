"""Advection kernels where they can go wrong: cells that are their own
neighbours, rows that a workgroup crosses once or several times, partial
workgroups, slabs of fewer layers, every order, velocities of both signs and
zero; apply, fused stage, transpose and velocity gradient against the oracle."""
import numpy as np
import pytest

import oracle_bindings as ob
import sum_factorization_kernels_amd as sfk
from helpers import TOL_FP32, TOL_FP64, rel_err, to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("degree", range(1, 10))
def test_advection_kernels(cuda, degree, prec):
    import torch
    p, dtype, tol = (sfk.FP32, torch.float32, TOL_FP32) if prec == "fp32" else (sfk.FP64, torch.float64, TOL_FP64)
    real = np.float32 if prec == "fp32" else np.float64
    ij = (3.0, 5.0, 4.0)
    for nc in ((1, 1, 1), (2, 1, 3), (19, 3, 6) if degree < 5 else (5, 2, 6)):
        op = sfk.Operator(sfk.DG_ADVECT, degree, nc, inv_jac=ij, precision=p, flags=sfk.FLAG_VARIABLE_VELOCITY)
        n = op.vector_size
        rng = np.random.default_rng(7900 + degree)
        values = lambda k: rng.standard_normal(k).astype(real).astype(np.float64)
        cv, fv, u, w, upd = values(3 * op.n_cell_q), values(3 * op.n_face_q), values(n), values(n), values(n)
        fv[rng.random(fv.size) < 0.1] = 0.0
        op.set_velocity(cv, fv)
        au = ob.dg_advect_var(degree, nc, ij, cv, fv, u)
        atw = ob.dg_advect_var_transpose(degree, nc, ij, cv, fv, w)
        rc, rf = ob.dg_advect_velocity_grad(degree, nc, ij, fv, u, w)
        for order in (0, 1, 2):
            op.set_schedule(0, order, -1)
            out = torch.full((n,), float("nan"), dtype=dtype, device="cuda")
            assert rel_err(to_np(op.apply(to_dev(u, dtype), dst=out)), au) < tol, (nc, order)
            out.fill_(float("nan"))
            assert rel_err(to_np(op.apply_transpose(to_dev(w, dtype), dst=out)), atw) < tol, (nc, order)
            tm = torch.full_like(out, float("nan"))
            op.rk_stage(to_dev(u, dtype), to_dev(upd, dtype), out, tm, 0.3, 0.2)
            assert rel_err(to_np(out), upd + 0.3 * au) < tol, (nc, order)
            assert rel_err(to_np(tm), upd + 0.5 * au) < tol, (nc, order)
            gc, gf = op.grad_velocity(to_dev(u, dtype), to_dev(w, dtype))
            assert rel_err(to_np(gc), rc) < tol and rel_err(to_np(gf), rf) < tol, (nc, order)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("degree", range(1, 10))
def test_velocity_passes(cuda, degree, prec):
    """the passes that read the caller's velocity and store it into the
    operator: their results, and those of the operator afterwards"""
    import torch
    p, dtype, tol = (sfk.FP32, torch.float32, TOL_FP32) if prec == "fp32" else (sfk.FP64, torch.float64, TOL_FP64)
    real = np.float32 if prec == "fp32" else np.float64
    ij = (3.0, 5.0, 4.0)
    for nc in ((1, 1, 1), (2, 1, 3), (19, 3, 6) if degree < 5 else (5, 2, 6)):
        op = sfk.Operator(sfk.DG_ADVECT, degree, nc, inv_jac=ij, precision=p, flags=sfk.FLAG_VARIABLE_VELOCITY)
        n = op.vector_size
        rng = np.random.default_rng(8100 + degree)
        values = lambda k: rng.standard_normal(k).astype(real).astype(np.float64)
        u, w = values(n), values(n)
        for order in (0, 2):
            op.set_schedule(0, order, -1)
            cv, fv = values(3 * op.n_cell_q), values(3 * op.n_face_q)
            fv[rng.random(fv.size) < 0.1] = 0.0
            au = ob.dg_advect_var(degree, nc, ij, cv, fv, u)
            atw = ob.dg_advect_var_transpose(degree, nc, ij, cv, fv, w)
            want = (atw, *ob.dg_advect_velocity_grad(degree, nc, ij, fv, u, w))
            dev = [to_dev(x, dtype) for x in (u, w, cv, fv)]
            assert rel_err(to_np(op.advect_forward(dev[0], *dev[2:])), au) < tol, (nc, order)
            assert rel_err(to_np(op.apply(dev[0])), au) < tol, (nc, order)
            other = sfk.Operator(sfk.DG_ADVECT, degree, nc, inv_jac=ij, precision=p, flags=sfk.FLAG_VARIABLE_VELOCITY)
            other.set_schedule(0, order, -1)
            for got, ref in zip(other.advect_backward(*dev), want):
                assert rel_err(to_np(got), ref) < tol, (nc, order)
            # bit for bit the velocity that was passed
            assert torch.equal(other.apply(dev[0]), op.apply(dev[0])), (nc, order)
