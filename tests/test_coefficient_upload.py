"""sfk_op_set_coefficient: no copy of the whole array on the host (an array that
the device cannot hold is refused by the device allocation), and the same stored
coefficient as the device setter over arrays longer than the upload's buffer."""
import os
import subprocess
import sys

import numpy as np
import pytest

import sum_factorization_kernels_amd as sfk

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ALLOC = 4  # SFK_ERR_ALLOC


@pytest.mark.parametrize("prec", [sfk.FP64, sfk.FP32])
def test_too_large_is_an_error(prec):
    """8.8e12 values: the call returns a status (in a process of its own: the C++
    exception of a host copy would end it)"""
    code = f"""
import ctypes, sys
sys.path.insert(0, {ROOT!r})
import sum_factorization_kernels_amd as sfk
op = sfk.Operator(sfk.CONT_LAPLACE, 15, (1290, 1290, 1290), inv_jac=(1.0, 1.0, 1.0), precision={prec},
                  flags=sfk.FLAG_VARIABLE_COEF)
one = (ctypes.c_double * 1)(1.0)
print("status", sfk.lib().sfk_op_set_coefficient(op.handle, one, op.n_cell_q), flush=True)
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    assert f"status {ALLOC}" in r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [sfk.FP64, sfk.FP32])
@pytest.mark.parametrize("degree,nc", [(8, (12, 12, 11)), (1, (60, 55, 43)), (15, (7, 6, 7))])
def test_equals_device_setter(cuda, degree, nc, prec):
    """FP64: the same products; FP32: the host setter rounds the product once
    where the device setter rounds coefficient, weight and product (each within
    2^-24), seen through an operator that is linear in the coefficient"""
    import torch
    from helpers import TOL_FP32, rel_err, to_dev, to_np
    dtype = torch.float32 if prec == sfk.FP32 else torch.float64
    op = sfk.Operator(sfk.CONT_LAPLACE, degree, nc, inv_jac=(1.0, 0.9, 1.2), precision=prec,
                      flags=sfk.FLAG_VARIABLE_COEF)
    assert op.n_cell_q > 1 << 20
    rng = np.random.default_rng(7800 + degree)
    k = np.exp(0.5 * rng.standard_normal(op.n_cell_q))
    u = to_dev(rng.standard_normal(op.vector_size), dtype)
    op.set_schedule(0, 1, 1)  # colored stores: a fixed order of the sums
    op.set_coefficient(k)
    host = to_np(op.apply(u))
    op.set_coefficient_device(to_dev(k, dtype))
    dev = to_np(op.apply(u))
    if prec == sfk.FP64:
        assert np.array_equal(host, dev)
    else:
        assert rel_err(host, dev) < TOL_FP32
