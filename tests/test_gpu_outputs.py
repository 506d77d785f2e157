"""Outputs that the wrappers allocate hold nothing but what the call wrote: each
call gets back memory that was filled with NaN."""
import pytest

import sum_factorization_kernels_amd as sfk

pytestmark = pytest.mark.gpu

KINDS = {
    "cell": (sfk.CELL_LAPLACE, {}),
    "cont": (sfk.CONT_LAPLACE, {}),
    "coef": (sfk.CONT_LAPLACE, {"flags": sfk.FLAG_VARIABLE_COEF, "n_rhs": 3}),
    "sipg": (sfk.DG_SIPG, {}),
    "refx": (sfk.DG_SIPG, {"flags": sfk.FLAG_REF_X_SWEEP}),
    "perq": (sfk.DG_SIPG, {"geometry": sfk.GEOM_PER_Q}),
    "advect": (sfk.DG_ADVECT, {"flags": sfk.FLAG_VARIABLE_VELOCITY}),
    "precomp": (sfk.DG_PRECOMP, {}),
}


@pytest.mark.parametrize("prec", [sfk.FP64, sfk.FP32])
@pytest.mark.parametrize("degree", [1, 3, 4, 9])
@pytest.mark.parametrize("kind", sorted(KINDS))
def test_outputs_are_written(cuda, kind, degree, prec):
    import torch
    k, more = KINDS[kind]
    if kind == "precomp" and degree == 9:
        degree = 8
    nc = (5, 3, 4)
    op = sfk.Operator(k, degree, nc, inv_jac=(5.0, 3.0, 4.0), precision=prec, **more)
    g = torch.Generator("cuda").manual_seed(11)
    rand = lambda n: torch.rand(n, dtype=torch.float64, device="cuda", generator=g).to(op.dtype) + 0.5
    if kind == "perq":
        op.set_sine_deformation(0.05)
    if kind == "coef":
        op.set_coefficient_device(rand(op.n_cell_q))
    vel = (rand(3 * op.n_cell_q), rand(3 * op.n_face_q)) if kind == "advect" else None
    if vel:
        op.set_velocity_device(*vel)
    n = op.vector_size * op.n_rhs
    u, w = rand(n) - 1.0, rand(n) - 1.0
    calls = [lambda: (op.apply(u),)]
    if kind != "refx":
        calls.append(lambda: (op.apply_transpose(u),))
    if kind == "coef":
        calls.append(lambda: (op.grad_coefficient(u, w),))
    if kind == "advect":
        calls += [lambda: op.grad_velocity(u, w), lambda: (op.advect_forward(u, *vel),),
                  lambda: op.advect_backward(u, w, *vel)]
    if kind == "cont" and degree <= 8:
        calls += [lambda d=d: (op.cheby_precondition(u, d, 0.1, 2.5),) for d in (2, 3, 6, 7)]
    for call in calls:
        first = call()
        want = [x.clone() for x in first]
        for x in first:
            x.fill_(float("nan"))
        del first, x
        junk = [torch.full((v.numel(),), float("nan"), dtype=op.dtype, device="cuda") for v in want for _ in range(3)]
        del junk
        for got, ref in zip(call(), want):
            assert torch.isfinite(got).all()
            assert (got - ref).abs().max() <= (1e-12 if prec == sfk.FP64 else 1e-5) * ref.abs().max()
