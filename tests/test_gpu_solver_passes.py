"""The solver's grid sums and its kept work space: few and odd numbers of
unknowns (fewer workgroups than the passes' grid, a value left over from the
pairs), repeated solves with another one between, both precisions, a caller's
stream, and two threads on one operator."""
import threading

import numpy as np
import pytest

import oracle_bindings as ob
import sum_factorization_kernels_amd as sfk
from helpers import rel_err, to_dev, to_np

pytestmark = pytest.mark.gpu

CASES = [(1, (2, 2, 2)), (1, (3, 2, 5)), (2, (3, 2, 2)), (3, (5, 4, 3)), (4, (7, 6, 5)), (6, (9, 8, 9))]


def _problem(degree, nc, seed):
    ij = (float(nc[0]), 1.1 * nc[1], 0.9 * nc[2])
    op = sfk.Operator(sfk.CONT_LAPLACE, degree, nc, inv_jac=ij)
    rng = np.random.default_rng(seed)
    inner = to_np(op.diagonal()) != 0
    return ij, op, [rng.standard_normal(op.vector_size) * inner for _ in range(2)]


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("degree,nc", CASES)
def test_solves(cuda, degree, nc, mixed):
    import torch
    ij, op, rhs = _problem(degree, nc, 8300 + degree)
    sm = sfk.Operator(sfk.CONT_LAPLACE, degree, nc, inv_jac=ij, precision=sfk.FP32) if mixed else op
    solutions = []
    stream = torch.cuda.Stream()
    for which, st in ((0, None), (1, None), (0, stream)):
        with torch.cuda.stream(st or torch.cuda.current_stream()):
            b = to_dev(rhs[which])
            x = torch.zeros_like(b)
            stats = sfk.solve_cg_cheby(op, sm, b, x, 1e-10, 500, 6, 12)
            torch.cuda.current_stream().synchronize()
        res = rhs[which] - ob.cont_laplacian(degree, nc, ij, to_np(x))
        assert np.linalg.norm(res) <= 1.01e-10 * np.linalg.norm(rhs[which]), which
        assert abs(np.linalg.norm(res) - stats.final_residual) <= 1e-2 * stats.final_residual + 1e-13
        solutions.append(to_np(x))
    # the work space's last contents do not matter
    assert np.array_equal(solutions[0], solutions[2])


def test_two_threads_on_one_operator(cuda):
    import torch
    degree, nc = 4, (12, 11, 13)
    ij, op, rhs = _problem(degree, nc, 8400)
    want = []
    for r in rhs:
        x = torch.zeros(op.vector_size, dtype=torch.float64, device="cuda")
        sfk.solve_cg_cheby(op, op, to_dev(r), x, 1e-10, 500, 6, 12)
        want.append(to_np(x))
    got = [None, None]
    start = threading.Barrier(2)

    def solve(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            b = to_dev(rhs[i])
            start.wait(timeout=60)
            for _ in range(3):
                x = torch.zeros_like(b)
                sfk.solve_cg_cheby(op, op, b, x, 1e-10, 500, 6, 12)
            torch.cuda.current_stream().synchronize()
            got[i] = to_np(x)

    threads = [threading.Thread(target=solve, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(got, want):
        assert rel_err(a, b) == 0.0
