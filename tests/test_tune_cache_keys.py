"""SFK_TUNE_CACHE lines that must not be taken: those of a library with other
tiles or kernels (the key lacks this library's part), and those whose tile for
the Chebyshev launches set_schedule refuses."""
import pytest

import sum_factorization_kernels_amd as sfk

NC, IJ = (24, 3, 4), (24.0, 3.0, 4.0)


@pytest.mark.parametrize("kind,basis,degree", [(sfk.CONT_LAPLACE, 1, 6), (sfk.DG_SIPG, 0, 5)])
def test_line_of_another_library(tmp_path, monkeypatch, kind, basis, degree):
    """without a device nothing can be timed: a line that is taken is the only
    way to a result"""
    path = tmp_path / "tune.txt"
    path.write_text(f"nodevice/k{kind}/p{degree}/f0/b{basis}/g0/fl0/n24x3x4/r1 1 0 {2 if kind == 1 else -1} "
                    f"{1 if kind == 1 else 0} 2 -1 0 0 0.125\n")
    monkeypatch.setenv("SFK_TUNE_CACHE", str(path))
    op = sfk.Operator(kind, degree, NC, inv_jac=IJ)
    before = op.schedule
    try:
        sched, t = op.tune(repeats=1, stream=0)
    except sfk.SfkError:  # no device: not timed
        assert op.schedule == before
    else:
        assert t != 0.125


@pytest.mark.gpu
def test_chebyshev_tile_that_does_not_fit(cuda, tmp_path, monkeypatch):
    path = tmp_path / "tune.txt"
    monkeypatch.setenv("SFK_TUNE_CACHE", str(path))
    sfk.Operator(sfk.CONT_LAPLACE, 6, NC, inv_jac=IJ).tune(repeats=1)
    f = path.read_text().split()
    op = sfk.Operator(sfk.CONT_LAPLACE, 6, NC, inv_jac=IJ)
    with pytest.raises(sfk.SfkError):
        op.set_schedule(0, 1, 2, 5, 2)  # the 24-cell tile fits FP32 only
    f[6:9], f[9] = ["5", "2", "1"], "0.125"
    path.write_text(" ".join(f) + "\n")
    _, t = op.tune(repeats=1)
    assert t != 0.125 and op.smoother_schedule[3] != 5
    f[6:9] = ["3", "2", "1"]
    path.write_text(" ".join(f) + "\n")
    op2 = sfk.Operator(sfk.CONT_LAPLACE, 6, NC, inv_jac=IJ)
    _, t = op2.tune(repeats=1)
    assert t == 0.125 and op2.smoother_schedule[3] == 3
