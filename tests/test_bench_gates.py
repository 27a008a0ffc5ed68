"""What the benchmark accepts as a solve: one that reaches its tolerance, and
only where a leg says so, one that ends at the FP64 floor short of its cap.
A stub stands in for the library."""
import types

import numpy as np
import pytest

import bench


def _stub(status, iters, relres=5e-11, n=1024):
    info = types.SimpleNamespace(iters=iters, replacements=1, status=status)
    vec = types.SimpleNamespace(zero=lambda: None)
    op = types.SimpleNamespace(n=n, vector=lambda: vec, rhs_fourier=lambda modes, b: None,
                               true_relres=lambda x, b: relres)
    for name in ("cg_ex", "pcg", "pcg2", "pcg2_mixed"):
        setattr(op, name, lambda *a, **k: (status, info))
    sipg = types.SimpleNamespace(OK=0, NOT_CONVERGED=6, ERR_BREAKDOWN=8, TOL_REL=1, F64=0, KERNEL_AUTO=0,
                                 synchronize=lambda: None, strerror=lambda s: f"status {s}", pen_sigma=lambda p: 1.0,
                                 Operator=lambda *a: op)
    return sipg, op, vec


@pytest.mark.parametrize("method", ["fp64", "pcg", "pcg2", "mixed"])
def test_a_solve_that_does_not_converge_raises(method):
    sipg, op, v = _stub(6, 1000)
    with pytest.raises(RuntimeError):
        bench.gpu_solve(sipg, op, v, v, method)


def test_the_floor_is_accepted_only_where_asked_and_short_of_the_cap():
    sipg, op, v = _stub(6, 1000)
    assert bench.gpu_solve(sipg, op, v, v, "fp64", floor_ok=True)[1].iters == 1000
    for method in ("pcg2", "mixed"):
        with pytest.raises(RuntimeError):
            bench.gpu_solve(sipg, op, v, v, method, floor_ok=True)
    for status, iters in ((6, bench.MAXIT_FP64), (8, 10)):
        sipg, op, v = _stub(status, iters)
        with pytest.raises(RuntimeError):
            bench.gpu_solve(sipg, op, v, v, "fp64", floor_ok=True)


def test_the_smallest_workload_must_converge():
    u = np.load(bench.ROOT + "/tests/golden/c1_solution.npz")
    for status, relres, ok in ((0, 9e-11, True), (6, 9e-11, False), (0, 2e-10, False)):
        sipg, op, v = _stub(status, 200, relres)
        op.download = lambda x: u["u"]
        if ok:
            assert bench.c1_leg(sipg)["fp64"]["true_relres"] == relres
        else:
            with pytest.raises(RuntimeError):
                bench.c1_leg(sipg)


def test_no_ratio_with_a_solve_that_missed_its_tolerance():
    assert bench.time_ratio(2.0, 4.0) == 0.5
    assert bench.time_ratio(2.0, None) is None and bench.time_ratio(None, 4.0) is None
