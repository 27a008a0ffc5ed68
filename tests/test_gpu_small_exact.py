"""Small CG solves do not run on past their tolerance: on so few unknowns that
the recursion would reach zero inside a chunk of iterations, and with a cap
just above what the tolerance takes, they finish on their true residual and
report no breakdown and no cap, in one workgroup as in launches."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dx,dy,p", [(1, 1, 1), (1, 1, 2), (2, 1, 1), (1, 2, 1), (2, 2, 1), (1, 1, 5)])
@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("one_group", [True, False])
def test_exact_solves_finish(sipg, dx, dy, p, f32, one_group):
    op = sipg.Operator(dx, dy, p, sipg.pen_sigma(p), sipg.F32 if f32 else sipg.F64)
    op.set_kernel(sipg.KERNEL_AUTO if one_group else sipg.KERNEL_VALU)
    b = op.to_device(np.random.default_rng(op.n).uniform(-1, 1, op.n))
    for tol in (0.4, 1e-3) if f32 else (0.4, 1e-3, 1e-9):
        for replace in (0.0, 1e-2):
            x = op.vector()
            x.zero()
            st, info = op.cg_ex(x, b, tol, sipg.TOL_REL, maxit=2000, replace_factor=replace)
            assert st == sipg.OK, (tol, replace, st, info.iters)
            assert info.true_res_norm <= tol * info.b_norm
            if not f32:
                assert op.true_relres(x, b) <= 1.0001 * tol


@pytest.mark.parametrize("dx,dy,p", [(1, 50, 2), (8, 8, 3), (6, 6, 4), (16, 16, 3), (3, 3, 16)])
def test_a_cap_above_what_the_tolerance_takes(sipg, oracle, dx, dy, p):
    # the oracle's count and eight: a final check, and room for the rounding
    # of another order of summation
    op = sipg.Operator(dx, dy, p, sipg.pen_sigma(p), sipg.F64)
    b = np.random.default_rng(op.n).uniform(-1, 1, op.n)
    bd, x = op.to_device(b), op.vector()
    _, its, _ = oracle.cg(dx, dy, p, sipg.pen_sigma(p), b, tol=1e-3, tol_mode=1)
    x.zero()
    st, info = op.cg_ex(x, bd, 1e-3, sipg.TOL_REL, maxit=its + 8)
    assert st == sipg.OK and info.iters <= its + 8, (st, info.iters, its)
