"""CG iterations inside one workgroup (problems of at most 4,096 unknowns)
against the three-launch iteration, which an explicit kernel setting
selects, and against the oracle.

Both run the same recurrence in FP64 with their sums in other orders: after
k iterations the iterates differ by rounding, amplified as CG amplifies it.
For five iterations 1e-12 relative covers n 2^-53 on sums of n <= 4,096
terms; converged solutions are compared at the tolerance of the other CG
tests, 1e-8, and iteration counts within 2 % and three."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 4,096 unknowns exactly, just below, single elements, single rows, every
# kind of row stride (p + 1 odd and even), and lines that do not divide 512
MESHES = [(16, 16, 3), (32, 32, 1), (4, 4, 15), (21, 21, 2), (1, 1, 8), (1, 1, 1), (1, 40, 5), (37, 1, 4), (7, 7, 8),
          (9, 3, 6), (5, 6, 10), (3, 3, 16), (2, 5, 13), (4, 6, 7)]


def _op(sipg, dx, dy, p, dtype, one_group):
    op = sipg.Operator(dx, dy, p, sipg.pen_sigma(p), dtype)
    op.set_kernel(sipg.KERNEL_AUTO if one_group else sipg.KERNEL_VALU)
    return op


@pytest.mark.parametrize("dx,dy,p", MESHES)
def test_small_cg_matches_launches_and_oracle(sipg, oracle, dx, dy, p):
    n = dx * dy * (p + 1) ** 2
    assert n <= 4096
    b = np.random.default_rng(dx + 10 * dy + 100 * p).uniform(-1, 1, n)
    got = {}
    for one in (True, False):
        op = _op(sipg, dx, dy, p, sipg.F64, one)
        bd, x = op.to_device(b), op.vector()
        x.zero()
        st, it, res = op.cg(x, bd, 1e-11, sipg.TOL_REL, maxit=4 * n + 100)
        assert st == sipg.OK, (one, st, it)
        got[one] = (it, op.download(x))
        x.zero()
        st, it, _ = op.cg(x, bd, 0.0, sipg.TOL_REL, maxit=5)
        assert it == 5 and st == sipg.NOT_CONVERGED
        got[one] += (op.download(x),)
    (i1, x1, y1), (i2, x2, y2) = got[True], got[False]
    assert abs(i1 - i2) <= max(3, 0.02 * i2), (i1, i2)
    if i2 > 10:                                           # (a few-unknown problem is exhausted by then)
        assert np.linalg.norm(y1 - y2) <= 1e-12 * np.linalg.norm(y2)
    xo, _, _ = oracle.cg(dx, dy, p, sipg.pen_sigma(p), b, tol=1e-13, maxit=8 * n + 100)
    assert np.linalg.norm(x1 - xo) <= 1e-8 * np.linalg.norm(xo)


@pytest.mark.parametrize("dx,dy,p", [(16, 16, 3), (5, 6, 10), (4, 4, 15)])
def test_small_cg_with_replacements_and_fp32(sipg, dx, dy, p):
    n = dx * dy * (p + 1) ** 2
    b = np.random.default_rng(n).uniform(-1, 1, n)
    op = _op(sipg, dx, dy, p, sipg.F64, True)
    bd, x = op.to_device(b), op.vector()
    x.zero()
    st, info = op.cg_ex(x, bd, 1e-10, sipg.TOL_REL, maxit=20000, replace_factor=3e-3, true_stop=True)
    assert st == sipg.OK and info.replacements >= 1 and op.true_relres(x, bd) <= 1e-10
    x.zero()
    st, info = op.cg_mixed(x, bd, 1e-10, sipg.TOL_REL, maxit=60000)
    assert st == sipg.OK and op.true_relres(x, bd) <= 1e-10


def test_small_cg_status_codes(sipg):
    # a zero right-hand side is met at once; NaN and an operator that is not
    # positive end the solve as in the launches
    op = _op(sipg, 6, 6, 4, sipg.F64, True)
    x, b = op.vector(), op.vector()
    x.zero()
    b.zero()
    st, it, res = op.cg(x, b, 1e-10, sipg.TOL_REL)
    assert st == sipg.OK and it == 0
    h = np.ones(op.n)
    h[7] = np.nan
    op.upload(h, b)
    assert op.cg(x, b, 1e-10, sipg.TOL_REL)[0] == sipg.ERR_NONFINITE
    bad = sipg.Operator(4, 4, 3, -400.0, sipg.F64)
    ref = sipg.Operator(4, 4, 3, -400.0, sipg.F64)
    ref.set_kernel(sipg.KERNEL_VALU)
    got = []
    for o in (bad, ref):
        bb, xx = o.to_device(np.random.default_rng(1).uniform(-1, 1, o.n)), o.vector()
        xx.zero()
        got.append(o.cg(xx, bb, 1e-10, sipg.TOL_REL, maxit=50)[:2])
    assert got[0] == got[1] and got[0][0] == sipg.ERR_BREAKDOWN
