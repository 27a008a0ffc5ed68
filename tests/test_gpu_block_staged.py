"""The block-staged operator at p = 10 and 12 in FP32, the kernel of these
degrees unless another is asked for: meshes at the edges of its blocks of
64 / (p+1) by 4 elements, against the oracle at the tolerance of the other
FP32 operator tests (2e-6 (p+1) of max|y|), to the bit the strip kernel's
results (the same arithmetic on a line), and driving CG with its own sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [10, 12])
def test_matches_oracle_and_strips(sipg, oracle, p):
    pen, w = sipg.pen_sigma(p), 64 // (p + 1)
    for dx, dy in [(1, 1), (w, 4), (w - 1, 3), (w + 1, 5), (2 * w, 1), (1, 9), (3 * w + 2, 13), (41, 30)]:
        op = sipg.Operator(dx, dy, p, pen, sipg.F32)
        assert op.kernel() == sipg.KERNEL_WAVE
        x = np.random.default_rng(100 * dx + dy).uniform(-1, 1, op.n).astype(np.float32).astype(np.float64)
        y = op.apply_host(x)
        op.set_kernel(sipg.KERNEL_VALU)
        assert op.kernel() == sipg.KERNEL_VALU and np.array_equal(op.apply_host(x), y), (dx, dy)
        ref = oracle.apply(dx, dy, p, pen, x)
        assert np.max(np.abs(y - ref)) <= 2e-6 * (p + 1) * np.max(np.abs(ref)), (dx, dy)


@pytest.mark.parametrize("p", [10, 12])
def test_in_fp64_strips_stay(sipg, p):
    op = sipg.Operator(5, 5, p, sipg.pen_sigma(p), sipg.F64)
    assert op.kernel() == sipg.KERNEL_VALU and op.kernel(sipg.F32) == sipg.KERNEL_WAVE
    op.set_kernel(sipg.KERNEL_WAVE)
    assert op.kernel() == sipg.KERNEL_VALU


@pytest.mark.parametrize("p", [10, 12])
def test_drives_mixed_cg(sipg, p):
    op = sipg.Operator(11, 9, p, sipg.pen_sigma(p), sipg.F64)
    b = op.to_device(np.random.default_rng(p).uniform(-1, 1, op.n))
    x = op.vector()
    x.zero()
    st, info = op.pcg_mixed(x, b, 1e-9, sipg.TOL_REL, maxit=60000, replace_factor=1e-1)
    assert st == sipg.OK and op.true_relres(x, b) <= 1.0001e-9
