"""The run-time-table operator (degrees above 16) on the matrix cores: degrees
at the edges of its 16-node tiles, and meshes of more elements than the
device holds workgroups, against the oracle at the tolerances of the other
tests of this operator (1e-12 and, in FP32, 2e-6 (p+1) of max|y|)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,dx,dy", [(17, 45, 43), (30, 2, 3), (31, 7, 1), (32, 1, 7), (33, 27, 23), (46, 3, 2),
                                     (47, 2, 2), (48, 2, 3), (62, 3, 1), (63, 18, 16)])
@pytest.mark.parametrize("f32", [False, True])
def test_tiles_match_oracle(sipg, oracle, p, dx, dy, f32):
    pen = sipg.pen_sigma(p)
    op = sipg.Operator(dx, dy, p, pen, sipg.F32 if f32 else sipg.F64)
    x = np.random.default_rng(p).uniform(-1, 1, op.n)
    if f32:
        x = x.astype(np.float32).astype(np.float64)
    y = op.apply_host(x)
    ref = oracle.apply(dx, dy, p, pen, x)
    assert np.max(np.abs(y - ref)) <= (2e-6 * (p + 1) if f32 else 1e-12) * np.max(np.abs(ref))


@pytest.mark.parametrize("p,dim", [(17, 5), (33, 3), (48, 2)])
def test_fused_product_drives_cg(sipg, p, dim):
    op = sipg.Operator(dim, dim, p, sipg.pen_sigma(p), sipg.F64)
    b, x = op.vector(), op.vector()
    op.rhs_fourier(sipg.forcing_draw(p, 1, 4, 4), b)
    x.zero()
    st, info = op.cg_ex(x, b, 1e-8, sipg.TOL_REL, maxit=30000, replace_factor=3e-3)
    assert st == sipg.OK, (st, info.iters)
    assert op.true_relres(x, b) <= 1.0001e-8
