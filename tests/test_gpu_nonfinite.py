"""A NaN reaches the outputs that depend on it and no others: the operator at
every kind of kernel against the oracle's mask (a node's value enters its two
lines, and through the faces the neighbours' lines), block-Jacobi within its
element, batches within their instance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [1, 2, 7, 8, 10, 12, 15, 16, 17, 20, 31, 33, 47, 63])
@pytest.mark.parametrize("f32", [False, True])
def test_operator(sipg, oracle, p, f32):
    dx, dy, n1 = 3, 4, p + 1
    pen, noe = sipg.pen_sigma(p), 12
    op = sipg.Operator(dx, dy, p, pen, sipg.F32 if f32 else sipg.F64)
    rng = np.random.default_rng(p)
    x0 = rng.uniform(-1, 1, op.n)
    mid = n1 // 2
    # reference order: node (i1, i2) of element e at (i1 n1 + i2) noe + e
    for e, i1, i2 in [(4, mid, mid), (4, 0, mid), (7, mid, p), (0, 0, 0), (11, p, mid)]:
        x = x0.copy()
        x[(i1 * n1 + i2) * noe + e] = np.nan
        want = np.isfinite(oracle.apply(dx, dy, p, pen, x))
        assert not want.all()
        # (the matrix cores' FP32 products at p = 15 carry it further, to
        # values of the same and the neighbouring elements)
        for kernel in (sipg.KERNEL_VALU,) if f32 and p == 15 else (sipg.KERNEL_AUTO, sipg.KERNEL_VALU):
            op.set_kernel(kernel)
            assert np.array_equal(np.isfinite(op.apply_host(x)), want), (e, i1, i2, kernel)


@pytest.mark.parametrize("p", [1, 4, 7, 8, 15, 16])
@pytest.mark.parametrize("f32", [False, True])
def test_block_jacobi(sipg, p, f32):
    op = sipg.Operator(9, 5, p, sipg.pen_sigma(p), sipg.F32 if f32 else sipg.F64)
    x = np.random.default_rng(p).uniform(-1, 1, op.n).reshape(-1, 45)
    x[(p + 1) // 2, 17] = np.nan
    r, z = op.to_device(x.reshape(-1)), op.vector()
    op.prec_apply(r, z)
    bad = ~np.isfinite(op.download(z).reshape(-1, 45))
    assert bad[:, 17].all() and not np.delete(bad, 17, axis=1).any()


@pytest.mark.parametrize("method", ["cg", "pcg"])
def test_batch(sipg, method):
    dims, ps = [7, 9, 30, 6], [3, 8, 2, 12]
    B = sipg.Batch(dims, dims, ps, [sipg.pen_sigma(p) for p in ps])
    x, b = B.vector(), B.vector()
    for i, (d, p) in enumerate(zip(dims, ps)):
        v = np.random.default_rng(i).uniform(-1, 1, d * d * (p + 1) ** 2)
        if i == 1:
            v[5] = np.nan
        B.upload(i, v, b)
        B.upload(i, np.zeros_like(v), x)
    st, info = getattr(B, method)(x, b, 1e-8, sipg.TOL_REL, maxit=20000, replace_factor=1e-2)
    assert [f.status for f in info] == [sipg.OK, sipg.ERR_NONFINITE, sipg.OK, sipg.OK]
    assert all(np.isfinite(B.download(i, x)).all() for i in (0, 2, 3))
