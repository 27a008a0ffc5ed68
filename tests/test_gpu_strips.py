"""The operator on strips marched in y, for one mesh and for batches.

Meshes at the edges of the split: one element, one row, one column, fewer
rows than waves, one column more than a strip or one less, more rows than a
band.  Against the oracle at the tolerance of the other operator tests (1e-12
of max|y| in FP64: 4 (p+1) products a value with an error of a few 2^-53
each; 2e-6 (p+1) in FP32), and to the bit where two kernels do the same
arithmetic: the block-staged kernel of the even degrees up to 8, and a batch
whatever degrees it holds (one launch, compiled in classes of up to 8, 12 and
16)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _meshes(p):
    w = 64 // (p + 1)
    return [(1, 1), (1, 9), (w, 1), (w + 1, 3), (2 * w - 1, 4), (3 * w, 13), (w + 2, 37)]


@pytest.mark.parametrize("p", range(1, 17))
@pytest.mark.parametrize("f32", [False, True])
def test_strips_match_oracle_and_block_staged(sipg, oracle, p, f32):
    pen = sipg.pen_sigma(p)
    for dx, dy in _meshes(p):
        op = sipg.Operator(dx, dy, p, pen, sipg.F32 if f32 else sipg.F64)
        x = np.random.default_rng(100 * dx + dy).uniform(-1, 1, op.n)
        if f32:
            x = x.astype(np.float32).astype(np.float64)
        op.set_kernel(sipg.KERNEL_VALU)
        y = op.apply_host(x)
        ref = oracle.apply(dx, dy, p, pen, x)
        assert np.max(np.abs(y - ref)) <= (2e-6 * (p + 1) if f32 else 1e-12) * np.max(np.abs(ref)), (dx, dy)
        if p % 2 == 0 and p <= 8:
            op.set_kernel(sipg.KERNEL_WAVE)
            assert np.array_equal(op.apply_host(x), y), (dx, dy)


def _batch(sipg, dims, ps, shape):
    B = sipg.Batch([d[0] for d in dims], [d[1] for d in dims], ps, [sipg.pen_sigma(p) for p in ps])
    for p in set(ps):
        assert B.set_shape(p, *shape) == sipg.OK
    return B


@pytest.mark.parametrize("shape,top", [((16, 4), 8), ((16, 4), 12), ((8, 4), 16), ((8, 2), 3), ((8, 2), 16)])
def test_batch_of_every_degree_equals_single_applies(sipg, shape, top):
    ps = list(range(1, top + 1))
    dims = [_meshes(p)[(p + top) % 7] for p in ps]
    B = _batch(sipg, dims, ps, shape)
    x, y = B.vector(), B.vector()
    xs = [np.random.default_rng(i).uniform(-1, 1, d[0] * d[1] * (p + 1) ** 2) for i, (d, p) in enumerate(zip(dims, ps))]
    for i, v in enumerate(xs):
        B.upload(i, v, x)
    assert B.apply(x, y) == sipg.OK
    for i, (d, p) in enumerate(zip(dims, ps)):
        op = sipg.Operator(d[0], d[1], p, sipg.pen_sigma(p), sipg.F64)
        assert np.array_equal(B.download(i, y), op.apply_host(xs[i])), (d, p)


@pytest.mark.parametrize("top", [8, 12, 16])
def test_batch_of_more_items_than_workgroups(sipg, top):
    """Workgroups take one item after another, of changing degrees whose tiles
    lie elsewhere in LDS: 200 instances of each degree, to the bit the single
    apply's results."""
    kinds = [((64 // (p + 1) + 1, 5 + p % 5), p) for p in range(1, top + 1)]
    xs = [np.random.default_rng(p).uniform(-1, 1, d[0] * d[1] * (p + 1) ** 2) for d, p in kinds]
    ref = [sipg.Operator(d[0], d[1], p, sipg.pen_sigma(p), sipg.F64).apply_host(x) for (d, p), x in zip(kinds, xs)]
    of = list(range(top)) * 200
    B = _batch(sipg, [kinds[k][0] for k in of], [kinds[k][1] for k in of], (8, 2))
    x, y = B.vector(), B.vector()
    for i, k in enumerate(of):
        B.upload(i, xs[k], x)
    assert B.apply(x, y) == sipg.OK
    bad = [(i, kinds[k]) for i, k in enumerate(of) if not np.array_equal(B.download(i, y), ref[k])]
    assert not bad, (len(bad), bad[:5])


@pytest.mark.parametrize("top", [8, 12, 16])
def test_batch_pcg_of_every_degree(sipg, top):
    """Every degree in one launch, replacements on: each instance meets its
    tolerance on the true residual, as the single solve does; the solution
    does not depend on the other instances."""
    ps = list(range(1, top + 1))
    dims = [_meshes(p)[(3 * p) % 7] for p in ps]
    bs = [np.random.default_rng(50 + i).uniform(-1, 1, d[0] * d[1] * (p + 1) ** 2)
          for i, (d, p) in enumerate(zip(dims, ps))]

    def solve(which):
        B = _batch(sipg, [dims[i] for i in which], [ps[i] for i in which], (8, 4))
        x, b = B.vector(), B.vector()
        for k, i in enumerate(which):
            B.upload(k, np.zeros_like(bs[i]), x)
            B.upload(k, bs[i], b)
        st, info = B.pcg(x, b, 1e-9, sipg.TOL_REL, maxit=5000, replace_factor=3e-2)
        assert st == sipg.OK and all(f.status == sipg.OK for f in info)
        return {i: (B.download(k, x), info[k].replacements) for k, i in enumerate(which)}

    got = solve(range(len(ps)))
    assert max(r for _, r in got.values()) >= 2
    for i, (d, p) in enumerate(zip(dims, ps)):
        op = sipg.Operator(d[0], d[1], p, sipg.pen_sigma(p), sipg.F64)
        assert op.true_relres(op.to_device(got[i][0]), op.to_device(bs[i])) <= 1.0001e-9, (d, p)
    for i in (0, top // 2, top - 1):
        assert np.array_equal(solve([i])[i][0], got[i][0]), ps[i]
