"""Batched and served PCG on instances of many items (strips by bands of
rows): sums over an instance with more than 512 are added up in launches of
their own.  Sizes on either side of that, and far above; the solution of an
instance does not depend on what else is in the batch, to the bit; and the
cost of an iteration follows the unknowns, not the square of them."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solve(sipg, dims, ps, bs, which):
    B = sipg.Batch([dims[i][0] for i in which], [dims[i][1] for i in which], [ps[i] for i in which],
                   [sipg.pen_sigma(ps[i]) for i in which])
    for p in {ps[i] for i in which}:
        assert B.set_shape(p, 8, 2) == sipg.OK                    # bands of four rows
    x, b = B.vector(), B.vector()
    for k, i in enumerate(which):
        B.upload(k, np.zeros_like(bs[i]), x)
        B.upload(k, bs[i], b)
    st, info = B.pcg(x, b, 1e-9, sipg.TOL_REL, maxit=30000, replace_factor=3e-2)
    assert st == sipg.OK and all(f.status == sipg.OK and f.replacements >= 1 for f in info)
    return [B.download(k, x) for k in range(len(which))]


def test_batch_on_either_side_of_the_limit(sipg):
    # 512, 513 and 528 items; 9 of degree 5; 2,106 of degree 8
    dims = [(16 * 21, 32 * 4), (27 * 21, 19 * 4), (16 * 21 - 5, 33 * 4 - 1), (20, 5), (7 * 27, 78 * 4)]
    ps = [2, 2, 2, 5, 8]
    bs = [np.random.default_rng(i).uniform(-1, 1, d[0] * d[1] * (p + 1) ** 2) for i, (d, p) in enumerate(zip(dims, ps))]
    got = _solve(sipg, dims, ps, bs, range(5))
    for i, (d, p) in enumerate(zip(dims, ps)):
        op = sipg.Operator(d[0], d[1], p, sipg.pen_sigma(p), sipg.F64)
        assert op.true_relres(op.to_device(got[i]), op.to_device(bs[i])) <= 1.0001e-9, (d, p)
        assert np.array_equal(_solve(sipg, dims, ps, bs, [i])[0], got[i]), (d, p)


@pytest.mark.parametrize("p", [3, 12])
def test_batch_of_one_degree_with_more_items_than_workgroups(sipg, p):
    # one list only: 6 items to an instance (2 strips, 3 bands)
    d = (64 // (p + 1) + 1, 9)
    x0 = np.random.default_rng(p).uniform(-1, 1, d[0] * d[1] * (p + 1) ** 2)
    B = sipg.Batch([d[0]] * 700, [d[1]] * 700, [p] * 700, [sipg.pen_sigma(p)] * 700)
    assert B.set_shape(p, 8, 2) == sipg.OK
    x, y = B.vector(), B.vector()
    for i in range(700):
        B.upload(i, x0 * (1 + i % 3), x)
    assert B.apply(x, y) == sipg.OK
    op = sipg.Operator(d[0], d[1], p, sipg.pen_sigma(p), sipg.F64)
    want = [op.apply_host(x0 * (1 + k)) for k in range(3)]
    assert all(np.array_equal(B.download(i, y), want[i % 3]) for i in range(700))


def test_server_takes_a_large_request_among_small_ones(sipg):
    # 300 x 300 of degree 2: 570 items, after the iterations were captured
    # for small requests of the same degrees
    def serve(reqs, late):
        S = sipg.Server(1e9)
        assert S.set_method(sipg.METHOD_PCG) == sipg.OK
        out, ids = {}, {}
        for step in range(20000):
            if step == 0 or step == 3:
                for k, (d, p) in reqs.items():
                    if (k in late) == (step == 3):
                        ids[S.submit(d, p, sipg.pen_sigma(p), sipg.forcing_draw(k, 1, 4, 4), 1e-9, maxit=30000)] = k
            S.progress()
            while (g := S.take_ex(-1)) is not None:
                assert g[1].status == sipg.OK, ids[g[0]]
                out[ids[g[0]]] = g[2]
            if step >= 3 and len(out) == len(reqs):
                return out
        raise AssertionError("not finished")

    reqs = {0: (40, 2), 1: (30, 8), 2: (300, 2), 3: (21, 2)}
    got = serve(reqs, late={2, 3})
    for k, (d, p) in reqs.items():
        op = sipg.Operator(d, d, p, sipg.pen_sigma(p), sipg.F64)
        b = op.vector()
        op.rhs_fourier(sipg.forcing_draw(k, 1, 4, 4), b)
        assert op.true_relres(op.to_device(got[k]), b) <= 1.0001e-9, (d, p)
        assert np.array_equal(serve({k: reqs[k]}, late=set())[k], got[k]), (d, p)


def test_cost_of_an_iteration_follows_the_unknowns(sipg):
    # 16.8 million unknowns as one instance (16,384 items) and as 64 of 256
    # each; the same passes over memory, so the same time.  Adding up all
    # items in each made it 4 times as long.
    def us(dims):
        B = sipg.Batch(dims, dims, [1] * len(dims), [sipg.pen_sigma(1)] * len(dims))
        assert B.set_shape(1, 8, 4) == sipg.OK
        x, b = B.vector(), B.vector()
        for i in range(len(dims)):
            B.rhs_fourier(i, sipg.forcing_draw(i, 4, 4, 4), b)
        best = 1e9
        for _ in range(4):
            x.zero()
            t = time.perf_counter()
            _, info = B.pcg(x, b, 1e-30, sipg.TOL_REL, maxit=64)
            best = min(best, (time.perf_counter() - t) / max(f.iters for f in info))
        return best
    one, many = us([2048]), us([256] * 64)
    assert one <= 1.6 * many, (one, many)
