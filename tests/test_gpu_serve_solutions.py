"""Served solutions are put in the reference's order on the device, in tiles of
32 elements by 32 nodes: one element, one node row more or less than a tile,
and ragged tiles.  Requests of changing degrees share a server, so that its
captured iterations outlive the degrees that finish first.  A solution in the
wrong order would leave a residual of the size of b."""
import pytest

pytestmark = pytest.mark.gpu
SHAPES = [(1, 1), (1, 16), (4, 5), (8, 4), (31, 1), (33, 2), (11, 11), (6, 16)]      # dim, p


@pytest.mark.parametrize("method", ["cg", "pcg"])
def test_every_solution_solves_its_request(sipg, method):
    S = sipg.Server(1e9)
    assert S.set_method(sipg.METHOD_PCG if method == "pcg" else sipg.METHOD_CG) == sipg.OK
    for burst in (SHAPES, SHAPES[::-1], SHAPES[2:5]):
        ids = {}
        for k, (d, p) in enumerate(burst):
            ids[S.submit(d, p, sipg.pen_sigma(p), sipg.forcing_draw(k, 1, 4, 4), 1e-9, maxit=30000)] = k
        left = len(ids)
        for _ in range(20000):
            if not left:
                break
            S.progress()
            while (got := S.take_ex(-1)) is not None:
                k = ids[got[0]]
                d, p = burst[k]
                assert got[1].status == sipg.OK, (d, p, got[1].status)
                op = sipg.Operator(d, d, p, sipg.pen_sigma(p), sipg.F64)
                b = op.vector()
                op.rhs_fourier(sipg.forcing_draw(k, 1, 4, 4), b)
                assert op.true_relres(op.to_device(got[2]), b) <= 1.0001e-9, (d, p)
                left -= 1
        assert left == 0
