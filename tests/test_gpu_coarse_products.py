"""The coarse solve's sine-transform products at the edges of their tiles:
16 indices of one parity per tile, k blocks of four shared out over the
waves, the folded middle of odd sizes, and the rocBLAS route above them.

The coarse part of the two-level preconditioner, z2 - z1 = P0^T A0^-1 P0 r,
is compared with A0 = Ky (x) Mx + My (x) Kx solved in numpy.  z1 and z2 are
rounded at the size of M_BJ^-1 r, so the difference carries a few 2^-53 of
max |z2|; the products themselves add n 2^-53 relative (n <= 130 here) in
four steps: 1e-11 max |coarse| covers both, as in the other coarse tests.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _vertex_weights(n1, xi, dx, dy, u):
    """P0 u: the bilinear vertex sums of u (reference order), interior vertices."""
    t = u.reshape(n1, n1, dy, dx)
    S = np.zeros((dy + 1, dx + 1))
    for wy, r0 in ((xi, 0), (1 - xi, 1)):                 # top vertex row of an element: weight y
        for wx, c0 in ((1 - xi, 0), (xi, 1)):
            S[r0:r0 + dy, c0:c0 + dx] += np.einsum("a,b,abrc->rc", wx, wy, t)
    return S[1:dy, 1:dx]


def _factors(n):
    K = 2 * np.eye(n) - np.eye(n, k=1) - np.eye(n, k=-1)
    M = (2 / 3) * np.eye(n) + (1 / 6) * (np.eye(n, k=1) + np.eye(n, k=-1))
    return K, M


@pytest.mark.parametrize("dx,dy", [(2, 2), (3, 2), (2, 9), (17, 18), (18, 17), (31, 34), (33, 32), (34, 33), (65, 67),
                                   (130, 66), (129, 131)])
def test_coarse_products_at_tile_edges(sipg, oracle, dx, dy):
    p = 2
    n1 = p + 1
    xi = (oracle.gll(p)[0] + 1) / 2
    op = sipg.Operator(dx, dy, p, sipg.pen_sigma(p), sipg.F64)
    r = np.random.default_rng(1000 * dx + dy).uniform(-1, 1, op.n)
    rd, z1, z2 = op.vector(), op.vector(), op.vector()
    op.upload(r, rd)
    op.prec_apply(rd, z1)
    op.prec2_apply(rd, z2)
    coarse = op.download(z2) - op.download(z1)
    S = _vertex_weights(n1, xi, dx, dy, r)
    (Kx, Mx), (Ky, My) = _factors(dx - 1), _factors(dy - 1)
    # both factors are diagonalised by the sine basis: solve there
    lx, Vx = np.linalg.eigh(Kx)
    ly, Vy = np.linalg.eigh(Ky)
    mx, my = np.diag(Vx.T @ Mx @ Vx), np.diag(Vy.T @ My @ Vy)
    C = np.zeros((dy + 1, dx + 1))
    C[1:dy, 1:dx] = Vy @ ((Vy.T @ S @ Vx) / (np.outer(my, lx) + np.outer(ly, mx))) @ Vx.T
    X, Y = xi[:, None, None, None], xi[None, :, None, None]
    tl, tr, bl, br = C[:-1, :-1], C[:-1, 1:], C[1:, :-1], C[1:, 1:]
    want = ((1 - Y) * ((1 - X) * bl + X * br) + Y * ((1 - X) * tl + X * tr)).reshape(-1)
    assert np.max(np.abs(coarse - want)) <= 1e-11 * np.max(np.abs(want)), np.max(np.abs(coarse - want))


def test_coarse_products_by_rocblas(sipg, oracle):
    # 545 x 544 elements lie above the size where the products go to rocBLAS;
    # the same problem's coarse part through a coarse function: r = A P0^T v
    # gives P0^T v back (A amplifies rounding by its norm: 1e-8)
    dx, dy, p = 545, 544, 1
    op = sipg.Operator(dx, dy, p, sipg.pen_sigma(p), sipg.F64)
    V = np.zeros((dy + 1, dx + 1))
    V[1:dy, 1:dx] = np.random.default_rng(7).uniform(-1, 1, (dy - 1, dx - 1))
    tl, tr, bl, br = V[:-1, :-1], V[:-1, 1:], V[1:, :-1], V[1:, 1:]
    u = np.stack([bl, tl, br, tr]).reshape(-1)            # p = 1: the nodes are the vertices, (i1, i2) order
    ud, rd, z1, z2 = op.vector(), op.vector(), op.vector(), op.vector()
    op.upload(u, ud)
    assert op.apply(ud, rd) == sipg.OK
    op.prec_apply(rd, z1)
    op.prec2_apply(rd, z2)
    coarse = op.download(z2) - op.download(z1)
    assert np.max(np.abs(coarse - u)) <= 1e-8 * np.max(np.abs(u))
