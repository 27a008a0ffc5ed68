"""The workloads that this framework's speed is judged on.

Each case is one pass through the public entry points of the `sipg` package,
as a program that holds its vectors in torch tensors calls them: the operator
apply on its own (every Krylov method is built on it), the solvers from x = 0
to a 1e-10 relative residual, a batch of uneven problems, and a server that
is handed a burst of requests.  The sizes are those of the benchmark's
configurations and the ranges around them.

exact() rebuilds each result in 64 bits from the discrete problem itself.
The SIPG matrix of a uniform mesh is the Kronecker sum A1 (x) W + W (x) A1 of
its one-dimensional matrix A1 and the diagonal of quadrature weights W, so an
apply is two passes along the mesh lines, and a solve is a fast
diagonalisation with iterative refinement.
"""
import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "cuda-sipg-matrix-free_amd"))
import sipg  # noqa: E402

TOL = 1e-10


class Vec:
    """A torch tensor as the vector argument of a sipg call."""

    def __init__(self, t):
        self.t = t
        self.ptr = ctypes.c_void_p(t.data_ptr())


def listed():
    return [
        # the smallest call: one operator application on the 8 x 8, p = 3 problem, where the launch is the cost
        {"name": "apply-8-p3-f64", "kind": "apply", "dimx": 8, "dimy": 8, "p": 3, "f32": False},
        # the operator at the benchmark's size, 5.3 million unknowns
        {"name": "apply-256-p8-f64", "kind": "apply", "dimx": 256, "dimy": 256, "p": 8, "f32": False},
        # the same with vectors of 680 MB, past every cache
        {"name": "apply-1024-p8-f64", "kind": "apply", "dimx": 1024, "dimy": 1024, "p": 8, "f32": False},
        # the single-precision operator of the high-degree mixed-precision solve
        {"name": "apply-128-p15-f32", "kind": "apply", "dimx": 128, "dimy": 128, "p": 15, "f32": True},
        # an odd degree on a rectangular mesh that no block size divides
        {"name": "apply-201x150-p7-f64", "kind": "apply", "dimx": 201, "dimy": 150, "p": 7, "f32": False},
        # the highest degree that the served requests have, on a ragged mesh
        {"name": "apply-131x77-p12-f64", "kind": "apply", "dimx": 131, "dimy": 77, "p": 12, "f32": False},
        # the smallest solve: the reference's own conjugate gradients on 1,024 unknowns
        {"name": "cg-8-p3", "kind": "cg", "dim": 8, "p": 3, "kmin": 4, "kmax": 4, "mmax": 4},
        # the reference's conjugate gradients on a middle size
        {"name": "cg-64-p6", "kind": "cg", "dim": 64, "p": 6, "kmin": 4, "kmax": 4, "mmax": 4},
        # the headline: 256 x 256 elements of degree 8 to 1e-10 by the two-level solver
        {"name": "pcg2-256-p8", "kind": "pcg2", "dim": 256, "p": 8, "kmin": 4, "kmax": 4, "mmax": 4},
        # mixed precision at high degree: FP32 cycles inside FP64 refinement
        {"name": "mixed-128-p15", "kind": "mixed", "dim": 128, "p": 15, "kmin": 1, "kmax": 8, "mmax": 12},
        # many uneven problems at once: side 4..64, degree 2..10
        {"name": "batch-128", "kind": "batch", "count": 128, "side": 64, "pmax": 10, "mix": 4},
        # a burst of requests to the server: side 8..128 by its logarithm, degree 2..12
        {"name": "serve-24", "kind": "serve", "count": 24, "side": 128, "pmax": 12, "mix": 24301},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["apply"] * 5 + ["cg", "pcg", "pcg2", "pcg2", "mixed", "batch", "serve"])
    if kind == "apply":
        p = rng.randint(1, 16) if rng.random() < 0.9 else rng.randint(17, 32)
        while True:
            dimx, dimy = _log_int(rng, 4, 1024), _log_int(rng, 4, 1024)
            if dimx * dimy * (p + 1) ** 2 <= 1024 * 1024 * 81:
                return {"kind": kind, "dimx": dimx, "dimy": dimy, "p": p, "f32": rng.random() < 0.3}
    if kind in ("batch", "serve"):
        return {"kind": kind, "count": rng.randint(24, 128) if kind == "batch" else rng.randint(8, 24),
                "side": rng.randint(32, 64) if kind == "batch" else rng.randint(48, 128), "pmax": rng.randint(6, 10),
                "mix": rng.randint(1, 99999)}
    # sides and degrees whose attainable residual in 64 bits lies well below the tolerance
    p = rng.randint(2, 8) if kind == "cg" else rng.randint(8, 15) if kind == "mixed" else rng.randint(2, 12)
    dim = _log_int(rng, 8, {"cg": 64, "pcg": 80, "pcg2": 160 if p <= 8 else 100, "mixed": 100}[kind])
    return {"kind": kind, "dim": dim, "p": p, "kmin": 1, "kmax": 4, "mmax": 4}


def _shapes(case):
    """Mesh sides and degrees of a batch or a burst (fixed by the case; the forcing comes from the seed)."""
    rng = random.Random(case["mix"])
    if case["kind"] == "batch":
        return [(rng.randint(4, case["side"]), rng.randint(2, case["pmax"])) for _ in range(case["count"])]
    return [(_log_int(rng, 8, case["side"]), rng.randint(2, case["pmax"])) for _ in range(case["count"])]


def _forcing(seed, k, kmin, kmax, mmax):
    """Amplitudes in (-1, 1) and wave numbers in 1..mmax of kmin..kmax Fourier modes."""
    rng = random.Random(1000003 * seed + k)
    nm = rng.randint(kmin, kmax)
    return ([rng.uniform(-1.0, 1.0) for _ in range(nm)], [rng.randint(1, mmax) for _ in range(nm)],
            [rng.randint(1, mmax) for _ in range(nm)])


def _input(case, seed):
    """The operand of an apply: what a solver hands to it has all scales, here uniform values."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    n = case["dimx"] * case["dimy"] * (case["p"] + 1) ** 2
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float32 if case["f32"] else torch.float64) * 2 - 1


def prepare(case, seed):
    kind = case["kind"]
    if kind == "apply":
        op = sipg.Operator(case["dimx"], case["dimy"], case["p"], sipg.pen_sigma(case["p"]),
                           sipg.F32 if case["f32"] else sipg.F64)
        x = _input(case, seed)
        return {"kind": kind, "op": op, "x": Vec(x), "y": Vec(torch.empty_like(x))}
    if kind == "batch":
        shapes = _shapes(case)
        dims, ps = [d for d, _ in shapes], [p for _, p in shapes]
        stream = torch.cuda.Stream()
        batch = sipg.Batch(dims, dims, ps, [sipg.pen_sigma(p) for p in ps], stream=stream.cuda_stream)
        b = Vec(torch.empty(batch.n, dtype=torch.float64, device="cuda"))
        torch.cuda.synchronize()
        for i in range(len(shapes)):
            batch.rhs_fourier(i, _forcing(seed, i, 1, 4, 4), b)
        batch.tune()
        return {"kind": kind, "batch": batch, "stream": stream, "b": b, "x": Vec(torch.empty_like(b.t))}
    if kind == "serve":
        server = sipg.Server(16e9)
        sipg.check(server.set_method(sipg.METHOD_PCG), "set_method")
        requests = [(d, p, sipg.pen_sigma(p), _forcing(seed, k, 1, 4, 4)) for k, (d, p) in enumerate(_shapes(case))]
        return {"kind": kind, "server": server, "requests": requests}
    op = sipg.Operator(case["dim"], case["dim"], case["p"], sipg.pen_sigma(case["p"]), sipg.F64)
    b = Vec(torch.empty(op.n, dtype=torch.float64, device="cuda"))
    op.rhs_fourier(_forcing(seed, 0, case["kmin"], case["kmax"], case["mmax"]), b)
    return {"kind": kind, "op": op, "b": b, "x": Vec(torch.empty_like(b.t))}


def run(state):
    kind = state["kind"]
    if kind == "apply":
        sipg.check(state["op"].apply(state["x"], state["y"]), "apply")
        return state["y"].t
    if kind == "batch":
        x = state["x"]
        with torch.cuda.stream(state["stream"]):
            x.t.zero_()
        state["batch"].pcg(x, state["b"], TOL, sipg.TOL_REL, maxit=20000, replace_factor=3e-3)
        return x.t
    if kind == "serve":
        server, ids, done = state["server"], {}, {}
        for k, (d, p, pen, modes) in enumerate(state["requests"]):
            ids[server.submit(d, p, pen, modes, TOL, maxit=30000)] = k
        while len(done) < len(ids):
            server.progress()
            while (got := server.take_ex(-1)) is not None:
                done[ids[got[0]]] = got[2]
        return [done[k] for k in range(len(done))]
    op, x, b = state["op"], state["x"], state["b"]
    x.t.zero_()
    if kind == "cg":
        op.cg_ex(x, b, TOL, sipg.TOL_REL, maxit=30000, replace_factor=3e-3)
    elif kind == "pcg":
        op.pcg(x, b, TOL, sipg.TOL_REL, maxit=30000, replace_factor=3e-3)
    elif kind == "pcg2":
        op.pcg2(x, b, TOL, sipg.TOL_REL, maxit=30000, replace_factor=1e-2)
    else:
        op.pcg2_mixed(x, b, TOL, sipg.TOL_REL, maxit=60000, replace_factor=1e-1, restart=1)
    return x.t


def _sizes(case):
    """(unknowns, degree) of each problem in the case."""
    if case["kind"] == "apply":
        return [(case["dimx"] * case["dimy"] * (case["p"] + 1) ** 2, case["p"])]
    shapes = _shapes(case) if case["kind"] in ("batch", "serve") else [(case["dim"], case["p"])]
    return [(d * d * (p + 1) ** 2, p) for d, p in shapes]


def work(case):
    """One read of the operand or right-hand side and one write of the result; the contractions of one apply."""
    es = 4 if case.get("f32") else 8
    sizes = _sizes(case)
    return {"bytes": 2 * es * sum(n for n, _ in sizes), "flops": sum(4 * (p + 1) * n for n, p in sizes)}


# ---- the same results in 64 bits, without the framework ------------------


def _gll(p):
    """GLL nodes and weights, and D[i, k] = phi_i'(z_k)."""
    c = np.zeros(p + 1)
    c[p] = 1.0
    leg = np.polynomial.legendre
    z = np.concatenate([[-1.0], np.sort(leg.legroots(leg.legder(c)).real) if p > 1 else [], [1.0]])
    d1, d2 = leg.legder(c), leg.legder(c, 2)
    for _ in range(3):                                        # Newton steps on P_p' for the inner nodes
        if p > 1:
            z[1:-1] -= leg.legval(z[1:-1], d1) / leg.legval(z[1:-1], d2)
    w = 2.0 / (p * (p + 1) * leg.legval(z, c) ** 2)
    lam = np.array([1.0 / np.prod([z[j] - z[k] for k in range(p + 1) if k != j]) for j in range(p + 1)])
    D = np.zeros((p + 1, p + 1))
    for k in range(p + 1):
        for i in range(p + 1):
            if i != k:
                D[i, k] = lam[i] / lam[k] / (z[k] - z[i])
        D[k, k] = -D[:, k].sum()
    return z, w, D


def _line(u, p, pen, low_is_first):
    """The one-dimensional SIPG matrix along a mesh line, without the cross weights: u is (..., elements, p + 1)."""
    _, w, D = _gll(p)
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=u.device, dtype=u.dtype)  # noqa: E731
    if not low_is_first:                                      # elements numbered against the coordinate
        u = u.flip(-2)
    d0, dp = t(D[:, 0]), t(D[:, p])
    y = u @ t((D * w) @ D.T)
    u0, up, g0, gp = u[..., 0], u[..., p], u @ d0, u @ dp
    jump, mean, weight = u0.clone(), g0.clone(), torch.full_like(u0, pen)       # at each element's lower face
    jump[..., 1:] = 0.5 * (u0[..., 1:] - up[..., :-1])
    mean[..., 1:] = 0.5 * (g0[..., 1:] + gp[..., :-1])
    weight[..., 1:] = 2 * pen
    y += jump[..., None] * d0
    y[..., 0] += mean + weight * jump
    jump, mean, weight = up.clone(), gp.clone(), torch.full_like(up, pen)       # at each element's upper face
    jump[..., :-1] = 0.5 * (up[..., :-1] - u0[..., 1:])
    mean[..., :-1] = 0.5 * (gp[..., :-1] + g0[..., 1:])
    weight[..., :-1] = 2 * pen
    y -= jump[..., None] * dp
    y[..., p] += weight * jump - mean
    return y if low_is_first else y.flip(-2)


def _apply(x, dimx, dimy, p, pen):
    """A x for a vector in the device layout (element-major, rows from the top, node = x index * (p+1) + y index)."""
    w = torch.as_tensor(_gll(p)[1], device=x.device)
    u = x.view(dimy, dimx, p + 1, p + 1)
    yx = _line(u.permute(0, 3, 1, 2), p, pen, True).permute(0, 2, 3, 1) * w
    yy = _line(u.permute(1, 2, 0, 3), p, pen, False).permute(2, 0, 1, 3) * w[:, None]
    return (yx + yy).reshape(-1)


def _nodes(dim, p):
    z = _gll(p)[0]
    e = np.arange(dim)[:, None]
    return ((e + 0.5 * (z + 1.0)) / dim).reshape(-1)


def _grid_to_device(a, dim, p):
    """(x index, y index) over the whole mesh -> the device layout."""
    n1 = p + 1
    return np.ascontiguousarray(a.reshape(dim, n1, dim, n1)[:, :, ::-1].transpose(2, 0, 1, 3)).reshape(-1)


def _solution(dim, p, modes):
    """The discrete solution of the Fourier problem in the device layout, or None where this would take too long."""
    s = _nodes(dim, p)
    if dim * (p + 1) > 1300:
        if p < 8:
            return None
        # the discretisation error of such meshes lies far below the solvers' tolerance
        u = sum(a * np.outer(np.sin(m * np.pi * s), np.sin(n * np.pi * s)) for a, m, n in zip(*modes))
        return _grid_to_device(u, dim, p)
    _, w, _ = _gll(p)
    f = sum(a * np.pi ** 2 * (float(m) ** 2 + float(n) ** 2) * np.outer(np.sin(m * np.pi * s), np.sin(n * np.pi * s))
            for a, m, n in zip(*modes))
    W = np.tile(w, dim)
    b = f * np.outer(W, W) * (0.5 / dim) ** 2
    pen = 5.0 * (p + 1) ** 2
    N = dim * (p + 1)

    def line(v):                                              # A1 v for the columns of v
        t = torch.from_numpy(np.ascontiguousarray(v.T)).view(-1, dim, p + 1)
        return _line(t, p, pen, True).reshape(-1, N).T.numpy()

    A1 = line(np.eye(N))
    r = np.sqrt(W)
    lam, V = np.linalg.eigh(0.5 * (A1 + A1.T) / np.outer(r, r))
    S = V / r[:, None]
    x = np.zeros_like(b)
    for _ in range(4):
        res = b - (line(x) * W + W[:, None] * line(x.T).T)
        x += S @ ((S.T @ res @ S) / (lam[:, None] + lam)) @ S.T
    return _grid_to_device(x, dim, p)


def exact(case, seed):
    kind = case["kind"]
    if kind == "apply":
        return _apply(_input(case, seed).double(), case["dimx"], case["dimy"], case["p"], 5.0 * (case["p"] + 1) ** 2)
    if kind in ("batch", "serve"):
        got = [_solution(d, p, _forcing(seed, k, 1, 4, 4)) for k, (d, p) in enumerate(_shapes(case))]
        if kind == "batch":
            return torch.from_numpy(np.concatenate(got))
        # a served solution comes in the reference's order: node-major, elements innermost
        return [None if v is None else np.ascontiguousarray(v.reshape(d * d, -1).T).reshape(-1)
                for v, (d, _) in zip(got, _shapes(case))]
    v = _solution(case["dim"], case["p"], _forcing(seed, 0, case["kmin"], case["kmax"], case["mmax"]))
    return None if v is None else torch.from_numpy(v)
