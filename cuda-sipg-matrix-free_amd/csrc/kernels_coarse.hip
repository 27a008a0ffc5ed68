// kernels_coarse.hip -- the coarse level of the two-level preconditioner.
//
// M2^-1 r = M_BJ^-1 r + P0^T A0^-1 P0 r: the block-Jacobi preconditioner of
// kernels_pcg.hip plus an exact solve on V0, the continuous bilinear (Q1)
// functions on the element vertices that vanish on the boundary.  P0^T
// interpolates vertex values bilinearly into every node of the adjacent
// elements; P0 is its transpose.  A continuous function has no jumps, so on
// V0 every face term of the SIPG form vanishes and A0 = P0 A P0^T is the Q1
// stiffness matrix, with the 1-D factors K = tridiag(-1, 2, -1) and the GLL
// quadrature mass M = tridiag(m1, 2 m0, m1) (exact for p >= 2: 1/6, 1/3;
// lumped for p = 1): A0 = Kx (x) My + Mx (x) Ky on the (dimy-1) x (dimx-1)
// interior vertices.  Both factors are diagonalised by the discrete sine
// transform Q_jk = sqrt(2/dim) sin(j k pi / dim), so
//
//   A0^-1 S = Qy [ (Qy S Qx) ./ Lambda ] Qx,
//   Lambda_ab = lamKy_a lamMx_b + lamMy_a lamKx_b
//
// four dense products of (dim-1)^2 matrices.  One coarse step per
// preconditioner application:
//   restrict  -- per element the four corner-weighted sums of r (E4); for
//                the standard penalty the block-Jacobi kernel forms them
//                from its own read of r (pcg_rz_kernel with RESTR), and
//                restrict_kernel runs only elsewhere
//   4 x gemm  -- the DST solve (dst_gemm_kernel, each product over half
//                the k range); the first gathers S(a,b), the sum of the
//                four elements meeting at interior vertex (a,b) (vertex
//                (a,b) sits at x = b hx, y = 1 - a hy; element (row, col)
//                has its top-left corner at vertex (row, col)), as it loads
//                it; the last writes C into the zero-bordered vertex grid
//                Cpad and the block partials of S.C
// and the p update interpolates Cpad into every node (p = z + P0^T C + beta p)
// with r.z = r.z_BJ + S.C.
//
// Large vertex grids (kBlasVertices and up: from about 541 x 541 elements)
// take the four products as rocBLAS FP64 GEMMs instead, with the
// gather, the 1/Lambda scaling and the S.C partials as small kernels of
// their own: the dense products grow as the cube of the mesh side, and the
// folded kernel, which reads its operands from L2 once per 16 x 16 tile, then
// is bound by those reads.  rocBLAS is opened on first use (dlopen); without
// it the folded kernel runs at every size.
#include "sipg_internal.hpp"
#include "partials.hpp"

#include <dlfcn.h>
#include <rocblas/rocblas.h>

#include <algorithm>
#include <map>

namespace sipg_internal {

namespace {

constexpr int VT = kVecThreads;
// elements per restrict workgroup: their tiles fill at most 32 KiB of LDS
template <int P>
constexpr int rne() { return 4096 / ((P + 1) * (P + 1)) < 32 ? 4096 / ((P + 1) * (P + 1)) : 32; }
constexpr int GT = 16;           // gemm output tile (GT x GT)
// waves per tile, which split the k range: more where an operand value is
// eight scattered loads (MODE 3)
__host__ __device__ constexpr int dst_waves(int mode) { return mode == 3 ? 16 : 8; }

typedef double dd4 __attribute__((ext_vector_type(4)));

// Tiles of GT indices of one parity in 0..n-1: the even indices, and all.
__host__ __device__ constexpr int dst_tiles_even(int n) { return ((n + 1) / 2 + GT - 1) / GT; }
__host__ __device__ constexpr int dst_tiles(int n) { return dst_tiles_even(n) + (n / 2 + GT - 1) / GT; }

// E4[c * noe + e] = sum_nodes r(e, i1, i2) wx_c(i1) wy_c(i2); corner c = 0
// bottom-left, 1 bottom-right, 2 top-left, 3 top-right; wx = 1 - xi or xi,
// wy = 1 - xi or xi (xi = (z+1)/2: x from the element's left, y from its
// bottom).
template <typename T, int P>
__global__ __launch_bounds__(VT) void restrict_kernel(const T *__restrict__ r, const double *__restrict__ xi,
                                                      int64_t noe, double *__restrict__ E4) {
    constexpr int N1 = P + 1, NQ = N1 * N1, RNE = rne<P>();
    __shared__ double tile[RNE * NQ];
    __shared__ double sx[N1];
    if (threadIdx.x < N1) sx[threadIdx.x] = xi[threadIdx.x];
    const int64_t e0 = (int64_t)blockIdx.x * RNE;
    const int ne = (int)min<int64_t>(RNE, noe - e0);
    const T *src = r + e0 * NQ;
    for (int i = threadIdx.x; i < ne * NQ; i += VT) tile[i] = (double)src[i];
    __syncthreads();
    const int t = threadIdx.x;
    if (t < 4 * ne) {
        const int el = t >> 2, c = t & 3;
        const double *u = tile + el * NQ;
        double acc = 0.0;
        for (int i1 = 0; i1 < N1; ++i1) {
            double line = 0.0;
#pragma unroll
            for (int i2 = 0; i2 < N1; ++i2) line += u[i1 * N1 + i2] * ((c & 2) ? sx[i2] : 1.0 - sx[i2]);
            acc += line * ((c & 1) ? sx[i1] : 1.0 - sx[i1]);
        }
        E4[(int64_t)c * noe + e0 + el] = acc;
    }
}

// The sine matrix Q (n x n, symmetric) has Q[j][n-1-k] = (-1)^j Q[j][k],
// so each product folds its k range in half: with h = n / 2,
//   (Q X)[j][m] = sum_{k<h} Q[j][k] (X[k][m] +- X[n-1-k][m]) (+ Q[j][h] X[h][m], n odd)
//   (X Q)[m][j] = sum_{k<h} (X[m][k] +- X[m][n-1-k]) Q[k][j]  (+ X[m][h] Q[h][j], n odd)
// with + for even j and - for odd j.  The products run on the FP64 matrix
// cores (v_mfma_f64_16x16x4f64: lane l holds A[l % 16][l / 16],
// B[l / 16][l % 16] and, in register r, D[4 r + l / 16][l % 16]).  An output
// tile takes 16 indices j of one parity (j = 2 t + parity), so that one fold
// of X serves the whole tile; the other dimension is cut plainly.  One
// workgroup per tile; its waves (KS of them) take the k blocks of four in
// turn, straight from memory (the operands are a few hundred KB and
// sit in L2), and the partial tiles are added in LDS in a fixed order.
//
// Bound: latency (33 MFLOP at 255 x 255).  All loads of a wave's k blocks
// are issued before the first product, so that a product is one round trip
// to L2, the matrix instructions and one LDS exchange; the previous kernel
// staged both operands in LDS and read two LDS values per multiply-add on
// the vector ALUs.  255 x 255: 8.8 + 6.9 + 7.2 + 6.9 -> 5.9 + 4.9 + 5.0 + 4.9 us for the four
// products; 127 x 127: 25.7 -> 18.7 us in all.
//   SIDE 0: out (n x N) = Q X (X: n x N);  SIDE 1: out (M x n) = X Q (X: M x n)
//   MODE 0: out = the product
//   MODE 1: out = product .* W               (W the 1/Lambda table)
//   MODE 2: Cpad[(i+1)*(cols+2) + j+1] = product, and per-workgroup partials of
//           sum product .* W into part[blockIdx.y * gridDim.x + blockIdx.x]
//   MODE 3: as MODE 0 with X = S gathered from the corner sums E4 (X is E4,
//           n + 1 by N + 1 elements; the first tile row also stores S into
//           W).  On SIDE 0, where a load covers 16 neighbouring vertices: the
//           rows of E4 are a power of two apart on the usual meshes, and four
//           vertices from each of 16 rows (SIDE 1) took 10.9 against 5.9 us.
template <int SIDE, int MODE>
__global__ __launch_bounds__(64 * dst_waves(MODE)) void dst_gemm_kernel(const double *__restrict__ X,
                                                          const double *__restrict__ Q, int M, int n, int N,
                                                          double *__restrict__ W, double *__restrict__ out,
                                                          double *__restrict__ part, const cg_state *st, int slot) {
    // inside a solve: nothing to do once it has finished (the launches
    // queued past the finish run as no-ops)
    if (st && (st->s[slot].done | st->err)) return;
    constexpr int KS = dst_waves(MODE);
    constexpr int KB = MODE == 3 ? 2 : 4;               // k blocks in flight per wave (n = 255: all of them)
    __shared__ double ps[KS][GT][GT + 1];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, lk = lane >> 4;
    const int rows = SIDE == 0 ? n : M, cols = SIDE == 0 ? N : n;
    const int h = n / 2, kh = h + (n & 1);              // folded length (with the middle)
    // the folded dimension's tiles: the even indices first, then the odd ones
    const int te = dst_tiles_even(n);
    const int tf = SIDE == 0 ? blockIdx.y : blockIdx.x;
    const int par = tf >= te ? 1 : 0, f0 = 2 * GT * (par ? tf - te : tf) + par, fs = 2;
    const int r0 = SIDE == 0 ? f0 : (int)blockIdx.y * GT, rs = SIDE == 0 ? fs : 1;
    const int c0 = SIDE == 0 ? (int)blockIdx.x * GT : f0, cs = SIDE == 0 ? 1 : fs;
    const double sgn = par ? -1.0 : 1.0;
    // X element (m, k): k in the folded direction
    const int dimx = N + 1;
    const int64_t noe = (int64_t)dimx * (n + 1);
    auto xval = [&](int m, int k) -> double {
        if (MODE == 3) {
            const int64_t a = (int64_t)k * dimx + m, b = a + dimx;
            return (X[1 * noe + a] + X[0 * noe + a + 1]) + (X[3 * noe + b] + X[2 * noe + b + 1]);
        }
        return SIDE == 0 ? X[(int64_t)k * N + m] : X[(int64_t)m * n + k];
    };
    // this lane's row of Q (its folded index) and its line of X
    const int jq = f0 + fs * li, mx = (SIDE == 0 ? c0 : r0) + li;
    const bool qok = jq < n, xok = mx < (SIDE == 0 ? N : M);
    const double *Qj = Q + (int64_t)(qok ? jq : 0) * n;
    const int m = xok ? mx : 0;
    const int nkb = (kh + 3) / 4;
    dd4 acc = {0.0, 0.0, 0.0, 0.0};
    for (int b0 = w; b0 < nkb; b0 += KS * KB) {
        double q[KB], xa[KB], xb[KB];
#pragma unroll
        for (int i = 0; i < KB; ++i) {
            // (clamped: blocks past the end are loaded from the last k and weighted zero)
            const int k = min(4 * (b0 + KS * i) + lk, kh - 1);
            q[i] = Qj[k];
            xa[i] = xval(m, k);
            xb[i] = xval(m, n - 1 - k);
        }
#pragma unroll
        for (int i = 0; i < KB; ++i) {
            const int k = 4 * (b0 + KS * i) + lk;
            if (MODE == 3 && blockIdx.y == 0 && xok && k < kh) {
                W[(int64_t)k * N + m] = xa[i];
                W[(int64_t)(n - 1 - k) * N + m] = xb[i];
            }
            // the middle (n odd) enters once
            const double xf = k < h ? xa[i] + sgn * xb[i] : xa[i];
            const double qv = qok && k < kh ? q[i] : 0.0, xv = xok && k < kh ? xf : 0.0;
            acc = SIDE == 0 ? __builtin_amdgcn_mfma_f64_16x16x4f64(qv, xv, acc, 0, 0, 0)
                            : __builtin_amdgcn_mfma_f64_16x16x4f64(xv, qv, acc, 0, 0, 0);
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) ps[w][4 * r + lk][li] = acc[r];
    __syncthreads();
    const int ty = threadIdx.x / GT, tx = threadIdx.x % GT;
    const int gr = r0 + rs * ty, gc = c0 + cs * tx;
    double dot = 0.0;
    if (ty < GT && gr < rows && gc < cols) {            // four waves finish the tile
        double v = 0.0;
#pragma unroll
        for (int i = 0; i < KS; ++i) v += ps[i][ty][tx];
        const int64_t oo = (int64_t)gr * cols + gc;
        if (MODE == 0 || MODE == 3) out[oo] = v;
        if (MODE == 1) out[oo] = v * W[oo];
        if (MODE == 2) {
            out[(int64_t)(gr + 1) * (cols + 2) + gc + 1] = v;
            dot = v * W[oo];
        }
    }
    if (MODE == 2) {
        __shared__ double red[KS];
        dot = wave_total(dot);
        if (lane == 0) red[w] = dot;                    // (waves 4 and up: zero)
        __syncthreads();
        if (threadIdx.x == 0) part[blockIdx.y * gridDim.x + blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
    }
}

// bilinear interpolation of the zero-bordered vertex grid Cpad
// ((dimy+1) x (dimx+1)) at node (i1, i2) of element e
template <int P>
__device__ __forceinline__ double prolong(const double *__restrict__ Cpad, const double *sx, int dimx, int e,
                                          int i1, int i2) {
    const int row = e / dimx, col = e - (e / dimx) * dimx;
    const int ld = dimx + 1;
    const double tl = Cpad[row * ld + col], tr = Cpad[row * ld + col + 1];
    const double bl = Cpad[(row + 1) * ld + col], br = Cpad[(row + 1) * ld + col + 1];
    const double x = sx[i1], y = sx[i2];
    return (1.0 - y) * ((1.0 - x) * bl + x * br) + y * ((1.0 - x) * tl + x * tr);
}

// p += P0^T C (the start of a solve: p = z_BJ was written by the
// preconditioner), or with z given: z += P0^T C (a plain application)
template <typename T, int P>
__global__ __launch_bounds__(VT) void add_coarse_kernel(T *__restrict__ v, const double *__restrict__ Cpad,
                                                        const double *__restrict__ xi, int dimx, int64_t n) {
    constexpr int N1 = P + 1, NQ = N1 * N1;
    __shared__ double sx[N1];
    if (threadIdx.x < N1) sx[threadIdx.x] = xi[threadIdx.x];
    __syncthreads();
    for (int64_t i = (int64_t)blockIdx.x * VT + threadIdx.x; i < n; i += (int64_t)gridDim.x * VT) {
        const int e = (int)(i / NQ), node = (int)(i - (int64_t)e * NQ);
        const int i1 = node / N1, i2 = node - (node / N1) * N1;
        v[i] = (T)((double)v[i] + prolong<P>(Cpad, sx, dimx, e, i1, i2));
    }
}

// Elements per group of the kernels that interpolate from the vertex grid:
// about 4096 values, a multiple of four elements (so that a group's values
// divide into 16-byte vectors).
template <int P>
constexpr int interp_elems() {
    constexpr int ne = (4096 / ((P + 1) * (P + 1))) & ~3;
    return ne < 4 ? 4 : (ne > 256 ? 256 : ne);
}

// pcg_update_p_kernel with the coarse level: r.z = sum(prz) + sum(pc)
// (the block-Jacobi part and S.C) and p = z + P0^T C + beta p.
//
// Bound: memory, five vector passes (x, p, z in; x, p out).  A workgroup
// takes groups of about 4096 values of whole elements; the interpolation
// along each element line x = const (the value at the line's lower end and
// its rise) is formed once per line in LDS, so that a value costs one fused
// multiply-add instead of a bilinear interpolation with four scattered
// vertex loads, and the streams move 16 bytes per lane.  alpha is the one
// that the block-Jacobi kernel of this iteration recorded in the slot.
// Measured per launch, one value per lane with the interpolation at every
// node -> this: 16x16-node FP32 elements (128 x 128) 30.1 -> 16.6 us,
// FP64 p = 8 (256 x 256) 44.6 -> 38.2 us.
template <typename T, int P>
__global__ __launch_bounds__(VT) void pcg2_update_p_kernel(T *__restrict__ x, T *__restrict__ p,
                                                           const T *__restrict__ z, int64_t noe,
                                                           const double *__restrict__ prr,
                                                           const double *__restrict__ prz, int np,
                                                           const double *__restrict__ pc, int npc,
                                                           const double *__restrict__ Cpad,
                                                           const double *__restrict__ xi, int dimx, cg_state *st,
                                                           int slot, T *__restrict__ xlo) {
    constexpr int N1 = P + 1, NQ = N1 * N1, NEG = interp_elems<P>(), VL = 16 / (int)sizeof(T);
    static_assert(NEG * NQ % VL == 0, "a group divides into vectors");
    __shared__ double sx[N1];
    __shared__ double lo[NEG * N1], up[NEG * N1];       // per line: value at its lower end, rise to the upper one
    const cg_slot cur = st->s[slot];
    if (cur.done | st->err) {
        if (blockIdx.x == 0 && threadIdx.x == 0) st->s[slot ^ 1] = cur;   // carry forward
        return;
    }
    if (threadIdx.x < N1) sx[threadIdx.x] = xi[threadIdx.x];
    double sum[3];
    multi_sum<VT, 3>({prr, prz, pc}, {np, np, npc}, sum);      // its barrier publishes sx
    const double rr_new = sum[0], rz_new = sum[1] + sum[2];
    const bool replaced = (cur.flags & kSlotReplaced) != 0;
    const double beta_d = (cur.flags & kSlotRestart) ? 0.0 : rz_new / cur.rz;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const bool met = !(sqrt(rr_new) > st->stop);
        const bool need_true = st->true_stop && !replaced;
        cg_slot nx;
        nx.rr = rr_new;
        nx.alpha = 0.0;
        nx.beta = beta_d;
        nx.pAp = 0.0;
        nx.rz = rz_new;
        nx.it = cur.it + 1;
        nx.done = ((met && !need_true) || nx.it >= st->maxit) ? 1 : 0;
        nx.checked = replaced ? 1 : 0;
        nx.flags = (met && need_true) ? kSlotWantCheck : 0;
        st->s[slot ^ 1] = nx;
        if (replaced) st->rr_ref = rr_new;
        if (!isfinite(rr_new) || !isfinite(rz_new)) st->err = 3;
        else if (!(rz_new > 0.0) && rr_new > 0.0) st->err = 2;   // M not positive on r
    }
    const T alpha = (T)cur.alpha;
    const T beta = (T)beta_d;
    const int ld = dimx + 1;
    const int64_t ngroup = (noe + NEG - 1) / NEG;
    for (int64_t g = blockIdx.x; g < ngroup; g += gridDim.x) {
        const int64_t e0 = g * NEG;
        const int ne = (int)min<int64_t>(NEG, noe - e0);
        for (int l = threadIdx.x; l < ne * N1; l += VT) {
            const int el = l / N1, i1 = l - el * N1;
            const int e = (int)e0 + el, row = e / dimx, col = e - row * dimx;
            const double *c = Cpad + (int64_t)row * ld + col;
            const double t = sx[i1];
            const double top = (1.0 - t) * c[0] + t * c[1], bot = (1.0 - t) * c[ld] + t * c[ld + 1];
            lo[l] = bot;
            up[l] = top - bot;
        }
        __syncthreads();
        const int n = ne * NQ;
        T *xg = x + e0 * NQ, *pg = p + e0 * NQ, *lg = xlo + (xlo ? e0 * NQ : 0);
        const T *zg = z + e0 * NQ;
#pragma unroll 2
        for (int i = VL * threadIdx.x; i < n; i += VL * VT) {
            if (i + VL <= n) {
                T pv[VL], zv[VL], xv[VL];
                load_vec<T, VL>(pg + i, pv);
                load_vec<T, VL>(zg + i, zv);
                if (!replaced) {
                    load_vec<T, VL>(xg + i, xv);
                    if (xlo) {
                        T xl[VL];
                        load_vec<T, VL>(lg + i, xl);
#pragma unroll
                        for (int q = 0; q < VL; ++q) comp_axpy(xv[q], xl[q], alpha, pv[q]);
                        store_vec<T, VL>(lg + i, xl);
                    } else {
#pragma unroll
                        for (int q = 0; q < VL; ++q) xv[q] = xv[q] + alpha * pv[q];
                    }
                    store_vec<T, VL>(xg + i, xv);
                }
#pragma unroll
                for (int q = 0; q < VL; ++q) {
                    const int l = (i + q) / N1, i2 = i + q - l * N1;
                    pv[q] = (T)((double)zv[q] + (lo[l] + sx[i2] * up[l])) + beta * pv[q];
                }
                store_vec<T, VL>(pg + i, pv);
            } else {                                     // the mesh's last values
                for (int q = i; q < n; ++q) {
                    const int l = q / N1, i2 = q - l * N1;
                    const T pi = pg[q];
                    if (!replaced) {
                        if (xlo) comp_axpy(xg[q], lg[q], alpha, pi);
                        else xg[q] = xg[q] + alpha * pi;
                    }
                    pg[q] = (T)((double)zg[q] + (lo[l] + sx[i2] * up[l])) + beta * pi;
                }
            }
        }
        __syncthreads();                                 // the lines are free for the next group
    }
}

struct coarse_args {
    const void *r = nullptr;
    void *v = nullptr, *x = nullptr, *xlo = nullptr;
    const void *z = nullptr;
    const double *xi = nullptr, *Cpad = nullptr, *prr = nullptr, *prz = nullptr, *pc = nullptr;
    double *E4 = nullptr;
    int64_t noe = 0, n = 0;
    int dimx = 0, nblk = 0, np = 0, npc = 0, slot = 0;
    cg_state *st = nullptr;
    hipStream_t s = nullptr;
};

template <int P>
struct CoarseFns {
    template <typename T>
    static void restrict_(const void *r, const double *xi, int64_t noe, double *E4, hipStream_t s) {
        const int nb = (int)((noe + rne<P>() - 1) / rne<P>());
        hipLaunchKernelGGL((restrict_kernel<T, P>), dim3(nb), dim3(VT), 0, s, (const T *)r, xi, noe, E4);
    }
    template <typename T>
    static void add_(void *v, const double *Cpad, const double *xi, int dimx, int64_t n, int nblk, hipStream_t s) {
        hipLaunchKernelGGL((add_coarse_kernel<T, P>), dim3(nblk), dim3(VT), 0, s, (T *)v, Cpad, xi, dimx, n);
    }
    template <typename T>
    static void update_(const coarse_args &a) {
        const int nb = (int)std::min<int64_t>((a.noe + interp_elems<P>() - 1) / interp_elems<P>(), 2048);
        hipLaunchKernelGGL((pcg2_update_p_kernel<T, P>), dim3(nb), dim3(VT), 0, a.s, (T *)a.x, (T *)a.v,
                           (const T *)a.z, a.noe, a.prr, a.prz, a.np, a.pc, a.npc, a.Cpad, a.xi, a.dimx, a.st, a.slot,
                           (T *)a.xlo);
    }
};

template <int P>
int dispatch_p(int p, int dtype, int what, const coarse_args &a) {
    if (p != P) {
        if constexpr (P < kMaxDegree) return dispatch_p<P + 1>(p, dtype, what, a);
        else return SIPG_ERR_UNSUPPORTED;
    }
    using F = CoarseFns<P>;
    const bool f64 = dtype == SIPG_F64;
    if (what == 0) {
        if (f64) F::template restrict_<double>(a.r, a.xi, a.noe, a.E4, a.s);
        else F::template restrict_<float>(a.r, a.xi, a.noe, a.E4, a.s);
    } else if (what == 1) {
        if (f64) F::template add_<double>(a.v, a.Cpad, a.xi, a.dimx, a.n, a.nblk, a.s);
        else F::template add_<float>(a.v, a.Cpad, a.xi, a.dimx, a.n, a.nblk, a.s);
    } else {
        if (f64) F::template update_<double>(a);
        else F::template update_<float>(a);
    }
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

dim3 tile_grid(int M, int N) { return dim3((N + GT - 1) / GT, (M + GT - 1) / GT); }

// ---- the rocBLAS route for large vertex grids -------------------------------
// A whole two-level preconditioner application at p = 4, us, folded kernel /
// rocBLAS: 288 x 288 elements 53.4 / 67.2, 384 x 384 87.2 / 84.0, 448 x 448
// 108.9 / 121.2, 512 x 512 121.2 / 137.1, 640 x 640 234 / 175, 1024 x 1024
// 685 / 405.
constexpr int64_t kBlasVertices = 540 * 540;

// S(a, b): the sum of the four elements' corner sums meeting at interior
// vertex (a, b) (the gather of dst_gemm_kernel MODE 3), into S (nvy x nvx)
__global__ __launch_bounds__(VT) void gather_vertex_kernel(const double *__restrict__ E4, int nvy, int nvx,
                                                           double *__restrict__ S) {
    const int64_t nv = (int64_t)nvy * nvx;
    const int dimx = nvx + 1;
    const int64_t noe = (int64_t)dimx * (nvy + 1);
    for (int64_t i = (int64_t)blockIdx.x * VT + threadIdx.x; i < nv; i += (int64_t)gridDim.x * VT) {
        const int a = (int)(i / nvx) + 1, b = (int)(i - (i / nvx) * nvx) + 1;
        S[i] = (E4[1 * noe + (int64_t)(a - 1) * dimx + (b - 1)] + E4[0 * noe + (int64_t)(a - 1) * dimx + b]) +
               (E4[3 * noe + (int64_t)a * dimx + (b - 1)] + E4[2 * noe + (int64_t)a * dimx + b]);
    }
}

// T .*= W (the 1/Lambda table), nv values
__global__ __launch_bounds__(VT) void scale_kernel(double *__restrict__ T, const double *__restrict__ W, int64_t nv) {
    for (int64_t i = (int64_t)blockIdx.x * VT + threadIdx.x; i < nv; i += (int64_t)gridDim.x * VT) T[i] *= W[i];
}

// per-tile sums of S .* C (C the interior of the zero-bordered grid Cpad)
__global__ __launch_bounds__(GT * GT) void sc_partials_kernel(const double *__restrict__ S,
                                                              const double *__restrict__ Cpad, int nvy, int nvx,
                                                              double *__restrict__ part) {
    __shared__ double red[GT * GT / 64];
    const int tx = threadIdx.x % GT, ty = threadIdx.x / GT;
    const int gr = blockIdx.y * GT + ty, gc = blockIdx.x * GT + tx;
    double dot = 0.0;
    if (gr < nvy && gc < nvx) dot = S[(int64_t)gr * nvx + gc] * Cpad[(int64_t)(gr + 1) * (nvx + 2) + gc + 1];
    dot = wave_total(dot);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = dot;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.y * gridDim.x + blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// The three rocBLAS entry points used, resolved once from the installed
// library.
struct BlasFns {
    using create_t = rocblas_status (*)(rocblas_handle *);
    using stream_t = rocblas_status (*)(rocblas_handle, hipStream_t);
    using dgemm_t = rocblas_status (*)(rocblas_handle, rocblas_operation, rocblas_operation, rocblas_int,
                                       rocblas_int, rocblas_int, const double *, const double *, rocblas_int,
                                       const double *, rocblas_int, const double *, double *, rocblas_int);
    create_t create = nullptr;
    stream_t set_stream = nullptr;
    dgemm_t dgemm = nullptr;
    bool ok() const { return create && set_stream && dgemm; }
};

const BlasFns &blas() {
    static const BlasFns fns = [] {
        BlasFns f;
        void *so = nullptr;
        for (const char *name : {"librocblas.so.5", "librocblas.so", "/opt/rocm/lib/librocblas.so.5"})
            if ((so = dlopen(name, RTLD_NOW | RTLD_LOCAL))) break;
        if (so) {
            f.create = reinterpret_cast<BlasFns::create_t>(dlsym(so, "rocblas_create_handle"));
            f.set_stream = reinterpret_cast<BlasFns::stream_t>(dlsym(so, "rocblas_set_stream"));
            f.dgemm = reinterpret_cast<BlasFns::dgemm_t>(dlsym(so, "rocblas_dgemm"));
        }
        return f;
    }();
    return fns;
}

// One handle per host thread and device, kept for the life of the process
// (a rocBLAS handle must not be used by two threads at once; the solver
// sets its stream before each use).
rocblas_handle blas_handle() {
    thread_local std::map<int, rocblas_handle> handles;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    auto it = handles.find(dev);
    if (it != handles.end()) return it->second;
    rocblas_handle h = nullptr;
    if (blas().create(&h) != rocblas_status_success) return nullptr;
    handles[dev] = h;
    return h;
}

// row-major C (m x n, ldc) = A (m x k, lda) B (k x n, ldb): the column-major
// product C^T = B^T A^T on the same storage
bool rm_gemm(rocblas_handle h, int m, int n, int k, const double *A, int lda, const double *B, int ldb, double *C,
             int ldc) {
    const double one = 1.0, zero = 0.0;
    return blas().dgemm(h, rocblas_operation_none, rocblas_operation_none, n, m, k, &one, B, ldb, A, lda, &zero, C,
                        ldc) == rocblas_status_success;
}

int coarse_solve_blas(int nvy, int nvx, const coarse_tables &c, hipStream_t s) {
    rocblas_handle h = blas_handle();
    if (!h || blas().set_stream(h, s) != rocblas_status_success) {
        set_last_hip_error(hipErrorNotInitialized);
        return SIPG_ERR_HIP;
    }
    const int64_t nv = (int64_t)nvy * nvx;
    const int nb = (int)std::min<int64_t>((nv + VT - 1) / VT, 4096);
    hipLaunchKernelGGL(gather_vertex_kernel, dim3(nb), dim3(VT), 0, s, c.E4, nvy, nvx, c.S);
    SIPG_HIP_TRY(hipGetLastError());
    // T1 = S Qx; T2 = (Qy T1) ./ Lambda; T1 = T2 Qx; C = Qy T1 into Cpad
    bool ok = rm_gemm(h, nvy, nvx, nvx, c.S, nvx, c.Qx, nvx, c.T1, nvx) &&
              rm_gemm(h, nvy, nvx, nvy, c.Qy, nvy, c.T1, nvx, c.T2, nvx);
    if (ok) {
        hipLaunchKernelGGL(scale_kernel, dim3(nb), dim3(VT), 0, s, c.T2, c.Linv, nv);
        SIPG_HIP_TRY(hipGetLastError());
        ok = rm_gemm(h, nvy, nvx, nvx, c.T2, nvx, c.Qx, nvx, c.T1, nvx) &&
             rm_gemm(h, nvy, nvx, nvy, c.Qy, nvy, c.T1, nvx, c.Cpad + (nvx + 2) + 1, nvx + 2);
    }
    if (!ok) {
        set_last_hip_error(hipErrorLaunchFailure);
        return SIPG_ERR_HIP;
    }
    hipLaunchKernelGGL(sc_partials_kernel, tile_grid(nvy, nvx), dim3(GT * GT), 0, s, c.S, c.Cpad, nvy, nvx, c.part);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

// Whether the four products of this vertex grid run as rocBLAS calls.
bool coarse_by_blas(int nvy, int nvx) { return (int64_t)nvx * nvy >= kBlasVertices && blas().ok(); }

}  // namespace

int coarse_num_partials(int dimx, int dimy) {
    const int nvx = dimx - 1, nvy = dimy - 1;
    if (nvx < 1 || nvy < 1) return 0;
    const dim3 g = coarse_by_blas(nvy, nvx) ? tile_grid(nvy, nvx) : dim3(dst_tiles(nvx), (nvy + GT - 1) / GT);
    return (int)(g.x * g.y);
}

int launch_coarse_solve(int dtype, int p, const void *r, int dimx, int dimy, const coarse_tables &c, hipStream_t s,
                        bool have_e4, const cg_state *st, int slot) {
    const int nvx = dimx - 1, nvy = dimy - 1;
    const int64_t noe = (int64_t)dimx * dimy;
    if (nvx < 1 || nvy < 1) return SIPG_OK;          // no interior vertex: C = 0, no partials
    coarse_args a{};
    a.r = r;
    a.xi = c.xi;
    a.noe = noe;
    a.E4 = c.E4;
    a.s = s;
    int rc = have_e4 ? SIPG_OK : dispatch_p<1>(p, dtype, 0, a);
    if (rc) return rc;
    if (coarse_by_blas(nvy, nvx)) return coarse_solve_blas(nvy, nvx, c, s);
    // T1 = Qy S (S gathered from E4 on the fly, and stored); T2 = (T1 Qx) ./
    // Lambda; T1 = Qy T2; C = T1 Qx (into Cpad), partials of S.C
    const dim3 gx(dst_tiles(nvx), (nvy + GT - 1) / GT), gy((nvx + GT - 1) / GT, dst_tiles(nvy));
    hipLaunchKernelGGL((dst_gemm_kernel<0, 3>), gy, dim3(64 * dst_waves(3)), 0, s, c.E4, c.Qy, nvy, nvy, nvx, c.S, c.T1,
                       nullptr, st, slot);
    hipLaunchKernelGGL((dst_gemm_kernel<1, 1>), gx, dim3(64 * dst_waves(1)), 0, s, c.T1, c.Qx, nvy, nvx, nvx, c.Linv,
                       c.T2, nullptr, st, slot);
    hipLaunchKernelGGL((dst_gemm_kernel<0, 0>), gy, dim3(64 * dst_waves(0)), 0, s, c.T2, c.Qy, nvy, nvy, nvx, nullptr,
                       c.T1, nullptr, st, slot);
    hipLaunchKernelGGL((dst_gemm_kernel<1, 2>), gx, dim3(64 * dst_waves(2)), 0, s, c.T1, c.Qx, nvy, nvx, nvx, c.S,
                       c.Cpad, c.part, st, slot);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

int launch_coarse_add(int dtype, int p, void *v, int dimx, int64_t n, const coarse_tables &c, int nblk,
                      hipStream_t s) {
    coarse_args a{};
    a.v = v;
    a.Cpad = c.Cpad;
    a.xi = c.xi;
    a.dimx = dimx;
    a.n = n;
    a.nblk = nblk;
    a.s = s;
    return dispatch_p<1>(p, dtype, 1, a);
}

int launch_pcg2_update_p(int dtype, int p, void *x, void *pv, const void *z, int64_t n, const double *part_rr,
                         const double *part_rz, int np, int npc, int dimx, const coarse_tables &c, cg_state *st,
                         int slot, hipStream_t s, void *xlo) {
    coarse_args a{};
    a.x = x;
    a.xlo = xlo;
    a.v = pv;
    a.z = z;
    a.noe = n / ((p + 1) * (p + 1));
    a.prr = part_rr;
    a.prz = part_rz;
    a.np = np;
    a.pc = c.part;
    a.npc = npc;
    a.Cpad = c.Cpad;
    a.xi = c.xi;
    a.dimx = dimx;
    a.st = st;
    a.slot = slot;
    a.s = s;
    return dispatch_p<1>(p, dtype, 2, a);
}

}  // namespace sipg_internal
