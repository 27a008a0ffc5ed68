// kernels_pcg.hip -- block-Jacobi preconditioner and the PCG pieces.
//
// The reference's preconditioned CG (conjugate_gradient_gpu.hpp:116-213)
// applies a block-diagonal preconditioner built from the element Laplacian
// (laplacian_operator.hpp:95-186, mode_matrix.hpp:474-521): a dense block
// per element, with pen truncated to an integer and only the Laplacian-
// pattern entries of the inverse kept.  Here the preconditioner is the
// exact inverse of an interior element's diagonal block of A, applied to
// every element:
//
//   A_ee U = K U W + W U K,   K = K1 + (the element's own face terms in one
//                             direction; the same matrix in x and y for an
//                             interior element),  W = diag(w)
//
// a Kronecker sum, so with K S = W S diag(lambda), S^T W S = I (host side,
// precond.cpp) its inverse is
//
//   U = S [ (S^T R S) ./ (lambda_a + lambda_c) ] S^T
//
// four (p+1)-long contractions per node -- the cost of a volume apply, with
// no neighbour data.  Elements on the mesh boundary get the interior block
// too (still SPD; about 11 % more iterations than their own blocks, in
// exchange for coefficients that are uniform across every wave).
#include "apply_block.hpp"
#include "prec_block.hpp"
#include "partials.hpp"

#include <algorithm>
#include <atomic>

namespace sipg_internal {

namespace {

// Sum over the workgroup, returned to every thread (fixed order).
template <int NT>
__device__ __forceinline__ double group_sum_all(double v, double *red, double *total) {
    const double s = block_sum<NT>(v, red);
    if (threadIdx.x == 0) *total = s;
    __syncthreads();
    const double out = *total;
    __syncthreads();
    return out;
}

// ---- z = M^-1 r -----------------------------------------------------------
// Over every element, with the block sums of r.r and r.z.
//   UPDATE: first r -= alpha Ap with alpha = slot.rz / p.Ap (the p.Ap block
//   sums of this iteration's apply), r written back -- the r half of the
//   reference's alpha step; returns at once when the slot is finished.
//   COPYP:  also p = z (the start of the iteration).
// prec = [S (row-major, S[i][a] = eigenvector a at node i), Linv[a][c] =
// 1 / (lambda_a + lambda_c)], in T.
//   CX: the coefficients are the compile-time tables of the standard penalty
//   pen = 5 (p+1)^2 (prec is then unused); otherwise they are read from prec.
//   RESTR: with E4, also the two-level restriction's corner sums (its own
//   instantiation, so that the plain kernel keeps its registers).
// A wave streams runs of EPW consecutive elements on its own
// (prec_block.hpp): the transposes between the three contraction passes stay
// inside the wave, so the element loop has no workgroup barrier; with the
// standard penalty the contractions take the even-odd form of S
// (cx::PrecEvenOdd), half the multiplies of the plain one.
//
// Bound: memory at p = 8 (four passes: 28 us cached, 36 us inside a solve
// whose vectors do not all stay in the last-level cache); at high degree the
// LDS transposes, whose rows are padded to an odd stride: FP32 p = 15
// (128 x 128) 21.0 -> 17.9 us.  A workgroup-wide split that had the small
// degrees before was up to 15 % faster there than the wave's 8-byte accesses,
// and is slower than these: block-Jacobi PCG at p = 1 (1118 x 1118) 100.7 ->
// 83.5 us an iteration, p = 3 97.2 -> 82.7, FP32 p = 7 (279 x 279) 66 -> 52.
constexpr int kRzWaves = 4, kRzThreads = 64 * kRzWaves;       // per workgroup

template <typename T, int P, bool UPDATE, bool COPYP, bool CX, bool RESTR = false>
__global__ __launch_bounds__(kRzThreads)
void pcg_rz_kernel(T *__restrict__ r, const T *__restrict__ Ap, T *__restrict__ z,
                        T *__restrict__ pcopy, int64_t noe, const T *__restrict__ prec,
                        const double *__restrict__ ppAp, int np, double *__restrict__ prr,
                        double *__restrict__ prz, cg_state *st, int slot, double *__restrict__ E4)
{
    using G = RunGeo<T, P>;
    constexpr int N1 = G::N1, NQ = G::NQ, EPW = G::EPW, NV = G::NV, W = kRzWaves, NT = kRzThreads;
    __shared__ __attribute__((aligned(16))) T lds[W * G::BUF];
    __shared__ T linv[NQ];
    __shared__ double csum[RESTR ? W * 2 * 64 : 1];
    __shared__ double eta[N1];
    __shared__ double red[W];
    __shared__ double total;

    T alpha = T(0);
    if (UPDATE) {
        if (st->s[slot].done | st->err) return;
        const double pAp = group_sum_all<NT>(strided_sum<NT>(ppAp, 0, np), red, &total);
        const double a = st->s[slot].rz / pAp;
        if (!(pAp > 0.0) || !isfinite(a)) {
            if (blockIdx.x == 0 && threadIdx.x == 0) st->err = isfinite(pAp) ? 2 : 3;
            return;
        }
        alpha = (T)a;
        if (blockIdx.x == 0 && threadIdx.x == 0) st->s[slot].alpha = a;    // for the p update
    }
    // 1 / (lambda_a + lambda_c), read per lane (row j) from LDS
    for (int q = threadIdx.x; q < NQ; q += NT) {
        if constexpr (CX) linv[q] = (T)PrecEO<P>::V.Linv[q / N1][q % N1];
        else linv[q] = prec[NQ + q];
    }
    if (RESTR && threadIdx.x < N1) eta[threadIdx.x] = 0.5 * (cx::Basis<P>::T.z[threadIdx.x] + 1.0);
    __syncthreads();

    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t nval = noe * NQ;
    const int64_t nrun = (noe + EPW - 1) / EPW;
    double srr = 0.0, srz = 0.0;
    for (int64_t run = (int64_t)blockIdx.x * W + w; run < nrun; run += (int64_t)gridDim.x * W) {
        const int64_t base = run * NV;
        const int nv = (int)min<int64_t>(NV, nval - base);
        double x0 = 0.0, x1 = 0.0;
        prec_run<T, P, UPDATE, COPYP, CX, RESTR>(r + base, r + base, UPDATE ? Ap + base : nullptr, z + base,
                                                 COPYP ? pcopy + base : nullptr, nv, [&] { return alpha; }, prec,
                                                 linv, lds + w * G::BUF, lane, srr, srz, x0, x1);
        if (RESTR && E4) {
            // E4[c * noe + e]: the lines' x sums, weighted in y, in a fixed
            // order; corner c = 0 bottom-left, 1 bottom-right, 2 top-left, 3
            // top-right (lane q: element q / 2, x half q % 2)
            double *cs = csum + w * 128;
            cs[lane] = x0;
            cs[64 + lane] = x1;
            run_sync();
            if (lane < 2 * EPW) {
                const int el = lane >> 1, h = lane & 1;
                const int64_t e = run * EPW + el;
                double lo = 0.0, hi = 0.0;
#pragma unroll
                for (int jj = 0; jj < N1; ++jj) {
                    const double v = cs[64 * h + el * N1 + jj];
                    lo += (1.0 - eta[jj]) * v;
                    hi += eta[jj] * v;
                }
                if (e < noe) {
                    E4[(int64_t)h * noe + e] = lo;
                    E4[(int64_t)(2 + h) * noe + e] = hi;
                }
            }
            run_sync();
        }
    }
    const double a = block_sum<NT>(srr, red);
    __syncthreads();
    const double b = block_sum<NT>(srz, red);
    if (threadIdx.x == 0) {
        prr[blockIdx.x] = a;
        prz[blockIdx.x] = b;
    }
}

// Workgroups of one pcg_rz kernel that the device holds at once, cached per
// device; the grid is min(groups, that, kMaxPartials).
template <typename T, int P, bool UPDATE, bool COPYP, bool CX>
int pcg_resident() {
    constexpr int kMaxDev = 64;
    static std::atomic<int> cache[kMaxDev];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDev) dev = 0;
    int g = cache[dev].load(std::memory_order_relaxed);
    if (g > 0) return g;
    int cus = 0, per = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 0;
    // the instantiation that also restricts (more registers) where it exists
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &per, reinterpret_cast<const void *>(&pcg_rz_kernel<T, P, UPDATE, COPYP, CX, CX>), kRzThreads, 0);
    if (e != hipSuccess) per = 0;
    g = (cus > 0 ? cus : 1) * (per > 0 ? per : 1);
    cache[dev].store(g, std::memory_order_relaxed);
    return g;
}

// One run of EPW elements per wave and pass, in as many passes as it takes
// for the grid to fit on the device at once (at most kMaxPartials
// workgroups), with the runs spread evenly over the passes.  Fewer
// workgroups also means fewer block sums for the kernels that reduce them
// afterwards (each of their workgroups reads all of them).
template <typename T, int P, bool UPDATE, bool COPYP, bool CX>
int pcg_grid(int64_t noe) {
    const int64_t epw = RunGeo<T, P>::EPW, runs = (noe + epw - 1) / epw;
    const int64_t wgs = std::max<int64_t>(1, (runs + kRzWaves - 1) / kRzWaves);
    const int64_t cap = std::min<int64_t>(pcg_resident<T, P, UPDATE, COPYP, CX>(), kMaxPartials);
    const int64_t rounds = (wgs + cap - 1) / cap;
    return (int)((wgs + rounds - 1) / rounds);
}

// grid: that of the plain kernel (the block-sum count the solver expects);
// with E4, the restricting instantiation
template <typename T, int P, bool UPDATE, bool COPYP, bool CX>
void rz_launch(dim3 grid, void *r, const void *Ap, void *z, void *pcopy, int64_t noe, const void *prec,
               const double *ppAp, int np, double *prr, double *prz, cg_state *st, int slot, double *E4,
               hipStream_t s) {
    if (CX && E4)
        hipLaunchKernelGGL((pcg_rz_kernel<T, P, UPDATE, COPYP, CX, CX>), grid, dim3(kRzThreads), 0, s, (T *)r,
                           (const T *)Ap, (T *)z, (T *)pcopy, noe, (const T *)prec, ppAp, np, prr, prz, st, slot, E4);
    else
        hipLaunchKernelGGL((pcg_rz_kernel<T, P, UPDATE, COPYP, CX>), grid, dim3(kRzThreads), 0, s, (T *)r,
                           (const T *)Ap, (T *)z, (T *)pcopy, noe, (const T *)prec, ppAp, np, prr, prz, st, slot,
                           nullptr);
}

// The standard penalty 5 (p+1)^2 takes the kernel with compile-time
// coefficients; any other the one that reads the op's tables.
inline bool standard_pen(int p, double pen) { return pen == 5.0 * (p + 1) * (p + 1); }

template <typename T, int P>
int launch_rz_one(int mode, bool cx, void *r, const void *Ap, void *z, void *pcopy, int64_t noe,
                  const void *prec, const double *ppAp, int np, double *prr, double *prz, cg_state *st,
                  int slot, double *E4, hipStream_t s)
{
    if (cx) {
        if (mode == 1)
            rz_launch<T, P, true, false, true>(dim3(pcg_grid<T, P, true, false, true>(noe)), r, Ap, z, pcopy,
                                               noe, prec, ppAp, np, prr, prz, st, slot, E4, s);
        else if (mode == 2)
            rz_launch<T, P, false, true, true>(dim3(pcg_grid<T, P, false, true, true>(noe)), r, Ap, z, pcopy,
                                               noe, prec, ppAp, np, prr, prz, st, slot, E4, s);
        else
            rz_launch<T, P, false, false, true>(dim3(pcg_grid<T, P, false, false, true>(noe)), r, Ap, z,
                                                pcopy, noe, prec, ppAp, np, prr, prz, st, slot, E4, s);
    } else {
        if (mode == 1)
            rz_launch<T, P, true, false, false>(dim3(pcg_grid<T, P, true, false, false>(noe)), r, Ap, z,
                                                pcopy, noe, prec, ppAp, np, prr, prz, st, slot, E4, s);
        else if (mode == 2)
            rz_launch<T, P, false, true, false>(dim3(pcg_grid<T, P, false, true, false>(noe)), r, Ap, z,
                                                pcopy, noe, prec, ppAp, np, prr, prz, st, slot, E4, s);
        else
            rz_launch<T, P, false, false, false>(dim3(pcg_grid<T, P, false, false, false>(noe)), r, Ap, z,
                                                 pcopy, noe, prec, ppAp, np, prr, prz, st, slot, E4, s);
    }
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

template <typename T, int P>
int grid_one(int mode, bool cx, int64_t noe) {
    if (cx)
        return mode == 1 ? pcg_grid<T, P, true, false, true>(noe)
                         : mode == 2 ? pcg_grid<T, P, false, true, true>(noe)
                                     : pcg_grid<T, P, false, false, true>(noe);
    return mode == 1 ? pcg_grid<T, P, true, false, false>(noe)
                     : mode == 2 ? pcg_grid<T, P, false, true, false>(noe)
                                 : pcg_grid<T, P, false, false, false>(noe);
}

template <typename T, int... Ps>
struct PcgDispatch;

template <typename T>
struct PcgDispatch<T> {
    static int launch(int, int, bool, void *, const void *, void *, void *, int64_t, const void *,
                      const double *, int, double *, double *, cg_state *, int, double *, hipStream_t) {
        return SIPG_ERR_UNSUPPORTED;
    }
    static int grid(int, int, bool, int64_t) { return -1; }
};

template <typename T, int P0, int... Ps>
struct PcgDispatch<T, P0, Ps...> {
    static int launch(int p, int mode, bool cx, void *r, const void *Ap, void *z, void *pcopy, int64_t noe,
                      const void *prec, const double *ppAp, int np, double *prr, double *prz, cg_state *st,
                      int slot, double *E4, hipStream_t s) {
        if (p == P0)
            return launch_rz_one<T, P0>(mode, cx, r, Ap, z, pcopy, noe, prec, ppAp, np, prr, prz, st, slot, E4, s);
        return PcgDispatch<T, Ps...>::launch(p, mode, cx, r, Ap, z, pcopy, noe, prec, ppAp, np, prr, prz, st,
                                             slot, E4, s);
    }
    static int grid(int p, int mode, bool cx, int64_t noe) {
        if (p == P0) return grid_one<T, P0>(mode, cx, noe);
        return PcgDispatch<T, Ps...>::grid(p, mode, cx, noe);
    }
};

template <typename T>
using PcgDegrees = PcgDispatch<T, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16>;

constexpr int VT = kVecThreads;

__device__ __forceinline__ double vsum_all(double v) {
    __shared__ double red[VT / 64];
    __shared__ double total;
    return group_sum_all<VT>(v, red, &total);
}

__device__ __forceinline__ double vreduce(const double *__restrict__ part, int np) {
    return vsum_all(strided_sum<VT>(part, 0, np));
}

// The step after z = M^-1 r: beta = r.z(new) / r.z(old) and p = z + beta p;
// unless this iteration's r was replaced by the true residual (whose x
// update ran before it), also x += alpha p with the old p.  Block 0 writes
// the next slot: rr = r.r (the stopping test and the host's decisions),
// rz = r.z.  Flag semantics are those of the CG p update.
template <typename T>
__global__ __launch_bounds__(VT) void pcg_update_p_kernel(T *__restrict__ x, T *__restrict__ p,
                                                          const T *__restrict__ z, int64_t n,
                                                          const double *__restrict__ prr,
                                                          const double *__restrict__ prz, int np,
                                                          cg_state *st, int slot, T *__restrict__ xlo) {
    const cg_slot cur = st->s[slot];
    if (cur.done | st->err) {
        if (blockIdx.x == 0 && threadIdx.x == 0) st->s[slot ^ 1] = cur;   // carry forward
        return;
    }
    double sum[2];
    multi_sum<VT, 2>({prr, prz}, {np, np}, sum);
    const double rr_new = sum[0], rz_new = sum[1];
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
    const T alpha = (T)cur.alpha;                        // recorded by the block-Jacobi kernel
    const T beta = (T)beta_d;
    constexpr int VL = 16 / (int)sizeof(T);
    const int64_t nv = n / VL;
    for (int64_t k = (int64_t)blockIdx.x * VT + threadIdx.x; k < nv; k += (int64_t)gridDim.x * VT) {
        const int64_t i = k * VL;
        T pv[VL], zv[VL], xv[VL];
        load_vec<T, VL>(p + i, pv);
        load_vec<T, VL>(z + i, zv);
        if (!replaced) {
            load_vec<T, VL>(x + i, xv);
            if (xlo) {
                T xl[VL];
                load_vec<T, VL>(xlo + i, xl);
#pragma unroll
                for (int q = 0; q < VL; ++q) comp_axpy(xv[q], xl[q], alpha, pv[q]);
                store_vec<T, VL>(xlo + i, xl);
            } else {
#pragma unroll
                for (int q = 0; q < VL; ++q) xv[q] = xv[q] + alpha * pv[q];
            }
            store_vec<T, VL>(x + i, xv);
        }
#pragma unroll
        for (int q = 0; q < VL; ++q) pv[q] = zv[q] + beta * pv[q];
        store_vec<T, VL>(p + i, pv);
    }
    if (blockIdx.x == 0 && threadIdx.x < n - nv * VL) {
        const int64_t i = nv * VL + threadIdx.x;
        const T pi = p[i];
        if (!replaced) {
            if (xlo) comp_axpy(x[i], xlo[i], alpha, pi);
            else x[i] = x[i] + alpha * pi;
        }
        p[i] = z[i] + beta * pi;
    }
}

// x += alpha p (alpha = slot.rz / p.Ap): the x half of the step, run before
// a true residual replaces r in the same iteration.
template <typename T>
__global__ __launch_bounds__(VT) void pcg_x_kernel(T *__restrict__ x, const T *__restrict__ p, int64_t n,
                                                   const double *__restrict__ ppAp, int np,
                                                   const cg_state *st, int slot, T *__restrict__ xlo) {
    if (st->s[slot].done | st->err) return;
    const double pAp = vreduce(ppAp, np);
    const T alpha = (T)(st->s[slot].rz / pAp);
    for (int64_t i = (int64_t)blockIdx.x * VT + threadIdx.x; i < n; i += (int64_t)gridDim.x * VT) {
        if (xlo) {
            T xh = x[i], xl = xlo[i];
            comp_axpy(xh, xl, alpha, p[i]);
            x[i] = xh;
            xlo[i] = xl;
        } else {
            x[i] = x[i] + alpha * p[i];
        }
    }
}

// Initial state: r.r and r.z from the preconditioner's block sums, b.b
// from the true residual's.
__global__ __launch_bounds__(VT) void pcg_init_finalize_kernel(const double *__restrict__ prr,
                                                               const double *__restrict__ prz, int np,
                                                               const double *__restrict__ pbb, int npb,
                                                               cg_state *st, double tol, int tol_mode,
                                                               int maxit, int true_stop,
                                                               const double *__restrict__ pc, int npc) {
    const double rr = vreduce(prr, np);
    const double rz = vreduce(prz, np) + vreduce(pc, npc);     // + S.C of a coarse level
    const double bb = vreduce(pbb, npb);
    if (threadIdx.x == 0) {
        const double stop = tol_mode == SIPG_TOL_REL ? tol * sqrt(bb) : tol;
        cg_slot s0;
        s0.rr = rr;
        s0.alpha = s0.beta = s0.pAp = 0.0;
        s0.rz = rz;
        s0.it = 0;
        s0.done = (sqrt(rr) > stop && maxit > 0) ? 0 : 1;
        s0.checked = 1;
        s0.flags = 0;
        st->s[0] = s0;
        st->s[1] = s0;
        st->rr0 = rr;
        st->stop_true = stop;
        st->rr_ref = rr;
        st->bb = bb;
        st->stop = stop;
        st->maxit = maxit;
        st->nrep = 0;
        st->err = (!isfinite(rr) || !isfinite(bb) || !isfinite(rz)) ? 3 : 0;
        st->true_stop = true_stop;
    }
}

}  // namespace

int pcg_num_blocks(int dtype, int p, double pen, int mode, int64_t noe) {
    const bool cx = standard_pen(p, pen);
    return dtype == SIPG_F64 ? PcgDegrees<double>::grid(p, mode, cx, noe)
                             : PcgDegrees<float>::grid(p, mode, cx, noe);
}

bool pcg_rz_fuses_restrict(int dtype, int p, double pen) {
    (void)dtype;
    return p >= 1 && p <= kMaxDegree && standard_pen(p, pen);
}

int launch_pcg_rz(int dtype, int p, double pen, int mode, void *r, const void *Ap, void *z, void *pcopy,
                  int64_t noe, const void *prec, const double *part_pAp, int np_pAp, double *part_rr,
                  double *part_rz, cg_state *st, int slot, hipStream_t s, double *E4) {
    const bool cx = standard_pen(p, pen);
    if (dtype == SIPG_F64)
        return PcgDegrees<double>::launch(p, mode, cx, r, Ap, z, pcopy, noe, prec, part_pAp, np_pAp, part_rr,
                                          part_rz, st, slot, E4, s);
    return PcgDegrees<float>::launch(p, mode, cx, r, Ap, z, pcopy, noe, prec, part_pAp, np_pAp, part_rr,
                                     part_rz, st, slot, E4, s);
}

int launch_pcg_update_p(int dtype, void *x, void *p, const void *z, int64_t n, const double *part_rr,
                        const double *part_rz, int np, int nblk, cg_state *st, int slot, hipStream_t s, void *xlo) {
    if (dtype == SIPG_F64)
        hipLaunchKernelGGL(pcg_update_p_kernel<double>, dim3(nblk), dim3(VT), 0, s, (double *)x, (double *)p,
                           (const double *)z, n, part_rr, part_rz, np, st, slot, (double *)xlo);
    else
        hipLaunchKernelGGL(pcg_update_p_kernel<float>, dim3(nblk), dim3(VT), 0, s, (float *)x, (float *)p,
                           (const float *)z, n, part_rr, part_rz, np, st, slot, (float *)xlo);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

int launch_pcg_x(int dtype, void *x, const void *p, int64_t n, const double *part_pAp, int np_pAp, int nblk,
                 const cg_state *st, int slot, hipStream_t s, void *xlo) {
    if (dtype == SIPG_F64)
        hipLaunchKernelGGL(pcg_x_kernel<double>, dim3(nblk), dim3(VT), 0, s, (double *)x, (const double *)p, n,
                           part_pAp, np_pAp, st, slot, (double *)xlo);
    else
        hipLaunchKernelGGL(pcg_x_kernel<float>, dim3(nblk), dim3(VT), 0, s, (float *)x, (const float *)p, n,
                           part_pAp, np_pAp, st, slot, (float *)xlo);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

int launch_pcg_init_finalize(const double *part_rr, const double *part_rz, int np, const double *part_bb,
                             int npb, cg_state *st, double tol, int tol_mode, int maxit, int true_stop,
                             hipStream_t s, const double *part_c, int npc) {
    hipLaunchKernelGGL(pcg_init_finalize_kernel, dim3(1), dim3(VT), 0, s, part_rr, part_rz, np, part_bb, npb,
                       st, tol, tol_mode, maxit, true_stop, part_c, npc);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

}  // namespace sipg_internal
