// kernels_small.hip -- CG iterations of a small problem inside one workgroup.
//
// A problem of a few thousand unknowns is a few KB: an iteration of the
// three-launch CG (fused apply + p.Ap, x/r update + r.r, p update) then
// costs its launches and reductions (12 us traced, 15 us with the gaps, at
// 8 x 8 elements of degree 3) and no data motion to speak of.  Here one
// workgroup runs a whole chunk of iterations: p and the two directions'
// line results live in LDS, x, r and p in registers, the two sums of an
// iteration cross eight waves through LDS, and nothing leaves the CU until
// the chunk ends.  The iteration is the one of conjugate_gradient
// (conjugate_gradient_gpu.hpp:69-100) with the slot rules of
// cg_update_xr_kernel / cg_update_p_kernel, so the host's chunk loop, its
// replacements and its stopping decisions are unchanged.  A chunk is long: it
// stops where the recursion first wants its final check (hold), where
// iterations past that could use up the iteration cap, or run a few unknowns
// until p.Ap is zero.  Where the host lets it go on all the same, a zero p.Ap
// is an exact solution that waits for its check, not a breakdown.
//
// Bound: latency of four barriers and the dependent LDS reads between them.
// Measured 8 x 8, p = 3 (1,024 unknowns): 15 -> 3.1 us per iteration, a solve
// to 1e-10 2.8 -> 0.56 ms.  kSmallMax: three arrays of 4,096 padded values fill the
// LDS; there (16 x 16, p = 3 and 4 x 4, p = 15) the
// workgroup takes 4.9 and 4.1 us per iteration against 14.0 and 19.5 for the launches.
#include "line_math.hpp"
#include "partials.hpp"

namespace sipg_internal {

namespace {

constexpr int kSmallMax = 4096;      // unknowns
constexpr int NT = 512;              // threads: eight waves
constexpr int KR = kSmallMax / NT;   // values per thread

// One barrier: the waves' sums cross through red, which alternates between
// two buffers, and every thread adds them in the same order.
__device__ __forceinline__ double group_total(double v, double *red) {
    v = wave_total(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    static_assert(NT == 512, "a tree over eight waves: three dependent adds");
    return ((red[0] + red[1]) + (red[2] + red[3])) + ((red[4] + red[5]) + (red[6] + red[7]));
}

template <typename T, int P>
__global__ __launch_bounds__(NT) void cg_small_kernel(T *__restrict__ x, T *__restrict__ r, T *__restrict__ p, int dimx,
                                                      int dimy, T pen, int n_it, int hold, cg_state *st,
                                                      int slot)
{
    constexpr int N1 = P + 1, NQ = N1 * N1;
    constexpr int RS = N1 % 2 ? N1 : N1 + 1, TS = N1 * RS;       // odd row stride: rows hit distinct banks
    constexpr int NP = (kSmallMax / NQ + 1) * TS;
    constexpr int MT = (2 * kSmallMax / N1 + NT - 1) / NT;       // line tasks per thread
    __shared__ T sp[NP], sx[NP], sy[NP];
    __shared__ double red[2][NT / 64];
    cg_slot cur = st->s[slot];
    const int last = (slot + n_it) & 1;
    if (cur.done | st->err) {
        if (threadIdx.x == 0) st->s[last] = cur;                  // carry forward
        return;
    }
    const double stop = st->stop;
    const int maxit = st->maxit, true_stop = st->true_stop;
    const CxCoef<T, P> c{};
    const int tid = threadIdx.x, noe = dimx * dimy, n = noe * NQ, nl = noe * N1;
    auto pos = [](int idx) { return RS == N1 ? idx : idx + idx / N1; };

    // this thread's lines: where they start, their stride, and their
    // neighbours (negative: the mesh ends there)
    int base[MT], low[MT], high[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int task = tid + t * NT;
        const bool dirx = task < nl;
        const int q = dirx ? task : task - nl, e = q / N1, j = q - e * N1;
        const int gy = e / dimx, gx = e - gy * dimx;
        const int o = dirx ? j : j * RS;
        base[t] = e * TS + o;
        if (dirx) {
            low[t] = gx > 0 ? (e - 1) * TS + o : -1;
            high[t] = gx < dimx - 1 ? (e + 1) * TS + o : -1;
        } else {                                                  // y grows downwards
            low[t] = gy < dimy - 1 ? (e + dimx) * TS + o : -1;
            high[t] = gy > 0 ? (e - dimx) * TS + o : -1;
        }
    }
    T xv[KR], rv[KR], pv[KR];
#pragma unroll
    for (int k = 0; k < KR; ++k) {
        const int i = tid + k * NT;
        xv[k] = rv[k] = pv[k] = T(0);
        if (i < n) {
            xv[k] = x[i];
            rv[k] = r[i];
            pv[k] = p[i];
            sp[pos(i)] = pv[k];
        }
    }
    __syncthreads();
    int err = 0;
    for (int it = 0; it < n_it && !cur.done && !(hold && (cur.flags & kSlotWantCheck)); ++it) {
        // both directions' lines
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const int task = tid + t * NT;
            if (task < 2 * nl) {
                const bool dirx = task < nl;
                const int sd = dirx ? RS : 1;
                T u[N1], o[N1];
                Line<T, P> L, Q;
#pragma unroll
                for (int i = 0; i < N1; ++i) u[i] = sp[base[t] + i * sd];
                L.from(u, c);
                T tl = -L.t0, dl = L.d0, tr = -L.tP, dr = L.dP, pl = T(0.5) * pen, pr = pl;
                if (low[t] >= 0) {
#pragma unroll
                    for (int i = 0; i < N1; ++i) u[i] = sp[low[t] + i * sd];
                    Q.from(u, c);
                    tl = Q.tP;
                    dl = Q.dP;
                    pl = pen;
                }
                if (high[t] >= 0) {
#pragma unroll
                    for (int i = 0; i < N1; ++i) u[i] = sp[high[t] + i * sd];
                    Q.from(u, c);
                    tr = Q.t0;
                    dr = Q.d0;
                    pr = pen;
                }
                line_apply<T, P>(L, tl, dl, tr, dr, pl, pr, o, c);
                const T wj = c.w((dirx ? task : task - nl) % N1);
                T *out = dirx ? sx : sy;
#pragma unroll
                for (int i = 0; i < N1; ++i) out[base[t] + i * sd] = wj * o[i];
            }
        }
        __syncthreads();
        T av[KR];
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < KR; ++k) {
            const int i = tid + k * NT;
            av[k] = T(0);
            if (k * NT < n && i < n) {
                av[k] = sx[pos(i)] + sy[pos(i)];
                s += (double)pv[k] * (double)av[k];
            }
        }
        const double pAp = group_total(s, red[0]);
        if (pAp == 0.0 && (cur.flags & kSlotWantCheck)) break;    // solved exactly: only the final check is left
        const double alpha_d = cur.rr / pAp;
        if (!(pAp > 0.0) || !isfinite(alpha_d)) {                 // the same in every thread
            err = isfinite(pAp) ? 2 : 3;
            break;
        }
        const T alpha = (T)alpha_d;
        s = 0.0;
#pragma unroll
        for (int k = 0; k < KR; ++k) {
            if (k * NT >= n) break;
            xv[k] = xv[k] + alpha * pv[k];
            rv[k] = rv[k] - alpha * av[k];
            s += (double)rv[k] * (double)rv[k];
        }
        const double rr_new = group_total(s, red[1]);
        const double beta_d = rr_new / cur.rr;
        const bool met = !(sqrt(rr_new) > stop);
        cur.rr = cur.rz = rr_new;
        cur.alpha = 0.0;
        cur.beta = beta_d;
        cur.pAp = 0.0;
        cur.it += 1;
        cur.done = ((met && !true_stop) || cur.it >= maxit) ? 1 : 0;
        cur.checked = 0;
        cur.flags = (met && true_stop) ? kSlotWantCheck : 0;
        const T beta = (T)beta_d;
#pragma unroll
        for (int k = 0; k < KR; ++k) {
            const int i = tid + k * NT;
            if (k * NT < n && i < n) {
                pv[k] = rv[k] + beta * pv[k];
                sp[pos(i)] = pv[k];
            }
        }
        if (!isfinite(rr_new)) {
            err = 3;
            break;
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < KR; ++k) {
        const int i = tid + k * NT;
        if (i < n) {
            x[i] = xv[k];
            r[i] = rv[k];
            p[i] = pv[k];
        }
    }
    if (tid == 0) {
        st->s[last] = cur;
        if (err) st->err = err;
    }
}

template <typename T, int P>
void launch_one(void *x, void *r, void *p, int dimx, int dimy, double pen, int n_it, bool hold, cg_state *st,
                int slot, hipStream_t s) {
    hipLaunchKernelGGL((cg_small_kernel<T, P>), dim3(1), dim3(NT), 0, s, (T *)x, (T *)r, (T *)p, dimx, dimy, (T)pen,
                       n_it, hold ? 1 : 0, st, slot);
}

template <typename T, int P = 1>
int dispatch(int deg, void *x, void *r, void *p, int dimx, int dimy, double pen, int n_it, bool hold, cg_state *st,
             int slot, hipStream_t s) {
    if constexpr (P <= kMaxDegree) {
        if (deg != P) return dispatch<T, P + 1>(deg, x, r, p, dimx, dimy, pen, n_it, hold, st, slot, s);
        launch_one<T, P>(x, r, p, dimx, dimy, pen, n_it, hold, st, slot, s);
        SIPG_HIP_TRY(hipGetLastError());
        return SIPG_OK;
    }
    return SIPG_ERR_UNSUPPORTED;
}

}  // namespace

bool cg_small_fits(int p, int dimx, int dimy) {
    return p >= 1 && p <= kMaxDegree && (int64_t)dimx * dimy * (p + 1) * (p + 1) <= kSmallMax;
}

int launch_cg_small(int dtype, int deg, void *x, void *r, void *p, int dimx, int dimy, double pen, int n_it,
                    bool hold, cg_state *st, int slot, hipStream_t s) {
    if (!cg_small_fits(deg, dimx, dimy) || n_it < 1) return SIPG_ERR_INVALID;
    return dtype == SIPG_F64 ? dispatch<double>(deg, x, r, p, dimx, dimy, pen, n_it, hold, st, slot, s)
                             : dispatch<float>(deg, x, r, p, dimx, dimy, pen, n_it, hold, st, slot, s);
}

}  // namespace sipg_internal
