// strip_apply.hpp -- the fused SIPG operator on a strip of elements, marched
// row by row: the core of the vector-ALU apply of one mesh
// (kernels_apply.hip) and of a batch (kernels_batch.hip).
//
// A wave holds EPW = 64 / (p+1) whole elements of one mesh row (7 at p = 8),
// lane s (p+1) + j on line j of element s, and walks its strip in y.  Each
// row is loaded once, column by column into registers (a lane's column is
// the x line of its node row), while the row before it is computed; one LDS
// transpose gives the y lines.  The neighbours in y are the same lanes'
// previous and next rows, those in x the lanes p+1 away, so only the end
// values and derivatives of lines are exchanged (line_math.hpp) and the
// operator has no workgroup barrier in its loop.
//
// A workgroup of four waves takes a band of rows.  Waves 0 and 1 start at
// the rows where they meet and walk apart, so do 2 and 3, and 1 and 2 end
// where they meet: the faces inside a band are exchanged through LDS, once
// at the start and once at the end, and only the band's two outer rows are
// loaded twice.  The next row's loads are in flight while a row is
// computed.
//
// Bound: on meshes past the caches the stores, columns of p+1 values as they
// sit in the lanes, sizeof(T) (p+1) bytes to a segment: 322 us at 1024 x 1024,
// p = 8 FP64, 151 with the stores left out, where a copy takes 258.  On cached
// ones the issue of vector-memory instructions (3 (p+1) a row) and the FP64
// arithmetic, 218 instructions a row at p = 8: 18.8 us at 256 x 256, 12.8
// without the stores.  Storing through LDS as whole rows instead cost more LDS
// time than it saved.
#pragma once
#include "line_math.hpp"

#include <type_traits>

namespace sipg_internal {

template <typename T, int P>
struct StripGeo {
    static constexpr int N1 = P + 1, NQ = N1 * N1;
    static constexpr int EPW = 64 / N1;                           // elements of a strip
    static constexpr int RS = N1 % 2 ? N1 : N1 + 1;               // odd row stride: lines hit distinct banks
    static constexpr int TS = N1 * RS;
    static constexpr int W = 4;                                   // waves
    static constexpr int BUF = (EPW + (64 % N1 ? 1 : 0)) * TS;    // one row, with a slot for the spare lanes
    static constexpr int LDS = W * 2 * BUF;
    static constexpr int EXCH = 2 * W * 2 * 64;
};

// LDS writes of the wave become visible to all of its lanes
__device__ __forceinline__ void strip_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// y = A x on the elements [x0, x0 + ncol) x [yA, yB) of a dimx x dimy mesh,
// by the whole workgroup of 256 threads (two barriers), tid = threadIdx.x;
// returns this thread's share of x.y over them when DOT.
template <typename T, int P, bool DOT, class C = CxCoef<T, P>>
__device__ __forceinline__ double strip_apply(const T *__restrict__ x, T *__restrict__ y, int dimx, int dimy, T pen,
                                              int x0, int ncol, int yA, int yB, T *lds, T *exch,
                                              int tid)
{
    using G = StripGeo<T, P>;
    constexpr int N1 = G::N1, NQ = G::NQ, EPW = G::EPW, RS = G::RS, TS = G::TS;
    const C c{};
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the band's rows, split over the waves that get one
    const int nb = yB - yA, na = min(nb, G::W);
    const bool active = w < na;
    const int ya = yA + (active ? nb * w / na : 0), yb = yA + (active ? nb * (w + 1) / na : 0);
    const int nrow = yb - ya;
    const int s = lane / N1, j = lane - s * N1;                   // s >= ncol: spare lanes
    const T wj = c.w(j);
    T *tile = lds + w * 2 * G::BUF + s * TS;
    const int off = min(s, ncol - 1) * NQ + j;
    // the side tiles: lanes from the last group on (or the first spare one)
    // take the right tile, the others the left one.  At a mesh edge it is
    // the lane's own element, whose mirror image is the ghost.
    const bool isR = s >= min(ncol, EPW - 1);
    const bool edge = isR ? x0 + ncol == dimx : x0 == 0;
    const int hoff = (isR ? (edge ? (ncol - 1) * NQ : ncol * NQ) : (edge ? 0 : -NQ)) + j;
    const bool hP = isR == edge;                                  // its right end counts (else its left one)
    const T hsgn = edge ? T(-1) : T(1);
    const T pL = (x0 == 0 && s == 0) ? T(0.5) * pen : pen;
    const T pR = (x0 + ncol == dimx && s == ncol - 1) ? T(0.5) * pen : pen;
    double dot[2] = {0.0, 0.0};                                   // two chains of sums

    T ua[N1], ha[N1];                                             // the next row's column; the side tile's
    auto row = [&](int gy) { return x + ((size_t)gy * dimx + x0) * NQ; };
    auto load = [&](int gy) {
        const T *r = row(gy);
#pragma unroll
        for (int i = 0; i < N1; ++i) ua[i] = r[off + i * N1];
    };
    auto load_side = [&](int gy) {
        const T *r = row(gy);
#pragma unroll
        for (int i = 0; i < N1; ++i) ha[i] = r[hoff + i * N1];
    };
    auto put = [&](T *t) {
#pragma unroll
        for (int i = 0; i < N1; ++i) t[i * RS + j] = ua[i];
        strip_sync();
    };
    auto lines = [&](const T *t, Line<T, P> &V) {
        T v[N1];
#pragma unroll
        for (int i = 0; i < N1; ++i) v[i] = t[j * RS + i];
        V.from(v, c);
    };
    // Finishes row gy, held in tile t with its y lines V; (tB, nB) the
    // neighbour below, (tA, nA) above.  Then loads row gnext's side tile.
    auto finish = [&](int gy, int gnext, T *t, const Line<T, P> &V, T tB, T nB, T tA, T nA) {
        T ht, hn;
        {
            Line<T, P> Q;
            Q.from(ha, c);
            ht = hsgn * (hP ? Q.tP : Q.t0);
            hn = hP ? Q.dP : Q.d0;
        }
        if (gnext >= 0) load_side(gnext);
        Line<T, P> U;
        T u[N1];
#pragma unroll
        for (int i = 0; i < N1; ++i) u[i] = t[i * RS + j];
        U.from(u, c);
        T tL = __shfl(U.tP, lane - N1, 64), nL = __shfl(U.dP, lane - N1, 64);
        T p0 = U.t0, p1 = U.d0;
        if (ncol < EPW && s >= ncol) {                            // the first spare group speaks for the right tile
            p0 = ht;
            p1 = hn;
        }
        T tR = __shfl(p0, lane + N1, 64), nR = __shfl(p1, lane + N1, 64);
        if (s == 0) {
            tL = ht;
            nL = hn;
        }
        if (s == EPW - 1) {
            tR = ht;
            nR = hn;
        }
        T o[N1];
        line_apply<T, P>(V, tB, nB, tA, nA, gy == dimy - 1 ? T(0.5) * pen : pen, gy == 0 ? T(0.5) * pen : pen, o, c);
        strip_sync();
#pragma unroll
        for (int a = 0; a < N1; ++a) t[j * RS + a] = wj * o[a];
        strip_sync();
        line_apply<T, P>(U, tL, nL, tR, nR, pL, pR, o, c);
#pragma unroll
        for (int a = 0; a < N1; ++a) o[a] = line_fma(wj, o[a], t[a * RS + j]);
        strip_sync();
        if (s < ncol) {
            T *dst = y + ((size_t)gy * dimx + x0) * NQ + off;
#pragma unroll
            for (int a = 0; a < N1; ++a) {
                dst[a * N1] = o[a];
                if (DOT) dot[a & 1] += (double)u[a] * (double)o[a];
            }
        }
    };

    auto walk = [&](auto dn) {
        constexpr bool down = decltype(dn)::value;
        constexpr int d = down ? 1 : -1;
        auto near_t = [](const Line<T, P> &L) { return down ? L.tP : L.t0; };   // the face towards the row before
        auto near_n = [](const Line<T, P> &L) { return down ? L.dP : L.d0; };
        auto far_t = [](const Line<T, P> &L) { return down ? L.t0 : L.tP; };    // ... towards the row after
        auto far_n = [](const Line<T, P> &L) { return down ? L.d0 : L.dP; };
        const int first = down ? ya : yb - 1, last = down ? yb - 1 : ya;
        auto inside = [&](int gy) { return gy >= 0 && gy < dimy; };
        const bool meets0 = (w ^ 1) < na, meets1 = (w == 1 || w == 2) && 3 - w < na;
        const int nload = nrow + (!meets1 && inside(last + d) ? 1 : 0);
        T *t0 = tile, *t1 = tile + G::BUF;
        Line<T, P> V, Vn;
        T pt = 0, pn = 0;                                         // the row before's face
        auto done = [&](int gy, int gnext, T *t, const Line<T, P> &L, T qt, T qn) {
            finish(gy, gnext, t, L, down ? qt : pt, down ? qn : pn, down ? pt : qt, down ? pn : qn);
        };
        if (active) {
            const bool before = !meets0 && inside(first - d);     // a row of another workgroup's
            if (before) {
                load(first - d);
                put(t1);
                lines(t1, Vn);
                pt = far_t(Vn);
                pn = far_n(Vn);
            }
            load(first);
            load_side(first);
            put(t0);
            if (nload > 1) load(first + d);
            lines(t0, V);
            if (!before) {
                pt = -near_t(V);                                  // the ghost, unless a wave is met
                pn = near_n(V);
            }
            if (meets0) {
                exch[(2 * w) * 64 + lane] = near_t(V);
                exch[(2 * w + 1) * 64 + lane] = near_n(V);
            }
        }
        __syncthreads();
        if (active) {
            if (meets0) {
                pt = exch[(2 * (w ^ 1)) * 64 + lane];
                pn = exch[(2 * (w ^ 1) + 1) * 64 + lane];
            }
            for (int k = 1; k < nrow; ++k) {
                put(t1);
                if (k + 1 < nload) load(first + d * (k + 1));
                lines(t1, Vn);
                done(first + d * (k - 1), first + d * k, t0, V, near_t(Vn), near_n(Vn));
                pt = far_t(V);
                pn = far_n(V);
                V = Vn;
                T *tt = t0;
                t0 = t1;
                t1 = tt;
            }
            if (meets1) {
                exch[G::EXCH / 2 + (2 * w) * 64 + lane] = far_t(V);
                exch[G::EXCH / 2 + (2 * w + 1) * 64 + lane] = far_n(V);
            }
        }
        __syncthreads();
        if (active) {
            T qt = -far_t(V), qn = far_n(V);                      // the ghost
            if (meets1) {
                qt = exch[G::EXCH / 2 + (2 * (3 - w)) * 64 + lane];
                qn = exch[G::EXCH / 2 + (2 * (3 - w) + 1) * 64 + lane];
            } else if (nload > nrow) {
                put(t1);
                lines(t1, Vn);
                qt = near_t(Vn);
                qn = near_n(Vn);
            }
            done(last, -1, t0, V, qt, qn);
        }
    };
    // waves 1 and 3 walk down, 0 and 2 up (every wave reaches both barriers)
    if (w & 1) walk(std::true_type{});
    else walk(std::false_type{});
    return dot[0] + dot[1];
}

}  // namespace sipg_internal
