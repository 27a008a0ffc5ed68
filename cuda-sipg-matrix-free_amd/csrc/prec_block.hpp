// prec_block.hpp -- the contractions of the block-Jacobi preconditioner
// z = M^-1 r on one element line, shared by the single-mesh kernels
// (kernels_pcg.hip) and the batched ones (kernels_batch_pcg.hip).
//
// M^-1 R = S [ (S^T R S) ./ (lambda_a + lambda_c) ] S^T per element, S the
// W-orthonormal eigenvectors of the interior element block (precond.cpp,
// cx::make_prec): each pass contracts one line of the element's tile with
// S or S^T.
#pragma once
#include "basis_constexpr.hpp"
#include "partials.hpp"

namespace sipg_internal {

// The standard penalty's tables as device constants, in even-odd form where
// the eigenvectors have parities (every degree but p = 1).
template <int P>
struct PrecEO {
    static constexpr cx::PrecEvenOdd<P> V = cx::make_prec_even_odd<P>();
    static constexpr bool EO = V.ok();
    static_assert(EO || P == 1, "block-Jacobi eigenvectors without a parity");
};

// out[a] = sum_i S[i][a] in[i] (S^T in) and out[d] = sum_c S[d][c] in[c]
// (S in).  The standard penalty's table in even-odd form works on the pair
// sums e[i] = in[i] + in[p-i] and differences o[i] = in[i] - in[p-i];
// otherwise the plain sums run over the compile-time Jacobi table (CX, a
// degree without parities) or a row-major table in memory.
template <typename T, int P, bool CX>
__device__ __forceinline__ T s_coef(const T *__restrict__ S, int i, int a) {
    if constexpr (CX) return (T)PrecEO<P>::V.S0[i][a];
    else return S[i * (P + 1) + a];
}

template <typename T, int P, bool CX>
__device__ __forceinline__ void contract_st(const T *__restrict__ S, const T (&in)[P + 1], T (&out)[P + 1]) {
    constexpr int N1 = P + 1, H = N1 / 2;
    if constexpr (CX && PrecEO<P>::EO) {
        using E = PrecEO<P>;
        T e[H], o[H];
#pragma unroll
        for (int i = 0; i < H; ++i) {
            e[i] = in[i] + in[P - i];
            o[i] = in[i] - in[P - i];
        }
#pragma unroll
        for (int a = 0; a < N1; ++a) {
            T acc = T(0);
            if (E::V.sig[a] > 0) {
#pragma unroll
                for (int i = 0; i < H; ++i) acc += (T)E::V.S[i][a] * e[i];
                if (P % 2 == 0) acc += (T)E::V.S[H][a] * in[H];
            } else {
#pragma unroll
                for (int i = 0; i < H; ++i) acc += (T)E::V.S[i][a] * o[i];
            }
            out[a] = acc;
        }
    } else {
#pragma unroll
        for (int a = 0; a < N1; ++a) {
            T acc = T(0);
#pragma unroll
            for (int i = 0; i < N1; ++i) acc += s_coef<T, P, CX>(S, i, a) * in[i];
            out[a] = acc;
        }
    }
}

template <typename T, int P, bool CX>
__device__ __forceinline__ void contract_s(const T *__restrict__ S, const T (&in)[P + 1], T (&out)[P + 1]) {
    constexpr int N1 = P + 1, H = N1 / 2;
    if constexpr (CX && PrecEO<P>::EO) {
        using E = PrecEO<P>;
#pragma unroll
        for (int d = 0; d < H; ++d) {
            T ev = T(0), od = T(0);
#pragma unroll
            for (int c = 0; c < N1; ++c) {
                if (E::V.sig[c] > 0) ev += (T)E::V.S[d][c] * in[c];
                else od += (T)E::V.S[d][c] * in[c];
            }
            out[d] = ev + od;
            out[P - d] = ev - od;
        }
        if (P % 2 == 0) {
            T ev = T(0);
#pragma unroll
            for (int c = 0; c < N1; ++c)
                if (E::V.sig[c] > 0) ev += (T)E::V.S[H][c] * in[c];
            out[H] = ev;
        }
    } else {
#pragma unroll
        for (int d = 0; d < N1; ++d) {
            T acc = T(0);
#pragma unroll
            for (int c = 0; c < N1; ++c) acc += s_coef<T, P, CX>(S, d, c) * in[c];
            out[d] = acc;
        }
    }
}

// ---- a run of whole elements in one wave -----------------------------------
// EPW = 64 / (p+1) elements (7 at p = 8), lane (s, j) = s (p+1) + j on line j
// of element s; the tiles sit in the wave's LDS with an odd row stride, so
// that lanes on consecutive rows hit distinct banks.
template <typename T, int P>
struct RunGeo {
    static constexpr int N1 = P + 1, NQ = N1 * N1;
    static constexpr int EPW = 64 / N1;
    static constexpr int RS = N1 % 2 ? N1 : N1 + 1, TS = N1 * RS;
    static constexpr int NV = EPW * NQ;                 // values of a full run
    // values per lane and access: 16 bytes, inside one row where rows are padded
    static constexpr int VL = sizeof(T) == 8 ? 2 : (N1 % 2 == 1 || N1 % 4 == 0) ? 4 : 2;
    static constexpr int KR = (NV + 64 * VL - 1) / (64 * VL);
    static constexpr int BUF = (EPW + (64 % N1 ? 1 : 0)) * TS;   // with a slot for the spare lanes
    static __device__ __forceinline__ int pos(int idx) { return RS == N1 ? idx : idx + idx / N1; }
};

__device__ __forceinline__ void run_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// z = M^-1 r on the nv values (whole elements) at rs, by one wave; UPDATE:
// first r -= alpha() Ap, written to r (alpha() is called once the loads are
// under way); COPYP: also pc = z.  linv: 1 / (lambda_a
// + lambda_c) in LDS.  Adds this lane's shares of r.r and r.z; RESTR: x0,
// x1 = the lane's column sums of r weighted 1 - xi and xi (xi the node's
// position in the element), the x half of the coarse restriction.
//
// The values move in vectors of VL, lane l of chunk k on values o = VL (l +
// 64 k) and up; a vector past the end moves back to the last VL values (the
// same values written twice, counted once).  All loads are issued before
// the first is used.
template <typename T, int P, bool UPDATE, bool COPYP, bool CX, bool RESTR, class A>
__device__ __forceinline__ void prec_run(const T *rs, T *r, const T *__restrict__ Ap, T *__restrict__ z,
                                         T *__restrict__ pc, int nv, A alpha, const T *__restrict__ prec,
                                         const T *linv, T *wl, int lane, double &srr, double &srz, double &x0,
                                         double &x1)
{
    using G = RunGeo<T, P>;
    constexpr int N1 = G::N1, RS = G::RS, VL = G::VL, KR = G::KR;
    const int s = lane / N1, j = lane - s * N1;         // lanes past the last element: the spare slot
    T *tile = wl + s * G::TS;
    T rv[KR][VL], av[KR][VL];
#pragma unroll
    for (int k = 0; k < KR; ++k) {
        const int idx = min(VL * (lane + 64 * k), nv - VL);
        load_vec<T, VL>(rs + idx, rv[k]);
        if (UPDATE) load_vec<T, VL>(Ap + idx, av[k]);
    }
    const T al = UPDATE ? alpha() : T(0);
#pragma unroll
    for (int k = 0; k < KR; ++k) {
        const int o = VL * (lane + 64 * k), idx = min(o, nv - VL);
#pragma unroll
        for (int q = 0; q < VL; ++q) {
            if (UPDATE) rv[k][q] = rv[k][q] - al * av[k][q];
            srr += idx + q >= o ? (double)rv[k][q] * (double)rv[k][q] : 0.0;
        }
        if (UPDATE) store_vec<T, VL>(r + idx, rv[k]);
        store_vec<T, VL>(wl + G::pos(idx), rv[k]);
    }
    run_sync();
    {   // 1: column j of S^T R
        T c[N1], t[N1];
#pragma unroll
        for (int i = 0; i < N1; ++i) c[i] = tile[i * RS + j];
        if (RESTR) {
            double a = 0.0, b = 0.0;
#pragma unroll
            for (int i = 0; i < N1; ++i) {
                const double xi = 0.5 * (cx::Basis<P>::T.z[i] + 1.0);
                a += (1.0 - xi) * (double)c[i];
                b += xi * (double)c[i];
            }
            x0 = a;
            x1 = b;
        }
        contract_st<T, P, CX>(prec, c, t);
#pragma unroll
        for (int a = 0; a < N1; ++a) tile[a * RS + j] = t[a];
    }
    run_sync();
    {   // 2: row j of ((S^T R S) ./ L) S^T
        T w[N1], v[N1];
#pragma unroll
        for (int b = 0; b < N1; ++b) w[b] = tile[j * RS + b];
        contract_st<T, P, CX>(prec, w, v);
#pragma unroll
        for (int c = 0; c < N1; ++c) v[c] *= linv[j * N1 + c];
        contract_s<T, P, CX>(prec, v, w);
#pragma unroll
        for (int d = 0; d < N1; ++d) tile[j * RS + d] = w[d];
    }
    run_sync();
    {   // 3: column j of S (...)
        T c[N1], t[N1];
#pragma unroll
        for (int i = 0; i < N1; ++i) c[i] = tile[i * RS + j];
        contract_s<T, P, CX>(prec, c, t);
#pragma unroll
        for (int a = 0; a < N1; ++a) tile[a * RS + j] = t[a];
    }
    run_sync();
    T zv[KR][VL];
#pragma unroll
    for (int k = 0; k < KR; ++k) load_vec<T, VL>(wl + G::pos(min(VL * (lane + 64 * k), nv - VL)), zv[k]);
#pragma unroll
    for (int k = 0; k < KR; ++k) {
        const int o = VL * (lane + 64 * k), idx = min(o, nv - VL);
        store_vec<T, VL>(z + idx, zv[k]);
        if (COPYP) store_vec<T, VL>(pc + idx, zv[k]);
#pragma unroll
        for (int q = 0; q < VL; ++q) srz += idx + q >= o ? (double)rv[k][q] * (double)zv[k][q] : 0.0;
    }
    run_sync();                                         // the wave's LDS is free for its next run
}

}  // namespace sipg_internal
