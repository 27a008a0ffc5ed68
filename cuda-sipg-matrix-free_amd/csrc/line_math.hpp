// line_math.hpp -- the SIPG operator on one element line, without its cross
// weight, in even-odd form.
//
// K1 is centrosymmetric and the derivative table antisymmetric (DP[i] =
// -D0[p-i], exactly), so the contraction, the line's end derivatives and the
// face terms all act on the pair sums e = u[i] + u[p-i] and differences
// o = u[i] - u[p-i].  A neighbour enters by its end value t and end
// derivative n on the shared face only (volume_gpu_kernels.hpp:46-83 and
// flux_term6a/6b, sipg_sem_2d_gpu_kernels.hpp:212-247, 279-312).  A boundary
// face is an interior one whose neighbour is the ghost (-t, d) of the line's
// own end (t, d), with half the penalty: 1/2 (t - (-t)) = t, 1/2 (d + d) = d
// and 2 pen / 2 = pen, the one-sided rule, exactly.
#pragma once
#include "apply_block.hpp"

namespace sipg_internal {

template <typename T>
__device__ __forceinline__ T line_fma(T a, T b, T c) {
    if constexpr (sizeof(T) == 8) return __builtin_fma(a, b, c);
    else return __builtin_fmaf(a, b, c);
}

// A line's pair sums and differences, end values and end derivatives.
template <typename T, int P>
struct Line {
    static constexpr int N1 = P + 1, H = N1 / 2, ME = (N1 + 1) / 2;
    T e[ME], o[H];
    T t0, tP, d0, dP;

    template <class C>
    __device__ __forceinline__ void from(const T (&u)[N1], const C &c) {
        T s = 0, b = 0;
#pragma unroll
        for (int i = 0; i < H; ++i) {
            e[i] = u[i] + u[P - i];
            o[i] = u[i] - u[P - i];
            s = line_fma(c.DA(i), e[i], s);
            b = line_fma(c.DB(i), o[i], b);
        }
        if (ME > H) {
            e[ME - 1] = u[H];
            s = line_fma(c.DM(), u[H], s);
        }
        t0 = u[0];
        tP = u[P];
        d0 = s + b;
        dP = b - s;
    }
};

// out = the operator on the line L between the neighbours' (value,
// derivative) (tl, nl) at its lower and (tr, nr) at its upper end; pl, pr:
// pen, or pen / 2 against a ghost.
template <typename T, int P, class C>
__device__ __forceinline__ void line_apply(const Line<T, P> &L, T tl, T nl, T tr, T nr, T pl, T pr, T (&out)[P + 1],
                                           const C &c) {
    constexpr int H = Line<T, P>::H, ME = Line<T, P>::ME;
    const T sl = L.t0 - tl, sr = tr - L.tP;
    const T s0 = T(0.5) * (sl - sr), s1 = T(0.5) * (sl + sr);
#pragma unroll
    for (int a = 0; a < ME; ++a) {
        T ex = (a < H ? c.DA(a) : c.DM()) * s0;
#pragma unroll
        for (int i = 0; i < ME; ++i) ex = line_fma(c.E(a, i), L.e[i], ex);
        if (a < H) {
            T ox = c.DB(a) * s1;
#pragma unroll
            for (int i = 0; i < H; ++i) ox = line_fma(c.O(a, i), L.o[i], ox);
            out[a] = ex + ox;
            out[P - a] = ex - ox;
        } else {
            out[a] = ex;
        }
    }
    out[0] += line_fma(T(0.5), L.d0 + nl, pl * sl);
    out[P] += line_fma(T(-0.5), L.dP + nr, -(pr * sr));
}

}  // namespace sipg_internal
