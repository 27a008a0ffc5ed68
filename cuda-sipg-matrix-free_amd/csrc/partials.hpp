// partials.hpp -- the first stage of every reduction of block sums, and the
// compensated update of an iterate.
#pragma once
#include <hip/hip_runtime.h>

namespace sipg_internal {

// Sum over a whole wave, in every lane, in the order of the row shifts: rows of 16 lanes, then
// across rows; the total is read from lane 63.  (Register moves inside the
// SIMD: a cross-lane exchange through LDS costs several times as much, six
// times over: 0.3 us at the end of a kernel of 4.)
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, true);
    return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_total(double v) {
    v = dpp_add<0x111, 0xf>(v);      // row_shr:1
    v = dpp_add<0x112, 0xf>(v);      // row_shr:2
    v = dpp_add<0x114, 0xf>(v);      // row_shr:4
    v = dpp_add<0x118, 0xf>(v);      // row_shr:8: lane 15 of each row holds its sum
    v = dpp_add<0x142, 0xa>(v);      // row_bcast:15 into rows 1 and 3
    v = dpp_add<0x143, 0xc>(v);      // row_bcast:31 into rows 2 and 3
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                            __builtin_amdgcn_readlane(__double2loint(v), 63));
}

// Thread t's share of part[b] + ... + part[e-1]: the entries b + t,
// b + t + NT, b + t + 2 NT, ... in eight accumulators, so that eight loads
// are in flight at once (a loop with one accumulator waits for each load
// before issuing the next: (e - b) / NT dependent round trips to the cache,
// which for a few thousand block sums is several microseconds at the start
// of every workgroup that needs them).  Added in a fixed order.
template <int NT>
__device__ __forceinline__ double strided_sum(const double *__restrict__ part, int b, int e) {
    double a[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    int i = b + (int)threadIdx.x;
    for (; i + 7 * NT < e; i += 8 * NT) {
#pragma unroll
        for (int u = 0; u < 8; ++u) a[u] += part[i + u * NT];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
        if (i + u * NT < e) a[u] += part[i + u * NT];
    return ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
}

// The sums of K arrays of block sums (np[k] values each), returned to every
// thread of a workgroup of NT, in one exchange: the K wave sums are formed
// together and cross the workgroup behind one barrier, where K separate
// reductions would wait for two each.  Loads past the end of an array are
// clamped to its last value and discarded, so that all of them are in
// flight at once.  Fixed order, as strided_sum.
template <int NT, int K>
__device__ __forceinline__ void multi_sum(const double *const (&part)[K], const int (&np)[K], double (&out)[K]) {
    __shared__ double red[K][NT / 64];
    double v[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        double a[4] = {0.0, 0.0, 0.0, 0.0};
        for (int i = (int)threadIdx.x; i < np[k]; i += 4 * NT) {
            double t[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) t[u] = part[k][min(i + u * NT, np[k] - 1)];
#pragma unroll
            for (int u = 0; u < 4; ++u) a[u] += i + u * NT < np[k] ? t[u] : 0.0;
        }
        v[k] = (a[0] + a[1]) + (a[2] + a[3]);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = wave_total(v[k]);
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int k = 0; k < K; ++k) red[k][threadIdx.x >> 6] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < NT / 64; ++i) s += red[k][i];
        out[k] = s;
    }
}

// VL consecutive values at an address that is aligned to one value only
// (one 16-byte access where the hardware allows it, which on gfx950 is any
// multiple of four bytes).
template <typename T, int VL>
struct __attribute__((packed, aligned(sizeof(T)))) VecU {
    T v[VL];
};
template <typename T, int VL>
__device__ __forceinline__ void load_vec(const T *p, T (&r)[VL]) {
    const VecU<T, VL> v = *reinterpret_cast<const VecU<T, VL> *>(p);
#pragma unroll
    for (int i = 0; i < VL; ++i) r[i] = v.v[i];
}
template <typename T, int VL>
__device__ __forceinline__ void store_vec(T *p, const T (&r)[VL]) {
    VecU<T, VL> v;
#pragma unroll
    for (int i = 0; i < VL; ++i) v.v[i] = r[i];
    *reinterpret_cast<VecU<T, VL> *>(p) = v;
}

// xh += a p with the rounding errors kept in xl, so that xh + xl carries
// the running sum to about twice the working precision: the product's
// error from an fma, the sum's by Knuth's TwoSum (both exact).  Contraction
// is off so that the error terms are formed as written.  Used for the
// increments of the single-problem solvers: accumulated plainly, their
// rounding (eps |x| per step, amplified by |A|) leaves b - A x about 1e-9
// of |b| away from the recursion at 256 x 256, p = 8.
template <typename T>
__device__ __forceinline__ void comp_axpy(T &xh, T &xl, T a, T pv) {
#pragma clang fp contract(off)
    const T t = a * pv;
    const T tp = fma(a, pv, -t);
    const T s = xh + t;
    const T bb = s - xh;
    const T e = (xh - (s - bb)) + (t - bb);
    xh = s;
    xl = xl + (e + tp);
}

}  // namespace sipg_internal
