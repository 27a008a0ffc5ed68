// batch_items.hpp -- the work lists of a batched launch over all degrees:
// item k of the launch is item k - first[g] of group g.
#pragma once
#include "sipg_internal.hpp"

#include <type_traits>

namespace sipg_internal {

// One device function per degree, picked by the (uniform) degree of an item.
template <int P, class F>
__device__ __forceinline__ auto by_degree(int p, F f) {
    if constexpr (P == 1) {
        return f(std::integral_constant<int, 1>{});
    } else {
        if (p == P) return f(std::integral_constant<int, P>{});
        return by_degree<P - 1>(p, f);
    }
}

// A copy of v that the compiler cannot see through.  A loop over items of
// any degree takes its thread index from it in every pass: the lane's
// places in the tiles of every degree, hoisted out of the loop, would fill
// the registers.  (A register move; no memory access.)
__device__ __forceinline__ int opaque(int v) {
    int r;
    asm volatile("v_mov_b32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

// first[g] = items of the groups before g; returns the number of all items.
// One barrier, and none for a single group, whose first is not stored; first
// stays valid to the kernel's end.
__device__ __forceinline__ int batch_offsets(const batch_groups &G, int (&first)[kMaxDegree + 1]) {
    if (G.n == 1) return *G.g[0].count;
    if (threadIdx.x < 64) {
        const int l = threadIdx.x;
        int c = 0;
#pragma unroll
        for (int g = 0; g < kMaxDegree; ++g)
            if (l == g && g < G.n) c = *G.g[g].count;
        int s = c;
#pragma unroll
        for (int off = 1; off <= kMaxDegree; off <<= 1) {    // (up to the lane after the last group)
            const int o = __shfl_up(s, off, 64);
            if (l >= off) s += o;
        }
        if (l <= kMaxDegree) first[l] = s - c;          // the lane after the last group: the total
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(first[G.n]);
}

// the group of item k, uniform over the wave, and the item's place in it
__device__ __forceinline__ int batch_group_at(const batch_groups &G, const int (&first)[kMaxDegree + 1], int k,
                                              int &at) {
    at = k;
    if (G.n == 1) return 0;
    const int l = threadIdx.x & 63;
    const bool in = l >= 1 && l < G.n && k >= first[min(l, kMaxDegree)];
    const int g = __builtin_amdgcn_readfirstlane(__popcll(__ballot(in)));
    at = k - __builtin_amdgcn_readfirstlane(first[g]);
    return g;
}

}  // namespace sipg_internal
