// apply_block.hpp -- device pieces that the operator kernels share: the
// workgroup order, block sums, the operator's coefficients, and the geometry
// and direct global -> LDS staging of a block of elements with its halo ring.
#pragma once
#include "sipg_internal.hpp"
#include "basis_constexpr.hpp"
#include "partials.hpp"

#include <utility>

namespace sipg_internal {

__device__ __forceinline__ int xcd_remap(int b, int nblk) {
    // workgroup id b runs on XCD (b % 8); give XCD k the k-th contiguous
    // share of the logical block range.
    const int xcd = b & 7;
    const int idx = b >> 3;
    const int q = nblk >> 3, r = nblk & 7;
    const int start = xcd * q + (xcd < r ? xcd : r);
    return start + idx;
}

// The workgroup's sum, valid in thread 0 (one barrier): the waves' sums,
// then these in order.
template <int NT>
__device__ __forceinline__ double block_sum(double v, double *red) {
    static_assert(NT % 64 == 0, "whole waves");
    constexpr int NW = NT / 64;
    v = wave_total(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 0; i < NW; ++i) s += red[i];
    }
    return s;
}

// Odd LDS row stride (in elements of T) for a (p+1)^2 tile: lanes that read
// the same node of consecutive tiles then hit distinct banks.
__host__ __device__ constexpr int tile_stride(int nq) { return (nq % 2) ? nq : nq + 1; }

// Compile-time geometry of a BX x BY block of degree-P elements.  LDS slots:
// (BY+2) rows of BX tiles for the element rows y0-1 .. y0+BY (slot r*BX + t
// holds element (x0+t, y0-1+r)), then the left halo column (x0-1, y0+k) at
// SL_COL+k and the right one (x0+BX, y0+k) at SL_COL+BY+k.  A block's own
// element (ex, ey) sits in slot (ey+1)*BX+ex, so its up/down neighbours are
// always slot -/+ BX.
template <typename T, int P, int BX, int BY>
struct BlockGeo {
    static constexpr int N1 = P + 1;
    static constexpr int NQ = N1 * N1;
    static constexpr int TS = tile_stride(NQ);
    static constexpr int NE = BX * BY;
    static constexpr int RUN = BX * NQ;                 // values of one row run
    static constexpr int SL_COL = (BY + 2) * BX;
    static constexpr int NS = SL_COL + 2 * BY;
    static constexpr int NT = NE * N1;                  // threads
    static constexpr int LDS = NS * TS;                 // elements of T
};

// Direct global -> LDS staging (global_load_lds_dword) takes a block whose
// LDS image is the concatenation of its row runs and halo-column tiles: no
// row padding, TS == NQ, and whole waves to issue it.
template <typename T, int P, int BX, int BY>
struct BlockDma {
    using G = BlockGeo<T, P, BX, BY>;
    static constexpr bool ok = G::TS == G::NQ && G::NT >= 64;
};

typedef __attribute__((address_space(3))) unsigned lds_dword;

// Direct loads of chunks C... of 64 dwords: lane l moves dword 64C + l of
// src to dword 64C + l of dst.  The chunk offset is the instruction's
// immediate (applied to both addresses), so a group costs one M0 write.
template <int... C>
__device__ __forceinline__ void dma_group(const unsigned *src, lds_dword *dst, std::integer_sequence<int, C...>)
{
    (__builtin_amdgcn_global_load_lds(src, dst, 4, C * 256, 0), ...);
}

// The first N full 64-dword chunks from src (per-lane pointer: base + lane)
// to dst (wave-uniform base), in groups of 16 (immediate offsets < 4 KiB).
template <int N>
__device__ __forceinline__ void dma_chunks(const unsigned *src, lds_dword *dst)
{
    if constexpr (N >= 16) {
        dma_group(src, dst, std::make_integer_sequence<int, 16>{});
        dma_chunks<N - 16>(src + 1024, dst + 1024);
    } else if constexpr (N > 0) {
        dma_group(src, dst, std::make_integer_sequence<int, N>{});
    }
}

// A run of exactly ND dwords: its full chunks, then the lanes of the last
// partial chunk that fall inside the run.
template <int ND>
__device__ __forceinline__ void dma_run(const unsigned *src, lds_dword *dst, int lane)
{
    dma_chunks<ND / 64>(src, dst);
    if constexpr (ND % 64 != 0) {
        if (lane < ND % 64)
            __builtin_amdgcn_global_load_lds(src + (ND / 64) * 64, dst + (ND / 64) * 64, 4, 0, 0);
    }
}

// Issues the loads of block (x0, y0) into the LDS image `lds`; returns
// without waiting.  Every lane of a load instruction writes the dword at
// (LDS base + 4 * lane), so an instruction moves 64 consecutive dwords of
// one row run or halo tile, and only full waves issue them.  Work items
// (BY + 2 row runs, then 2 BY halo tiles) go round-robin over the waves;
// runs and tiles outside the mesh are skipped (their slots are never read
// by a valid element), and a run cut by the right mesh edge loads only the
// elements that exist.
// NW: the number of (full) waves of the workgroup that issue.
template <typename T, int P, int BX, int BY, int NW = BlockGeo<T, P, BX, BY>::NT / 64>
__device__ __forceinline__ void block_issue(T *lds, const T *__restrict__ x, int dimx, int dimy, int x0, int y0)
{
    using G = BlockGeo<T, P, BX, BY>;
    static_assert(BlockDma<T, P, BX, BY>::ok, "direct staging needs unpadded tiles and full waves");
    constexpr int WD = sizeof(T) / 4;                   // dwords per value
    constexpr int NQD = G::NQ * WD, RUND = G::RUN * WD;
    constexpr int CHR = (RUND + 63) / 64;
    constexpr int NITEM = BY + 2 + 2 * BY;
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (wid >= NW) return;
    const unsigned *xd = reinterpret_cast<const unsigned *>(x);
    lds_dword *ld = (lds_dword *)lds;
    const int ncol = dimx - x0 < BX ? dimx - x0 : BX;
    for (int it = wid; it < NITEM; it += NW) {
        if (it < BY + 2) {
            const int gy = y0 - 1 + it;
            if (gy < 0 || gy >= dimy) continue;
            const unsigned *src = xd + ((size_t)gy * dimx + x0) * NQD + lane;
            lds_dword *dst = ld + it * RUND;
            if (ncol == BX) {
                dma_run<RUND>(src, dst, lane);
            } else {
                const int nd = ncol * NQD;
#pragma unroll
                for (int c = 0; c < CHR; ++c)
                    if (c * 64 + lane < nd)
                        __builtin_amdgcn_global_load_lds(src + c * 64, dst + c * 64, 4, 0, 0);
            }
        } else {
            const int k = it - (BY + 2);                // halo tile: left k < BY, right k >= BY
            const bool right = k >= BY;
            const int gy = y0 + (right ? k - BY : k), gx = right ? x0 + BX : x0 - 1;
            if (gy >= dimy || gx < 0 || gx >= dimx) continue;
            dma_run<NQD>(xd + ((size_t)gy * dimx + gx) * NQD + lane, ld + (G::SL_COL + k) * NQD, lane);
        }
    }
}

// Waits for this wave's outstanding vector-memory operations, the direct
// LDS loads included; a barrier after it publishes the staged block.
__device__ __forceinline__ void block_issue_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// The coefficients of the operator on a line (line_math.hpp) as
// compile-time constants: immediates built in scalar registers at each use.
template <typename T, int P>
struct CxCoef {
    static constexpr cx::Tables<P> CT = cx::make_tables<P>();
    static constexpr cx::EvenOdd<P> EO = cx::make_even_odd<P>();
    // E and O are symmetric (K1 symmetric and centrosymmetric); one copy of
    // each pair is used, so the two index orders give the same value
    __device__ T E(int a, int i) const { return (T)(a <= i ? EO.E[a][i] : EO.E[i][a]); }
    __device__ T O(int a, int i) const { return (T)(a <= i ? EO.O[a][i] : EO.O[i][a]); }
    __device__ T DA(int i) const { return (T)EO.DA[i]; }
    __device__ T DB(int i) const { return (T)EO.DB[i]; }
    __device__ T DM() const { return (T)EO.DM; }
    __device__ T w(int i) const { return (T)CT.w[i]; }
};

}  // namespace sipg_internal
