// kernels_apply_wave.hip -- the fused SIPG operator apply y = A x with
// wave-owned elements on a block staged in LDS (volume + flux_term6a +
// flux_term6b of the reference, volume_gpu_kernels.hpp:9-86,
// sipg_sem_2d_gpu_kernels.hpp:189-316), for even degrees up to 8, in FP32
// up to 12.
//
// The same line arithmetic as the strip kernel (line_math.hpp), to the bit,
// another work split: a wave holds EPW = 64 / (p+1) whole elements (7 at
// p = 8), one block row, with lane (s, j) = s (p+1) + j on line j of element
// s.  A workgroup of BY waves owns an EPW x BY block, staged in LDS with
// its halo ring by direct global -> LDS loads.  Neighbours in x are lanes of
// the same wave (the block's sides: their staged tiles), neighbours in y
// staged tiles.  Because each element's lines sit in one wave, the assembly
// of the output tile and the copy-out of the block row are wave-local: a
// block costs two workgroup barriers (the staged block is complete; every
// wave is done reading it).  Whole rows are stored as contiguous runs, which
// is what a store stream to memory needs.
//
// Launch: one block per workgroup, one LDS image per workgroup, so several
// workgroups share a CU and one computes while another streams its block
// in.  Block -> workgroup mapping is XCD-aware as in the other operator
// kernels.  Even degrees (unpadded tiles, which the direct loads need).
#include "line_math.hpp"

#include <type_traits>

namespace sipg_internal {

template <typename T, int P, int BY, bool DOT>
__global__ __launch_bounds__(64 * BY)
void apply_kernel_wave(const T *__restrict__ x, T *__restrict__ y, int dimx, int dimy, int nbx, int nblk, T pen,
                       double *__restrict__ partials, const cg_state *__restrict__ st, int slot)
{
    constexpr int N1 = P + 1, NQ = N1 * N1, BX = 64 / N1;
    using G = BlockGeo<T, P, BX, BY>;
    static_assert(G::TS == NQ, "wave-owned elements need unpadded tiles (even p)");
    __shared__ T lds[G::LDS];
    __shared__ double red[BY];

    if (DOT) {
        if (st->s[slot].done | st->err) return;
    }
    const int b = xcd_remap(blockIdx.x, nblk);
    const int x0 = (b % nbx) * BX, y0 = (b / nbx) * BY;
    block_issue<T, P, BX, BY, BY>(lds, x, dimx, dimy, x0, y0);      // every wave issues

    const CxCoef<T, P> coef{};
    const int lane = threadIdx.x & 63;
    const int ey = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int s = lane / N1, j = lane - s * N1;
    const int ex = s < BX ? s : BX - 1;                 // lanes past the last element: copies of it
    const int gx = x0 + ex, gy = y0 + ey;
    const bool valid = s < BX && gx < dimx && gy < dimy;
    const bool Lb = gx == 0, Rb = gx == dimx - 1;
    const int sl = (ey + 1) * BX + ex;
    T *tile = lds + sl * NQ;
    const bool isR = s >= BX - 1;                       // the side tile that this lane reads
    const T *side = lds + (G::SL_COL + (isR ? BY : 0) + ey) * NQ;
    const T pL = Lb ? T(0.5) * pen : pen, pR = Rb ? T(0.5) * pen : pen;
    const T wj = coef.w(j);

    block_issue_wait();
    __syncthreads();                                    // the staged block is complete
    T u[N1], q[N1], ox[N1], oy[N1];
    {
        Line<T, P> V, Q;
#pragma unroll
        for (int i = 0; i < N1; ++i) q[i] = tile[j * N1 + i];
        V.from(q, coef);
        // below (y grows downwards) and above: staged rows, or the ghost
        T tB = -V.t0, nB = V.d0, tA = -V.tP, nA = V.dP, pB = T(0.5) * pen, pA = pB;
        if (gy < dimy - 1) {
#pragma unroll
            for (int i = 0; i < N1; ++i) q[i] = tile[BX * NQ + j * N1 + i];
            Q.from(q, coef);
            tB = Q.tP;
            nB = Q.dP;
            pB = pen;
        }
        if (gy > 0) {
#pragma unroll
            for (int i = 0; i < N1; ++i) q[i] = (tile - BX * NQ)[j * N1 + i];
            Q.from(q, coef);
            tA = Q.t0;
            nA = Q.d0;
            pA = pen;
        }
        line_apply<T, P>(V, tB, nB, tA, nA, pB, pA, oy, coef);
    }
    {
        Line<T, P> U, Q;
#pragma unroll
        for (int i = 0; i < N1; ++i) {
            u[i] = tile[i * N1 + j];
            q[i] = side[i * N1 + j];
        }
        U.from(u, coef);
        Q.from(q, coef);
        T tL = __shfl(U.tP, lane - N1, 64), nL = __shfl(U.dP, lane - N1, 64);
        T tR = __shfl(U.t0, lane + N1, 64), nR = __shfl(U.d0, lane + N1, 64);
        if (s == 0) {
            tL = Lb ? -U.t0 : Q.tP;
            nL = Lb ? U.d0 : Q.dP;
        }
        if (isR) {
            tR = Q.t0;
            nR = Q.d0;
        }
        if (Rb) {
            tR = -U.tP;
            nR = U.dP;
        }
        line_apply<T, P>(U, tL, nL, tR, nR, pL, pR, ox, coef);
    }
    __syncthreads();                                    // every wave is done reading the block

    // wave-local from here: the element's tile takes the row results, then
    // each lane adds its column's
    if (valid) {
#pragma unroll
        for (int a = 0; a < N1; ++a) tile[j * N1 + a] = wj * oy[a];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    double dot = 0.0;
    if (valid) {
#pragma unroll
        for (int a = 0; a < N1; ++a) {
            const T yv = line_fma(wj, ox[a], tile[a * N1 + j]);
            tile[a * N1 + j] = yv;
            if (DOT) dot += (double)u[a] * (double)yv;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // this wave's block row is one contiguous run of ncol tiles in y
    if (gy < dimy) {
        const int ncol = dimx - x0 < BX ? dimx - x0 : BX;
        const int n = ncol * NQ;
        const T *src = lds + (ey + 1) * BX * NQ;
        T *dst = y + ((size_t)gy * dimx + x0) * NQ;
        // (all LDS reads first: a read inside the bounds check of its store
        // would wait for its own round trip nine times over)
        constexpr int KO = (BX * NQ + 63) / 64;
        static_assert((BY + 1) * BX * NQ + 64 * KO <= G::LDS, "the last read stays inside the image");
        T o[KO];
#pragma unroll
        for (int k = 0; k < KO; ++k) o[k] = src[lane + 64 * k];
#pragma unroll
        for (int k = 0; k < KO; ++k) {
            const int idx = lane + 64 * k;
            if (idx < n) dst[idx] = o[k];
        }
    }
    if (DOT) {
        const double bs = block_sum<64 * BY>(dot, red);
        if (threadIdx.x == 0) partials[blockIdx.x] = bs;
    }
}

namespace {

// Rows of elements per workgroup (waves), with one LDS image of (rows + 2) *
// BX + 2 rows tiles.  Measured at 256 x 256 and 1024 x 1024, p = 8, FP64, before
// a run's loads were issued ahead of its use (us per apply): 2: 22.2 / 281,
// 3: 21.7 / 277, 4: 21.1 / 277, 6: 24.3 / 301, 8: 22.8 / 297, 10: 26.9 / 374.
constexpr int kRows = 4;

template <typename T, int P, bool DOT>
void launch_wave(const void *x, void *y, int dimx, int dimy, double pen, double *partials, const cg_state *st,
                 int slot, hipStream_t s)
{
    constexpr int BX = 64 / (P + 1), BY = kRows;
    const int nbx = (dimx + BX - 1) / BX, nby = (dimy + BY - 1) / BY;
    const int nblk = nbx * nby;
    hipLaunchKernelGGL((apply_kernel_wave<T, P, BY, DOT>), dim3(nblk), dim3(64 * BY), 0, s, (const T *)x, (T *)y, dimx,
                       dimy, nbx, nblk, (T)pen, partials, st, slot);
}

template <typename T, int P>
int wave_blocks(int dimx, int dimy) {
    constexpr int BX = 64 / (P + 1), BY = kRows;
    return ((dimx + BX - 1) / BX) * ((dimy + BY - 1) / BY);
}

// f(std::integral_constant<int, P>) for a degree that has the kernel, else
// `none`.  FP32 at p = 10 and 12 too: strips there take 8.7 against 6.8 us and
// 10.7 against 7.6 at 128 x 128, 27.4 against 17.7 and 36.8 against 23.9 at
// 300 x 300.  In FP64 they are level or ahead (p = 12, 200 x 200: 23.9 against
// 25.8).
template <typename T, class F>
int by_wave_degree(int p, F f, int none) {
    if (p == 2) return f(std::integral_constant<int, 2>{});
    if (p == 4) return f(std::integral_constant<int, 4>{});
    if (p == 6) return f(std::integral_constant<int, 6>{});
    if (p == 8) return f(std::integral_constant<int, 8>{});
    if constexpr (sizeof(T) == 4) {
        if (p == 10) return f(std::integral_constant<int, 10>{});
        if (p == 12) return f(std::integral_constant<int, 12>{});
    }
    return none;
}

template <typename T>
int dispatch(int p, const void *x, void *y, int dimx, int dimy, double pen, double *partials, const cg_state *st,
             int slot, hipStream_t s)
{
    return by_wave_degree<T>(p, [&](auto deg) {
        constexpr int P = decltype(deg)::value;
        if (partials) launch_wave<T, P, true>(x, y, dimx, dimy, pen, partials, st, slot, s);
        else launch_wave<T, P, false>(x, y, dimx, dimy, pen, partials, st, slot, s);
        return (int)SIPG_OK;
    }, SIPG_ERR_UNSUPPORTED);
}

template <typename T>
int blocks(int p, int dimx, int dimy) {
    return by_wave_degree<T>(p, [&](auto deg) { return wave_blocks<T, decltype(deg)::value>(dimx, dimy); }, -1);
}

}  // namespace

bool wave_apply_available(int dtype, int p) {
    auto yes = [](auto) { return 1; };
    return dtype == SIPG_F64 ? by_wave_degree<double>(p, yes, 0) : by_wave_degree<float>(p, yes, 0);
}

int wave_apply_num_blocks(int dtype, int p, int dimx, int dimy) {
    if (!wave_apply_available(dtype, p)) return -1;
    return dtype == SIPG_F64 ? blocks<double>(p, dimx, dimy) : blocks<float>(p, dimx, dimy);
}

int launch_apply_wave(int dtype, int p, const void *x, void *y, int dimx, int dimy, double pen, double *partials,
                      const cg_state *st, int slot, hipStream_t s)
{
    if (!wave_apply_available(dtype, p)) return SIPG_ERR_UNSUPPORTED;
    const int rc = dtype == SIPG_F64 ? dispatch<double>(p, x, y, dimx, dimy, pen, partials, st, slot, s)
                                     : dispatch<float>(p, x, y, dimx, dimy, pen, partials, st, slot, s);
    if (rc) return rc;
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

}  // namespace sipg_internal
