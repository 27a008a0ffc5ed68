// kernels_apply.hip -- the fused SIPG operator apply y = A x for gfx950, and
// the choice among its kernels.
//
// The reference applies A with three launches (sipg_sem_2d.hpp:167-201):
// `volume` (volume_gpu_kernels.hpp:9-86, one thread per dof, O(p^2) work per
// dof with the 1-D stiffness rebuilt in the inner loop), then `flux_term6a`
// and `flux_term6b` (sipg_sem_2d_gpu_kernels.hpp:189-316, one thread per
// element, read-modify-write of the output).  Here one kernel does all of
// it in a single pass over the input and a single write of the output, on
// element-major vectors: the (p+1)^2 values of element e = dimx*y + x are
// contiguous at e*(p+1)^2 + i1*(p+1) + i2.
//
// This file has the kernel of every compiled degree, strips of whole
// elements per wave marched in y (strip_apply.hpp).  Even degrees up to 8, in
// FP32 up to 12, also have the block-staged kernel of kernels_apply_wave.hip.
//
// The discrete operator is exactly the reference's (see the oracle and the
// tests): Y = K1 U W + W U K1 + face terms of flux_term6a/6b, with the
// same interior (1/2-average, 2*pen) and Dirichlet (one-sided, pen) rules.
//
// Block -> strip mapping is XCD-aware: the eight XCDs of an MI355X take
// consecutive workgroup ids round-robin, so the ids are remapped such that
// each XCD walks neighbouring strips of consecutive bands and the rows they
// share are mostly in its own L2.
#include "strip_apply.hpp"
#include "strip_bands.hpp"

#include <atomic>

namespace sipg_internal {

// Workgroup (strip, band): EPW elements wide, the band's rows in y.
template <typename T, int P, bool DOT>
__global__ __launch_bounds__(256)
void apply_strip_kernel(const T *__restrict__ x, T *__restrict__ y, int dimx, int dimy, int nstrip, int nband, T pen,
                        double *__restrict__ partials, const cg_state *__restrict__ st, int slot)
{
    using G = StripGeo<T, P>;
    __shared__ __attribute__((aligned(16))) T lds[G::LDS];
    __shared__ T exch[G::EXCH];
    __shared__ double red[G::W];
    if (DOT) {
        if (st->s[slot].done | st->err) return;
    }
    const int b = xcd_remap(blockIdx.x, nstrip * nband);
    const int band = b / nstrip, x0 = (b - band * nstrip) * G::EPW;
    const int yA = (int)((int64_t)dimy * band / nband), yB = (int)((int64_t)dimy * (band + 1) / nband);
    const double dot = strip_apply<T, P, DOT>(x, y, dimx, dimy, pen, x0, min(G::EPW, dimx - x0), yA, yB, lds, exch,
                                                 threadIdx.x);
    if (DOT) {
        const double bs = block_sum<64 * G::W>(dot, red);
        if (threadIdx.x == 0) partials[blockIdx.x] = bs;
    }
}

namespace {

// Workgroups of one kernel that the device holds at once, cached per device
// (occupancy depends only on the kernel).
template <typename T, int P>
int resident_groups() {
    constexpr int kMaxDev = 64;
    static std::atomic<int> cache[kMaxDev];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDev) dev = 0;
    int g = cache[dev].load(std::memory_order_relaxed);
    if (g > 0) return g;
    int cus = 0, per = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per, reinterpret_cast<const void *>(&apply_strip_kernel<T, P, true>), 256, 0) != hipSuccess)
        per = 0;
    g = (cus > 0 ? cus : 1) * (per > 0 ? per : 1);
    cache[dev].store(g, std::memory_order_relaxed);
    return g;
}

// Bands per strip (strip_bands.hpp).  Measured, us for bands so chosen /
// twice as many / half as many: FP64 201 x 150, p = 7 8.7 / 10.9 / 10.0;
// 131 x 77, p = 12 11.8 / 12.3 / 13.7.
template <typename T, int P>
int num_bands(int dimx, int dimy) {
    constexpr int EPW = StripGeo<T, P>::EPW;
    return strip_bands((dimx + EPW - 1) / EPW, dimy, resident_groups<T, P>(), kMaxPartials);
}

template <typename T, int P>
int launch_one(const void *x, void *y, int dimx, int dimy, double pen, double *partials, const cg_state *st, int slot,
               hipStream_t s)
{
    constexpr int EPW = StripGeo<T, P>::EPW;
    const int nstrip = (dimx + EPW - 1) / EPW, nband = num_bands<T, P>(dimx, dimy);
    const dim3 grid(nstrip * nband), block(256);
    if (partials)
        hipLaunchKernelGGL((apply_strip_kernel<T, P, true>), grid, block, 0, s, (const T *)x, (T *)y, dimx, dimy,
                           nstrip, nband, (T)pen, partials, st, slot);
    else
        hipLaunchKernelGGL((apply_strip_kernel<T, P, false>), grid, block, 0, s, (const T *)x, (T *)y, dimx, dimy,
                           nstrip, nband, (T)pen, partials, st, slot);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

// Grid size of the fused apply + p.Ap launch = number of p.Ap partials.
template <typename T, int P>
int nblocks_one(int dimx, int dimy) {
    constexpr int EPW = StripGeo<T, P>::EPW;
    return (dimx + EPW - 1) / EPW * num_bands<T, P>(dimx, dimy);
}

template <typename T, int... Ps>
struct Dispatch;

template <typename T>
struct Dispatch<T> {
    static int launch(int, const void *, void *, int, int, double, double *, const cg_state *, int, hipStream_t) {
        return SIPG_ERR_UNSUPPORTED;
    }
    static int nblocks(int, int, int) { return -1; }
};

template <typename T, int P0, int... Ps>
struct Dispatch<T, P0, Ps...> {
    static int launch(int p, const void *x, void *y, int dimx, int dimy, double pen, double *partials,
                      const cg_state *st, int slot, hipStream_t s) {
        if (p == P0) return launch_one<T, P0>(x, y, dimx, dimy, pen, partials, st, slot, s);
        return Dispatch<T, Ps...>::launch(p, x, y, dimx, dimy, pen, partials, st, slot, s);
    }
    static int nblocks(int p, int dimx, int dimy) {
        if (p == P0) return nblocks_one<T, P0>(dimx, dimy);
        return Dispatch<T, Ps...>::nblocks(p, dimx, dimy);
    }
};

template <typename T>
using AllDegrees = Dispatch<T, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16>;

}  // namespace

int resolve_kernel(int dtype, int p, int kernel) {
    if (kernel == SIPG_KERNEL_WAVE) return wave_apply_available(dtype, p) ? SIPG_KERNEL_WAVE : SIPG_KERNEL_VALU;
    if (kernel == SIPG_KERNEL_MFMA) return mfma_apply_available(dtype, p) ? SIPG_KERNEL_MFMA : SIPG_KERNEL_VALU;
    if (kernel == SIPG_KERNEL_VALU) return SIPG_KERNEL_VALU;
    // AUTO: the matrix cores at p = 15 in FP32, the block-staged kernel at
    // even p <= 8 and in FP32 <= 12, strips elsewhere.  Strips store a lane's
    // column, sizeof(T) (p+1) bytes to a segment, which costs most where it is
    // short and the lines leave the caches partly written: 1024 x 1024, p = 8
    // FP64 322 against 279 us, FP32 256 x 256, p = 8 16.2 against 12.1.  At p = 15
    // in FP32 strips take 3.9 against 2.8 us at 4 x 4, 4.5 against 4.8 at 64 x 64
    // and 8.9 against 10.9 at 128 x 128, and are 5 % further from 64 bits (6.5e-8
    // against 6.2e-8 on uniform values): the matrix cores stay.
    if (mfma_apply_available(dtype, p)) return SIPG_KERNEL_MFMA;
    if (wave_apply_available(dtype, p)) return SIPG_KERNEL_WAVE;
    return SIPG_KERNEL_VALU;
}

int apply_num_blocks(int dtype, int p, int dimx, int dimy, int kernel) {
    if (p > kMaxDegree) return p <= kMaxGenericDegree ? generic_apply_num_blocks(dtype, p, dimx, dimy) : -1;
    const int k = resolve_kernel(dtype, p, kernel);
    if (k == SIPG_KERNEL_MFMA) return mfma_apply_num_blocks(dimx, dimy);
    if (k == SIPG_KERNEL_WAVE) return wave_apply_num_blocks(dtype, p, dimx, dimy);
    return dtype == SIPG_F64 ? AllDegrees<double>::nblocks(p, dimx, dimy)
                             : AllDegrees<float>::nblocks(p, dimx, dimy);
}

int launch_apply(int dtype, int p, const void *x, void *y, const void *tab, int dimx, int dimy,
                 double pen, double *partials, const cg_state *st, int slot, hipStream_t s, int kernel)
{
    // above the compiled degrees: the run-time-table operator, whatever the
    // setting (its only implementation)
    if (p > kMaxDegree)
        return launch_apply_generic(dtype, p, x, y, tab, dimx, dimy, pen, partials, st, slot, s);
    const int k = resolve_kernel(dtype, p, kernel);
    if (k == SIPG_KERNEL_MFMA)
        return launch_apply_mfma(dtype, p, x, y, dimx, dimy, pen, partials, st, slot, s);
    if (k == SIPG_KERNEL_WAVE)
        return launch_apply_wave(dtype, p, x, y, dimx, dimy, pen, partials, st, slot, s);
    if (dtype == SIPG_F64)
        return AllDegrees<double>::launch(p, x, y, dimx, dimy, pen, partials, st, slot, s);
    return AllDegrees<float>::launch(p, x, y, dimx, dimy, pen, partials, st, slot, s);
}

}  // namespace sipg_internal
