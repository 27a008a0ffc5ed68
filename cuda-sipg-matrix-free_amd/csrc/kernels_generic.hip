// kernels_generic.hip -- the SIPG operator y = A x for any degree up to
// kMaxGenericDegree (63, the reference's 64-point LGL tables,
// device_const.hpp:10-18), on run-time tables: the degrees above the
// compiled fused kernels (volume_gpu_kernels.hpp:9-86 + flux_term6a/6b,
// sipg_sem_2d_gpu_kernels.hpp:189-316).
//
// Two launches per apply.  (1) face_derivs: per element and line j the
// four normal derivatives on its sides, dx0[j] = sum_i D0[i] u(i,j),
// dxN[j] = sum_i DN[i] u(i,j), dy0[j] = sum_i D0[i] u(j,i), dyN[j] = sum_i
// DN[i] u(j,i) (D0[i] = phi_i'(-1), DN[i] = phi_i'(+1)), into a face buffer
// of 4 (p+1) values per element.  (2) apply: per element, the tile in LDS,
// the neighbours' traces from x and their derivatives from the face buffer,
// then every output
//   Y(i1,i2) = sum_i w[i2] K1[i][i1] U(i,i2) + w[i1] K1[i][i2] U(i1,i)
//            + D0[i1] ev[i2] + DN[i1] fv[i2] + D0[i2] g[i1] + DN[i2] h[i1]
//            + side corrections on the element's own boundary lines,
// with ev/fv/g/h the weighted jumps on the left/right/lower/upper sides
// and a/b/c/d the averaged normal derivatives (the reference's flux terms).
//
// The sums over i are products of (p+1) x (p+1) matrices and run on the
// matrix cores, in 2 to 4 tiles of 16 a side, for either type in FP64: its
// instruction takes no longer than FP32's here (v_mfma_f64_16x16x4f64 and
// v_mfma_f32_16x16x4f32, 32 cycles each), and FP32 sums in that order were 5 %
// further off than one multiply-add after the other.  A workgroup has one wave
// to a row of output tiles; K1 stays in registers for all elements, so that a
// step of four i costs NT + 1 LDS reads for 2 NT instructions.  The face terms are one more step, [D0 DN g h]
// times [ev; fv; D0; DN]; the corrections are added on the boundary lines only
// (as products with unit vectors they carried a NaN or an infinity of a
// neighbour's into whole lines: 0 times NaN).  The next element's values are
// in flight meanwhile.
//
// Bound: latency, with two or three waves per SIMD beside K1 in registers (20
// million unknowns in FP64 at p = 20: 148 us here and 65 in face_derivs, for
// 160 MB read by each and 160 MB written).  us an apply, with a thread to an
// output and every operand of its 4 (p+1) multiply-adds from memory and LDS
// before, and now: FP64 213 x 213, p = 20 780, 213; 135 x 135, p = 32 1016, 263;
// 70 x 70, p = 63 1334, 186; 6 x 6, p = 20 14.3, 9.4; FP32 213 x 213, p = 20
// 574, 193.  Waves per SIMD (launch bounds): without the bound p = 20 240, p = 32
// 338.
//
// One workgroup per element in a grid-stride loop over the workgroups that the
// device holds, so that the fused p.Ap partials stay within the partial buffer.
#include "apply_block.hpp"
#include "batch_items.hpp"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace sipg_internal {

namespace {

constexpr int kGenThreads = 256;

// run-time table views (the op's table layout: w, K1, D0, DP, z)
template <typename T>
struct RtTab {
    const T *w, *K1, *D0, *DN;
    __device__ RtTab(const T *tab, int n1)
        : w(tab), K1(tab + n1), D0(tab + n1 + n1 * n1), DN(tab + 2 * n1 + n1 * n1) {}
};

// Waves 0 and 2 sum along x, 1 and 3 along y, over half of the line each:
// lane j has line j.
template <typename T>
__global__ __launch_bounds__(kGenThreads) void face_derivs_kernel(int n1, const T *__restrict__ x,
                                                                  const T *__restrict__ tab, T *__restrict__ face,
                                                                  int noe, const cg_state *__restrict__ st, int slot)
{
    if (st && (st->s[slot].done | st->err)) return;
    constexpr int MV = 64 * 64 / kGenThreads;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    __shared__ T half1[2][2][64];
    T *U = reinterpret_cast<T *>(smem);
    const RtTab<T> t(tab, n1);
    const int nq = n1 * n1, ld = n1 | 1;                          // (odd: lines hit distinct banks)
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int dir = w & 1, lo = w < 2 ? 0 : n1 / 2, hi = w < 2 ? n1 / 2 : n1;
    int pos[MV];
    T v[MV];
#pragma unroll
    for (int i = 0; i < MV; ++i) {
        const int k = threadIdx.x + i * kGenThreads, row = k / n1;
        pos[i] = row * ld + (k - row * n1);
    }
    auto load = [&](int e) {
        const T *ue = x + (int64_t)e * nq;
#pragma unroll
        for (int i = 0; i < MV; ++i)
            if (i * kGenThreads < nq) v[i] = ue[min((int)threadIdx.x + i * kGenThreads, nq - 1)];
    };
    int e = xcd_remap(blockIdx.x, gridDim.x);
    if (e < noe) load(e);
    for (; e < noe; e += gridDim.x) {
#pragma unroll
        for (int i = 0; i < MV; ++i)
            if ((int)threadIdx.x + i * kGenThreads < nq) U[pos[i]] = v[i];
        __syncthreads();
        if (e + (int)gridDim.x < noe) load(e + gridDim.x);
        T s0 = 0, sN = 0;
        if (lane < n1) {
            const T *u = U + (dir ? lane * ld : lane);
            const int step = dir ? 1 : ld;
#pragma unroll 4
            for (int i = lo; i < hi; ++i) {
                const T uv = u[i * step];
                s0 += t.D0[i] * uv;
                sN += t.DN[i] * uv;
            }
        }
        if (w >= 2) {
            half1[dir][0][lane] = s0;
            half1[dir][1][lane] = sN;
        }
        __syncthreads();
        if (w < 2 && lane < n1) {
            T *fe = face + (int64_t)e * 4 * n1 + 2 * dir * n1 + lane;
            fe[0] = s0 + half1[dir][0][lane];
            fe[n1] = sN + half1[dir][1][lane];
        }
    }
}

// a 16 x 16 accumulator: register r of lane l holds D[4 r + l / 16][l % 16]
typedef double gd4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ gd4 gmul(double a, double b, gd4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// face buffer of element e: [dx0 | dxN | dy0 | dyN], n1 each.  NT =
// ceil(n1 / 16) waves; wave ti has the output tiles (ti, (ti + t) % NT).
template <typename T, int NT, bool DOT>
__global__ __launch_bounds__(64 * NT, NT == 2 ? 3 : NT == 3 ? 2 : 1) void apply_generic_kernel(int n1, const T *__restrict__ x, T *__restrict__ y,
                                                                const T *__restrict__ tab,
                                                                const T *__restrict__ face, int dimx, int dimy, T pen,
                                                                double *__restrict__ partials,
                                                                const cg_state *__restrict__ st, int slot)
{
    if (DOT) {
        if (st->s[slot].done | st->err) return;
    }
    constexpr int NTH = 64 * NT, D = 16 * NT, LD = D + 1, NK = 4 * NT;
    constexpr int MV = D * D / NTH;                               // values of a tile per thread
    __shared__ double U[D * LD];                                      // zero beyond n1
    __shared__ double F[8][D];                                        // the face steps' factors, zero beyond n1
    __shared__ double red[NT];
    const int nq = n1 * n1, N = n1 - 1;
    const RtTab<T> t(tab, n1);
    const int noe = dimx * dimy;
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int ti = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int i = tid; i < D * LD; i += NTH) U[i] = 0.0;
    for (int i = tid; i < 8 * D; i += NTH) F[i / D][i % D] = 0.0;

    int col[NT];                                                  // this lane's column of tile t
    double K[NK][NT], dE[NT], wc[NT], wr[4];
    const int o = lk & 1;                                         // this lane's side of a pair
    const bool own = lk < 2;
    // the tile that holds row (or column) N, another than tile 0 (N > 16), and
    // where this wave's boundary row sits in it
    const int tN = N >> 4, rS = ti == 0 ? 0 : (N & 15) >> 2, lkS = ti == 0 ? 0 : N & 3;
#pragma unroll
    for (int c = 0; c < NT; ++c) {
        const int tj = ti + c < NT ? ti + c : ti + c - NT;
        col[c] = 16 * tj + li;
        dE[c] = col[c] <= N ? (double)(o ? t.DN : t.D0)[col[c]] : 0.0;
        wc[c] = col[c] <= N ? (double)t.w[col[c]] : 0.0;
#pragma unroll
        for (int k = 0; k < NK; ++k) K[k][c] = 4 * k + lk <= N && col[c] <= N ? (double)t.K1[(4 * k + lk) * n1 + col[c]] : 0.0;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = 16 * ti + 4 * r + lk;
        wr[r] = row <= N ? (double)t.w[row] : 0.0;
    }
    // one entry of the faces per thread (4 n1 <= NTH): side 0 left, 1 right,
    // 2 lower (y = 0: the next row down), 3 upper; line j
    const int side = min(tid / n1, 3), j = min(tid - side * n1, N);
    const bool hasf = tid < 4 * n1;
    const int near = side == 0 ? j : side == 1 ? N * LD + j : side == 2 ? j * LD : j * LD + N;    // own trace, in U
    const int far = side == 0 ? N * n1 + j : side == 1 ? j : side == 2 ? j * n1 + N : j * n1;     // the neighbour's
    const double wj = t.w[j], pn = pen;

    // k / n1 = (k rn1) >> 18 for k < 4096 and n1 <= 64
    const unsigned rn1 = ((1u << 18) + n1 - 1) / n1;
    T v[MV], dn = 0, dnb = 0, tnb = 0;
    bool bnd = false;
    auto load = [&](int e) {
        const T *ue = x + (int64_t)e * nq;
#pragma unroll
        for (int i = 0; i < MV; ++i)
            if (i * NTH < nq) v[i] = ue[min(tid + i * NTH, nq - 1)];
        const int row = e / dimx, cx = e - row * dimx;
        bnd = side == 0 ? cx == 0 : side == 1 ? cx == dimx - 1 : side == 2 ? row == dimy - 1 : row == 0;
        const int64_t en = bnd ? e : side == 0 ? e - 1 : side == 1 ? e + 1 : side == 2 ? e + dimx : e - dimx;
        dn = face[((int64_t)e * 4 + side) * n1 + j];
        dnb = face[(en * 4 + (side ^ 1)) * n1 + j];
        tnb = x[en * nq + far];
    };
    double dot = 0.0;
    int e = xcd_remap(blockIdx.x, gridDim.x);
    if (e < noe) load(e);
    __syncthreads();                                              // U and F are cleared
    for (; e < noe; e += gridDim.x) {
#pragma unroll
        for (int i = 0; i < MV; ++i) {
            const int k = opaque(tid) + i * NTH, row = (int)(((unsigned)k * rn1) >> 18);
            if (k < nq) U[row * LD + (k - row * n1)] = v[i];
        }
        __syncthreads();
        if (hasf) {
            // the weighted jump of the traces and the averaged normal
            // derivative with the penalty; a boundary side takes the one-sided
            // Dirichlet form
            const double sg = side & 1 ? -1.0 : 1.0, tn = U[near];
            const double jump = bnd ? sg * tn : 0.5 * (sg * (tn - (double)tnb));
            const double der = bnd ? sg * (double)dn : sg * (0.5 * ((double)dn + (double)dnb));
            const double wjump = wj * jump;
            const int f = side < 2 ? 0 : 4;
            F[f + (side & 1)][j] = wjump;
            F[f + 2 + (side & 1)][j] = wj * der + sg * ((bnd ? pn : 2 * pn) * wjump);
        }
        if (e + (int)gridDim.x < noe) load(e + gridDim.x);
        gd4 ax[NT], ay[NT];
#pragma unroll
        for (int c = 0; c < NT; ++c) ax[c] = ay[c] = gd4{0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < NK; ++k) {
            if (4 * k > N) break;                                 // uniform
            const double ua = U[(16 * ti + li) * LD + 4 * k + lk];
#pragma unroll
            for (int c = 0; c < NT; ++c) {
                ax[c] = gmul(K[k][0], U[(4 * k + lk) * LD + col[c]], ax[c]);
                ay[c] = gmul(ua, K[k][c], ay[c]);
            }

        }
        __syncthreads();                                          // the faces are complete
        // k = 0, 1: along x (factors D0 or DN of i1), k = 2, 3: along y; then
        // the corrections, on the boundary lines alone
        const double a1 = own ? dE[0] : F[4 + o][col[0]];
        T *ye = y + (int64_t)e * nq;
#pragma unroll
        for (int c = 0; c < NT; ++c) {
            gd4 s = gmul(a1, own ? F[o][col[c]] : dE[c], gd4{0, 0, 0, 0});
            const int tj = ti + c < NT ? ti + c : ti + c - NT;
#pragma unroll
            for (int r = 0; r < 4; ++r) s[r] += wc[c] * ax[c][r] + wr[r] * ay[c][r];
            if (ti == 0 || ti == tN) {                            // this wave's tiles have row 0 or N
                const double v = F[ti == 0 ? 2 : 3][col[c]];
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (r == rS && lk == lkS) s[r] += v;
            }
            if (tj == 0 || tj == tN) {                            // column 0 or N
                if (li == (tj == 0 ? 0 : N & 15)) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[r] += F[tj == 0 ? 6 : 7][16 * ti + 4 * r + lk];
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * ti + 4 * r + lk;
                if (row <= N && col[c] <= N) {
                    const T out = (T)s[r];
                    ye[row * n1 + col[c]] = out;
                    if (DOT) dot += U[row * LD + col[c]] * (double)out;
                }
            }
        }
        __syncthreads();                                          // U and F are free
    }
    if (DOT) {
        const double s = block_sum<NTH>(dot, red);
        if (threadIdx.x == 0) partials[blockIdx.x] = s;
    }
}

// Workgroups of a kernel that the device holds at once, cached per device.
template <typename T, int NT>                                     // NT = 0: face_derivs_kernel
int resident_groups() {
    constexpr int kMaxDev = 64;
    static std::atomic<int> cache[kMaxDev];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDev) dev = 0;
    int g = cache[dev].load(std::memory_order_relaxed);
    if (g > 0) return g;
    const void *f;
    if constexpr (NT > 0) f = reinterpret_cast<const void *>(&apply_generic_kernel<T, NT, true>);
    else f = reinterpret_cast<const void *>(&face_derivs_kernel<T>);
    int cus = 0, per = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 0;
    // (the LDS that face_derivs_kernel is launched with: that of the lowest degree)
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, f, NT > 0 ? 64 * NT : kGenThreads,
                                                     NT > 0 ? 0 : 18 * 19 * sizeof(T)) != hipSuccess)
        per = 0;
    g = (cus > 0 ? cus : 1) * (per > 0 ? per : 1);
    cache[dev].store(g, std::memory_order_relaxed);
    return g;
}

// f(std::integral_constant<int, NT>) for the tiles of n1 nodes
template <class Fn>
auto by_tiles(int n1, Fn f) {
    if (n1 <= 32) return f(std::integral_constant<int, 2>{});
    if (n1 <= 48) return f(std::integral_constant<int, 3>{});
    return f(std::integral_constant<int, 4>{});
}

// A workgroup per element, as many as the device holds, within the partial
// buffer: each takes an equal share of the elements, where 2048 whatever the
// kernel left the last ones running alone.
template <typename T>
int grid_of(int p, int64_t noe) {
    return by_tiles(p + 1, [&](auto tiles) {
        return (int)std::min<int64_t>(noe, std::min(resident_groups<T, decltype(tiles)::value>(), kMaxPartials));
    });
}

template <typename T>
int launch_t(int p, const void *x, void *y, const void *tab, int dimx, int dimy, double pen, double *partials,
             const cg_state *st, int slot, hipStream_t s)
{
    const int n1 = p + 1;
    const int64_t noe = (int64_t)dimx * dimy;
    const T *tb = (const T *)tab;
    // the face buffer follows the tables in the op's table allocation
    T *face = const_cast<T *>(tb) + generic_face_offset(p, sizeof(T));
    const dim3 grid(grid_of<T>(p, noe)), gface((int)std::min<int64_t>(noe, resident_groups<T, 0>()));
    hipLaunchKernelGGL(face_derivs_kernel<T>, gface, dim3(kGenThreads), (size_t)n1 * (n1 | 1) * sizeof(T), s, n1,
                       (const T *)x, tb, face, (int)noe, partials ? st : nullptr, slot);
    by_tiles(n1, [&](auto tiles) {
        constexpr int NT = decltype(tiles)::value;
        if (partials)
            hipLaunchKernelGGL((apply_generic_kernel<T, NT, true>), grid, dim3(64 * NT), 0, s, n1, (const T *)x, (T *)y,
                               tb, (const T *)face, dimx, dimy, (T)pen, partials, st, slot);
        else
            hipLaunchKernelGGL((apply_generic_kernel<T, NT, false>), grid, dim3(64 * NT), 0, s, n1, (const T *)x,
                               (T *)y, tb, (const T *)face, dimx, dimy, (T)pen, partials, st, slot);
    });
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

}  // namespace

size_t generic_face_offset(int p, size_t elem) { return ((size_t)table_len(p) * elem + 255) / 256 * 256 / elem; }

size_t generic_table_len(int dtype, int p, int dimx, int dimy) {
    const size_t elem = dtype == SIPG_F64 ? 8 : 4;
    return generic_face_offset(p, elem) + (size_t)4 * (p + 1) * dimx * dimy;
}

int generic_apply_num_blocks(int dtype, int p, int dimx, int dimy) {
    const int64_t noe = (int64_t)dimx * dimy;
    return dtype == SIPG_F64 ? grid_of<double>(p, noe) : grid_of<float>(p, noe);
}

int launch_apply_generic(int dtype, int p, const void *x, void *y, const void *tab, int dimx, int dimy, double pen,
                         double *partials, const cg_state *st, int slot, hipStream_t s)
{
    if (p <= kMaxDegree || p > kMaxGenericDegree) return SIPG_ERR_UNSUPPORTED;
    return dtype == SIPG_F64 ? launch_t<double>(p, x, y, tab, dimx, dimy, pen, partials, st, slot, s)
                             : launch_t<float>(p, x, y, tab, dimx, dimy, pen, partials, st, slot, s);
}

}  // namespace sipg_internal
