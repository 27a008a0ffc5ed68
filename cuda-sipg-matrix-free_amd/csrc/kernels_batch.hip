// kernels_batch.hip -- many independent SIPG solves in the same launches.
//
// All instances share a launch of the operator kernel: the workgroups walk
// device-resident lists, one to a degree, of (instance, strip, rows) items,
// so the lists can shrink as instances finish without relaunching anything
// (the CG iterations are replayed from a captured hipGraph).  Vector updates walk a
// list of (instance, range) chunks.  Each instance has its own cg_state;
// its scalars are reduced per instance in a fixed order (deterministic, and
// independent of how the work is split).  All vectors of all instances are
// concatenated, element-major within each instance.
#include "batch_items.hpp"
#include "strip_apply.hpp"

#include <algorithm>
#include <array>
#include <atomic>

namespace sipg_internal {

namespace {

constexpr int NT = kVecThreads;

// LDS of a strip, and the most that degrees 1..p need, in doubles
template <int P>
constexpr int strip_lds = StripGeo<double, P>::LDS + StripGeo<double, P>::EXCH;
template <int... Ps>
constexpr std::array<int, sizeof...(Ps)> strip_lds_table(std::integer_sequence<int, Ps...>) {
    return {strip_lds<Ps + 1>...};
}
int strip_lds_upto(int p) {
    static constexpr auto need = strip_lds_table(std::make_integer_sequence<int, kMaxDegree>{});
    return *std::max_element(need.begin(), need.begin() + p);
}

// y = A x for the items of all groups (degrees), each a strip of whole
// elements by a band of rows (strip_apply.hpp); with DOT also the item's
// share of x.y into item_part, and items of instances already finished (per
// states[inst].s[slot].done) are skipped.  Persistent workgroups take every
// gridDim-th item, so that each gets a mix of degrees.
//
// One launch for all degrees: with a launch to each, a batch of 128
// instances of nine degrees took 87 us an iteration on average, one launch
// 34: the late iterations, with few instances left, were mostly launches.  The
// registers are those of the highest degree of the class PMAX, the LDS that
// of the highest degree present.
template <int PMAX, bool DOT>
__global__ __launch_bounds__(256, PMAX <= 8 ? 3 : PMAX <= 12 ? 2 : 1)
void batch_apply_kernel(batch_groups G, const double *__restrict__ X, double *__restrict__ Y,
                        const batch_inst *__restrict__ inst, double *__restrict__ item_part,
                        const cg_state *__restrict__ states, int slot)
{
    extern __shared__ __attribute__((aligned(16))) double lds[];
    __shared__ double red[4];
    __shared__ int first[kMaxDegree + 1];
    const int n = batch_offsets(G, first);
    for (int k = xcd_remap(blockIdx.x, gridDim.x); k < n; k += gridDim.x) {
        int i;
        const int g = batch_group_at(G, first, k, i);
        const batch_item it = G.g[g].items[i];
        if (DOT) {
            const cg_state *st = states + it.inst;
            if (st->s[slot].done | st->err) continue;             // uniform over the workgroup
        }
        const batch_inst in = inst[it.inst];
        const int tid = opaque(threadIdx.x);
        const double d = by_degree<PMAX>(G.g[g].p, [&](auto deg) {
            constexpr int P = decltype(deg)::value, EPW = StripGeo<double, P>::EPW;
            return strip_apply<double, P, DOT>(X + in.off, Y + in.off, in.dimx, in.dimy, in.pen, it.x0,
                                               min(EPW, in.dimx - it.x0), it.y0, min(it.y0 + it.rows, in.dimy), lds,
                                               lds + StripGeo<double, P>::LDS, tid);
        });
        if (DOT) {
            const double bs = block_sum<256>(d, red);
            if (threadIdx.x == 0) item_part[G.g[g].base + i] = bs;
        } else {
            // the next item's degree may place its waves' tiles where a wave
            // still works on this one (with DOT the sum's barrier is between)
            __syncthreads();
        }
    }
}

__device__ __forceinline__ double block_reduce(double v, double *red) {
    // fixed-order block sum, valid in every thread
    v = wave_total(v);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[wid] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) s += red[i];
    return s;
}

// sum of part[b, e) in a fixed order (strided per thread, then the block)
__device__ __forceinline__ double range_sum(const double *__restrict__ part, int b, int e, double *red) {
    double s = 0.0;
    for (int i = b + (int)threadIdx.x; i < e; i += NT) s += part[i];
    return block_reduce(s, red);
}

// alpha = r.z / p.Ap per active instance (r.z = r.r for plain CG; the host-side alpha of
// conjugate_gradient_gpu.hpp:75-83); breakdown and non-finite values end
// that instance only.
__global__ __launch_bounds__(NT) void batch_alpha_kernel(const int *__restrict__ list, const int *__restrict__ count,
                                                         const int2 *__restrict__ item_range,
                                                         const double *__restrict__ item_part,
                                                         cg_state *states, int slot) {
    __shared__ double red[NT / 64];
    const int n = *count;
    for (int k = blockIdx.x; k < n; k += gridDim.x) {
        const int i = list[k];
        cg_state *st = states + i;
        if (st->s[slot].done | st->err) continue;                 // uniform per block
        const int2 r = item_range[i];
        const double pAp = range_sum(item_part, r.x, r.y, red);
        if (threadIdx.x == 0) {
            const double alpha = st->s[slot].rz / pAp;
            if (!(pAp > 0.0) || !isfinite(alpha)) {
                st->err = isfinite(pAp) ? 2 : 3;
            } else {
                st->s[slot].alpha = alpha;
                st->s[slot].pAp = pAp;
            }
        }
    }
}

// x += alpha p, r -= alpha Ap over the listed chunks; chunk sums of r.r
template <typename T>
__global__ __launch_bounds__(NT) void batch_update_xr_kernel(T *__restrict__ X, const T *__restrict__ Pv,
                                                             T *__restrict__ Rv, const T *__restrict__ APv,
                                                             const batch_chunk *__restrict__ chunks,
                                                             const int *__restrict__ count,
                                                             double *__restrict__ chunk_part,
                                                             const cg_state *__restrict__ states, int slot) {
    __shared__ double red[NT / 64];
    const int n = *count;
    for (int k = blockIdx.x; k < n; k += gridDim.x) {
        const batch_chunk c = chunks[k];
        const cg_state *st = states + c.inst;
        if (st->s[slot].done | st->err) continue;
        const T alpha = (T)st->s[slot].alpha;
        double s = 0.0;
        for (int64_t i = c.begin + threadIdx.x; i < c.end; i += NT) {
            X[i] = X[i] + alpha * Pv[i];
            const T ri = Rv[i] - alpha * APv[i];
            Rv[i] = ri;
            s += (double)ri * (double)ri;
        }
        s = block_reduce(s, red);
        if (threadIdx.x == 0) chunk_part[k] = s;
    }
}

// beta = r.r(new) / r.r(old) per active instance; writes the next slot
// (conjugate_gradient_gpu.hpp:85-95 and the while-condition of :69).  An
// instance whose r was replaced by b - A x in this iteration (kSlotReplaced,
// set by batch_mark_kernel) takes r.r(new) from the replacement's chunk
// sums and keeps its direction (reliable update); with st->true_stop it
// finishes only on such a true residual, and a recursion that meets the
// tolerance raises kSlotWantCheck for the host to schedule one.
__global__ __launch_bounds__(NT) void batch_beta_kernel(const int *__restrict__ list, const int *__restrict__ count,
                                                        const int2 *__restrict__ chunk_range,
                                                        const double *__restrict__ chunk_part,
                                                        const int2 *__restrict__ repl_range,
                                                        const double *__restrict__ repl_part,
                                                        cg_state *states, int slot) {
    __shared__ double red[NT / 64];
    const int n = *count;
    for (int k = blockIdx.x; k < n; k += gridDim.x) {
        const int i = list[k];
        cg_state *st = states + i;
        const cg_slot cur = st->s[slot];
        if (cur.done | st->err) {
            if (threadIdx.x == 0) st->s[slot ^ 1] = cur;           // carry forward
            continue;
        }
        const bool replaced = (cur.flags & kSlotReplaced) != 0;
        const int2 r = replaced ? repl_range[i] : chunk_range[i];
        const double rr_new = range_sum(replaced ? repl_part : chunk_part, r.x, r.y, red);
        if (threadIdx.x == 0) {
            const bool met = !(sqrt(rr_new) > st->stop);
            const bool need_true = st->true_stop && !replaced;
            cg_slot nx{};
            nx.rr = rr_new;
            nx.rz = rr_new;
            nx.alpha = 0.0;
            nx.beta = rr_new / cur.rr;
            nx.pAp = 0.0;
            nx.it = cur.it + 1;
            nx.done = ((met && !need_true) || nx.it >= st->maxit) ? 1 : 0;
            nx.checked = replaced ? 1 : 0;
            nx.flags = (met && need_true) ? kSlotWantCheck : 0;
            st->s[slot ^ 1] = nx;
            if (replaced) st->rr_ref = rr_new;
            if (!isfinite(rr_new)) st->err = 3;
        }
    }
}

// marks the listed instances' slot as replaced (r is b - A x now and the
// replacement chunk sums hold its r.r); a no-op for finished instances
__global__ __launch_bounds__(NT) void batch_mark_kernel(const int *__restrict__ list, const int *__restrict__ count,
                                                        cg_state *states, int slot) {
    const int n = *count;
    for (int k = blockIdx.x * NT + threadIdx.x; k < n; k += gridDim.x * NT) {
        cg_state *st = states + list[k];
        cg_slot c = st->s[slot];
        if (c.done | st->err) continue;
        c.flags |= kSlotReplaced;
        st->s[slot] = c;
        st->nrep += 1;
    }
}

// x += z; z = 0 over the listed chunks: the group update (van der Vorst &
// Ye 2000) folds the increments accumulated since the last true residual
template <typename T>
__global__ __launch_bounds__(NT) void batch_fold_kernel(T *__restrict__ X, T *__restrict__ Z,
                                                        const batch_chunk *__restrict__ chunks,
                                                        const int *__restrict__ count) {
    const int n = *count;
    for (int k = blockIdx.x; k < n; k += gridDim.x) {
        const batch_chunk c = chunks[k];
        for (int64_t i = c.begin + threadIdx.x; i < c.end; i += NT) {
            X[i] += Z[i];
            Z[i] = T(0);
        }
    }
}

// p = r + beta p over the listed chunks of instances still iterating
template <typename T>
__global__ __launch_bounds__(NT) void batch_update_p_kernel(const T *__restrict__ Rv, T *__restrict__ Pv,
                                                            const batch_chunk *__restrict__ chunks,
                                                            const int *__restrict__ count,
                                                            const cg_state *__restrict__ states, int slot) {
    const int n = *count;
    for (int k = blockIdx.x; k < n; k += gridDim.x) {
        const batch_chunk c = chunks[k];
        const cg_state *st = states + c.inst;
        if (st->s[slot].done | st->err) continue;
        const T beta = (T)st->s[slot ^ 1].beta;
        for (int64_t i = c.begin + threadIdx.x; i < c.end; i += NT) Pv[i] = Rv[i] + beta * Pv[i];
    }
}

// r = b - Ax over the listed chunks (optionally p = r); chunk sums of r.r
// and b.b
template <typename T>
__global__ __launch_bounds__(NT) void batch_residual_kernel(const T *__restrict__ B, const T *__restrict__ AX,
                                                            T *__restrict__ Rv, T *__restrict__ Pv,
                                                            const batch_chunk *__restrict__ chunks,
                                                            const int *__restrict__ count,
                                                            double *__restrict__ part_rr,
                                                            double *__restrict__ part_bb) {
    __shared__ double red[NT / 64];
    const int n = *count;
    for (int k = blockIdx.x; k < n; k += gridDim.x) {
        const batch_chunk c = chunks[k];
        double srr = 0.0, sbb = 0.0;
        for (int64_t i = c.begin + threadIdx.x; i < c.end; i += NT) {
            const T bi = B[i];
            const T ri = bi - AX[i];
            Rv[i] = ri;
            if (Pv) Pv[i] = ri;
            srr += (double)ri * (double)ri;
            sbb += (double)bi * (double)bi;
        }
        srr = block_reduce(srr, red);
        sbb = block_reduce(sbb, red);
        if (threadIdx.x == 0) {
            part_rr[k] = srr;
            part_bb[k] = sbb;
        }
    }
}

// initial state of each listed instance from its r.r and b.b chunk sums
// (and, for PCG, its r.z item sums; otherwise r.z = r.r)
__global__ __launch_bounds__(NT) void batch_init_kernel(const int *__restrict__ list, const int *__restrict__ count,
                                                        const int2 *__restrict__ chunk_range,
                                                        const double *__restrict__ part_rr,
                                                        const double *__restrict__ part_bb, cg_state *states,
                                                        const batch_ctl *__restrict__ ctl,
                                                        const int2 *__restrict__ item_range,
                                                        const double *__restrict__ item_rz) {
    __shared__ double red[NT / 64];
    const int n = *count;
    for (int k = blockIdx.x; k < n; k += gridDim.x) {
        const int i = list[k];
        const int2 r = chunk_range[i];
        const double rr = range_sum(part_rr, r.x, r.y, red);
        const double bb = range_sum(part_bb, r.x, r.y, red);
        double rz = rr;
        if (item_rz) {
            const int2 q = item_range[i];
            rz = range_sum(item_rz, q.x, q.y, red);
        }
        if (threadIdx.x == 0) {
            cg_state *st = states + i;
            const batch_ctl c = ctl[i];
            const double stop = c.tol_mode == SIPG_TOL_REL ? c.tol * sqrt(bb) : c.tol;
            cg_slot s0{};
            s0.rr = rr;
            s0.rz = rz;
            s0.alpha = s0.beta = s0.pAp = 0.0;
            s0.it = 0;
            s0.done = (sqrt(rr) > stop && c.maxit > 0) ? 0 : 1;
            s0.checked = 1;
            s0.flags = 0;
            st->s[0] = s0;
            st->s[1] = s0;
            st->bb = bb;
            st->stop = stop;
            st->stop_true = stop;
            st->rr0 = rr;
            st->rr_ref = rr;
            st->maxit = c.maxit;
            st->nrep = 0;
            st->err = (!isfinite(rr) || !isfinite(bb) || !isfinite(rz)) ? 3 : 0;
            st->true_stop = 1;
        }
    }
}

// Workgroups of the apply kernel that the device holds at once with the LDS
// of degree pmax, cached per device.
template <int PMAX, bool DOT>
int resident_batch_groups(int pmax, size_t lds) {
    static std::atomic<int> cache[64][kMaxDegree + 1];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
    int g = cache[dev][pmax].load(std::memory_order_relaxed);
    if (g > 0) return g;
    int cus = 0, per = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per, reinterpret_cast<const void *>(&batch_apply_kernel<PMAX, DOT>), 256, lds) != hipSuccess)
        per = 0;
    g = (cus > 0 ? cus : 1) * (per > 0 ? per : 1);
    cache[dev][pmax].store(g, std::memory_order_relaxed);
    return g;
}

template <int PMAX>
int launch_apply_class(const batch_groups &G, int pmax, int max_items, const double *X, double *Y,
                       const batch_inst *inst, double *item_part, const cg_state *states, int slot, hipStream_t s) {
    const size_t lds = (size_t)strip_lds_upto(pmax) * sizeof(double);
    if (item_part) {
        const dim3 grid(std::min(max_items, resident_batch_groups<PMAX, true>(pmax, lds)));
        hipLaunchKernelGGL((batch_apply_kernel<PMAX, true>), grid, dim3(256), lds, s, G, X, Y, inst, item_part, states,
                           slot);
    } else {
        const dim3 grid(std::min(max_items, resident_batch_groups<PMAX, false>(pmax, lds)));
        hipLaunchKernelGGL((batch_apply_kernel<PMAX, false>), grid, dim3(256), lds, s, G, X, Y, inst, item_part,
                           states, slot);
    }
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

int vec_blocks(int nchunks) { return std::max(1, std::min(nchunks, 2048)); }
int inst_blocks(int ninst) { return std::max(1, std::min(ninst, 2048)); }

}  // namespace

const int kBatchShapeBX[kBatchShapes] = {16, 8, 8};
const int kBatchShapeBY[kBatchShapes] = {4, 4, 2};

bool batch_shape_supported(int p, int shape) {
    // 16 x 4 stays a choice up to degree 12
    return p >= 1 && p <= kMaxDegree && shape >= 0 && shape < kBatchShapes && (shape > 0 || p <= 12);
}

// An item is a strip of 64 / (p+1) elements by 16, 8 or 4 rows: one to four
// rows to a wave.  Fewer rows make more items, which a small batch and the
// last instances of a large one need; more rows load the rows between two
// bands less often.
void batch_item_extent(int p, int shape, int *bx, int *rows) {
    *bx = 64 / (p + 1);
    *rows = shape == 0 ? 16 : shape == 1 ? 8 : 4;
}

int launch_batch_apply_groups(const batch_groups &G, int max_items, const double *X, double *Y,
                              const batch_inst *inst, double *item_part, const cg_state *states, int slot,
                              hipStream_t s) {
    int pmax = 0;
    for (int g = 0; g < G.n; ++g) {
        if (G.g[g].p < 1 || G.g[g].p > kMaxDegree) return SIPG_ERR_UNSUPPORTED;
        pmax = std::max(pmax, G.g[g].p);
    }
    if (item_part && !states) return SIPG_ERR_INVALID;
    if (max_items <= 0 || pmax == 0) return SIPG_OK;
    // Classes by the registers their highest degree needs: 168 up to degree
    // 8 (three workgroups to a CU, as their LDS allows), 252 up to 12 (two)
    if (pmax <= 8) return launch_apply_class<8>(G, pmax, max_items, X, Y, inst, item_part, states, slot, s);
    if (pmax <= 12) return launch_apply_class<12>(G, pmax, max_items, X, Y, inst, item_part, states, slot, s);
    return launch_apply_class<16>(G, pmax, max_items, X, Y, inst, item_part, states, slot, s);
}

int launch_batch_apply(int p, int shape, const double *X, double *Y, const batch_inst *inst,
                       const batch_item *items, const int *count, int max_items, double *item_part,
                       const cg_state *states, int slot, hipStream_t s) {
    if (!batch_shape_supported(p, shape)) return SIPG_ERR_UNSUPPORTED;
    batch_groups G;
    G.n = 1;
    G.g[0] = {items, count, 0, p};
    return launch_batch_apply_groups(G, max_items, X, Y, inst, item_part, states, slot, s);
}

int launch_batch_alpha(const int *list, const int *count, int max_inst, const int2 *item_range,
                       const double *item_part, cg_state *states, int slot, hipStream_t s) {
    hipLaunchKernelGGL(batch_alpha_kernel, dim3(inst_blocks(max_inst)), dim3(NT), 0, s, list, count, item_range,
                       item_part, states, slot);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

int launch_batch_update_xr(double *X, const double *Pv, double *Rv, const double *APv, const batch_chunk *chunks,
                           const int *count, int max_chunks, double *chunk_part, const cg_state *states, int slot,
                           hipStream_t s) {
    hipLaunchKernelGGL(batch_update_xr_kernel<double>, dim3(vec_blocks(max_chunks)), dim3(NT), 0, s, X, Pv, Rv,
                       APv, chunks, count, chunk_part, states, slot);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

int launch_batch_beta(const int *list, const int *count, int max_inst, const int2 *chunk_range,
                      const double *chunk_part, const int2 *repl_range, const double *repl_part,
                      cg_state *states, int slot, hipStream_t s) {
    hipLaunchKernelGGL(batch_beta_kernel, dim3(inst_blocks(max_inst)), dim3(NT), 0, s, list, count, chunk_range,
                       chunk_part, repl_range, repl_part, states, slot);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

int launch_batch_update_p(const double *Rv, double *Pv, const batch_chunk *chunks, const int *count,
                          int max_chunks, const cg_state *states, int slot, hipStream_t s) {
    hipLaunchKernelGGL(batch_update_p_kernel<double>, dim3(vec_blocks(max_chunks)), dim3(NT), 0, s, Rv, Pv, chunks,
                       count, states, slot);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

int launch_batch_residual(const double *B, const double *AX, double *Rv, double *Pv, const batch_chunk *chunks,
                          const int *count, int max_chunks, double *part_rr, double *part_bb, hipStream_t s) {
    hipLaunchKernelGGL(batch_residual_kernel<double>, dim3(vec_blocks(max_chunks)), dim3(NT), 0, s, B, AX, Rv, Pv,
                       chunks, count, part_rr, part_bb);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

int launch_batch_init(const int *list, const int *count, int max_inst, const int2 *chunk_range,
                      const double *part_rr, const double *part_bb, cg_state *states, const batch_ctl *ctl,
                      const int2 *item_range, const double *item_rz, hipStream_t s) {
    hipLaunchKernelGGL(batch_init_kernel, dim3(inst_blocks(max_inst)), dim3(NT), 0, s, list, count, chunk_range,
                       part_rr, part_bb, states, ctl, item_range, item_rz);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

int launch_batch_fold(double *X, double *Z, const batch_chunk *chunks, const int *count, int max_chunks,
                      hipStream_t s) {
    hipLaunchKernelGGL(batch_fold_kernel<double>, dim3(vec_blocks(max_chunks)), dim3(NT), 0, s, X, Z, chunks, count);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

int launch_batch_mark(const int *list, const int *count, int max_inst, cg_state *states, int slot,
                      hipStream_t s) {
    hipLaunchKernelGGL(batch_mark_kernel, dim3(std::max(1, std::min((max_inst + NT - 1) / NT, 64))), dim3(NT), 0,
                       s, list, count, states, slot);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

}  // namespace sipg_internal
