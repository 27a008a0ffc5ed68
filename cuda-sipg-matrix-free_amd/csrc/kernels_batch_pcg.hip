// kernels_batch_pcg.hip -- block-Jacobi PCG for batched solves: z = M^-1 r
// over the (instance, block) items of the operator's lists, and the rest of
// an iteration fused around it.  M is the exact inverse of the interior
// element block of the standard penalty 5 (p+1)^2 (kernels_pcg.hip), so every
// coefficient is a compile-time constant of the degree; batched PCG requires
// that penalty.
//
// An iteration is three launches over all degrees: the operator with p.Ap
// (kernels_batch.hip); alpha, r -= alpha Ap and z = M^-1 r; beta, x += alpha
// p and p = z + beta p.  Each workgroup sums the p.Ap or r.r and r.z shares
// of its instance by itself, in a fixed order; where a large instance is in
// the lists, a launch after the operator's and one after the second add up
// its shares (batch_totals_kernel).  Where some instances' r is replaced by
// b - A x, a fold of their x and the operator on them come before the second,
// and that takes b - A x for its r.
//
// Within a launch, an instance's state is written by the workgroup of its
// first item or chunk only, in fields that the others do not read: the
// next slot, err (read by the launches that do not write it), alpha and the
// mark that the instance has been stepped.
#include "apply_block.hpp"
#include "batch_items.hpp"
#include "prec_block.hpp"

#include <algorithm>
#include <array>
#include <atomic>

namespace sipg_internal {

namespace {

constexpr int VT = kVecThreads;

// 1 / (lambda_a + lambda_c) of degree p starts at linv_at(p) in LDS
__host__ __device__ constexpr int linv_at(int p) { return p * (p + 1) * (2 * p + 1) / 6 - 1; }
static_assert(linv_at(2) - linv_at(1) == 4 && linv_at(1) == 0, "(q+1)^2 values for each degree q < p");

// LDS of the degrees up to p, in doubles: the four waves' tiles, the tables
template <int... Ps>
constexpr std::array<int, sizeof...(Ps)> prec_lds_table(std::integer_sequence<int, Ps...>) {
    return {4 * RunGeo<double, Ps + 1>::BUF...};
}
int prec_tiles_upto(int p) {
    static constexpr auto need = prec_lds_table(std::make_integer_sequence<int, kMaxDegree>{});
    return *std::max_element(need.begin(), need.begin() + p);
}

// the instance's sum, in every lane of the wave, in a fixed order
__device__ __forceinline__ double instance_sum(item_sum q, const int2 *__restrict__ item_range, int inst, int lane) {
    const int2 r = item_range[inst];
    if (r.y - r.x > kDirectItems) return q.total[inst];
    double s = 0.0;
    for (int i = r.x + lane; i < r.y; i += 64) s += q.part[i];
    return wave_total(s);
}

// The sums of the listed instances that have more than kDirectItems items,
// one workgroup to each.
//
// Without it every item and every chunk of such an instance adds up all its
// items, three times an iteration, which grows with the square of its size:
// us an iteration so, and now: one instance of 512 x 512 elements, p = 8 622,
// 458; 2048 x 2048, p = 2 3755, 825; 3000 x 3000, p = 1 4480, 811.  kDirectItems:
// with fewer items the two launches cost as much as they save (384 items, 192 x
// 192, p = 4: 35.9 directly, 36.6 with them; 672, 192 x 192, p = 8: 71.8, 70.0).
template <int K>
__global__ __launch_bounds__(VT) void batch_totals_kernel(const int *__restrict__ list, const int *__restrict__ count,
                                                          const int2 *__restrict__ item_range, item_sum a,
                                                          item_sum b) {
    const int n = *count;
    for (int k = blockIdx.x; k < n; k += gridDim.x) {
        const int inst = list[k];
        const int2 r = item_range[inst];
        const int m = r.y - r.x;
        if (m <= kDirectItems) continue;                          // uniform over the workgroup
        double out[K];
        if constexpr (K == 1) multi_sum<VT, 1>({a.part + r.x}, {m}, out);
        else multi_sum<VT, 2>({a.part + r.x, b.part + r.x}, {m, m}, out);
        if (threadIdx.x == 0) {
            a.total[inst] = out[0];
            if constexpr (K == 2) b.total[inst] = out[K - 1];
        }
        __syncthreads();                                          // the next instance's sums take the same LDS
    }
}

// z = M^-1 r for the items of all groups, and p = z at the start of a solve;
// an item's sums of r.r and r.z go to item_rr and item_rz.  STEP (inside an
// iteration): first alpha = r.z / p.Ap and r -= alpha Ap, or r = b - Ap for an
// instance marked replaced (Ap holds A x then); items of instances already
// finished at `slot` are skipped.  A breakdown (p.Ap not positive, or not
// finite) skips the instance; the update that follows sets its err.
//
// A wave streams the runs of its item's rows on its own (prec_block.hpp).
// With STEP four passes over memory, where the update of x and r and the
// preconditioner took eight in two sets of launches: 46 + 74 us an iteration
// on average over a solve of 128 instances of nine degrees, 44 now.
template <int PMAX, bool STEP>
__global__ __launch_bounds__(256, PMAX <= 12 ? 3 : 2)
void batch_prec_kernel(batch_groups G, int tiles, double *R, const double *__restrict__ AP,
                       const double *__restrict__ B, double *__restrict__ Zq, double *__restrict__ Pv,
                       const batch_inst *__restrict__ inst, const int2 *__restrict__ item_range,
                       item_sum part, double *__restrict__ item_rr, double *__restrict__ item_rz, cg_state *states,
                       int slot)
{
    extern __shared__ __attribute__((aligned(16))) double lds[];
    __shared__ double red[2][4];
    __shared__ int first[kMaxDegree + 1];
    const int n = batch_offsets(G, first);
    double *tab = lds + tiles;
    for (int g = 0; g < G.n; ++g)
        by_degree<PMAX>(G.g[g].p, [&](auto deg) {
            constexpr int P = decltype(deg)::value, N1 = P + 1;
            for (int q = threadIdx.x; q < N1 * N1; q += 256) tab[linv_at(P) + q] = PrecEO<P>::V.Linv[q / N1][q % N1];
        });
    __syncthreads();
    for (int k = xcd_remap(blockIdx.x, gridDim.x); k < n; k += gridDim.x) {
        int i;
        const int g = batch_group_at(G, first, k, i);
        const batch_item it = G.g[g].items[i];
        cg_state *st = states + it.inst;
        if (STEP && (st->s[slot].done | st->err)) continue;     // uniform over the workgroup
        const batch_inst in = inst[it.inst];
        const int at = G.g[g].base + i;
        const int tid = opaque(threadIdx.x);
        const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
        const bool replaced = STEP && (st->s[slot].flags & kSlotReplaced);
        double alpha = 0.0;
        if (STEP) {
            const double pAp = instance_sum(part, item_range, it.inst, lane);
            alpha = st->s[slot].rz / pAp;
            if (at == item_range[it.inst].x && tid == 0) {
                st->s[slot].alpha = alpha;
                st->s[slot].pAp = pAp;
                st->s[slot].flags |= kSlotStepped;
            }
            if (!(pAp > 0.0) || !isfinite(alpha)) continue;       // the same in every workgroup
            if (replaced) alpha = 1.0;
        }
        double srr = 0.0, srz = 0.0;
        by_degree<PMAX>(G.g[g].p, [&](auto deg) {
            constexpr int P = decltype(deg)::value;
            using Run = RunGeo<double, P>;
            const int nv = min(Run::EPW, in.dimx - it.x0) * Run::NQ;
            const int yb = min(it.y0 + it.rows, in.dimy);
            double x0, x1;
            for (int gy = it.y0 + w; gy < yb; gy += 4) {
                const int64_t o = in.off + ((int64_t)gy * in.dimx + it.x0) * Run::NQ;
                prec_run<double, P, STEP, !STEP, true, false>((replaced ? B : R) + o, R + o, AP + o, Zq + o, Pv + o, nv,
                                                              [&] { return alpha; }, nullptr, tab + linv_at(P),
                                                              lds + w * Run::BUF, lane, srr, srz, x0, x1);
            }
        });
        srr = wave_total(srr);
        srz = wave_total(srz);
        __syncthreads();                                          // the last item's sums have been read
        if (lane == 0) {
            red[0][w] = srr;
            red[1][w] = srz;
        }
        __syncthreads();
        if (tid < 2) {
            const double *v = red[tid];
            (tid ? item_rz : item_rr)[at] = (v[0] + v[1]) + (v[2] + v[3]);
        }
    }
}

template <int PMAX, bool STEP>
int resident_prec_groups(int pmax, size_t lds) {
    static std::atomic<int> cache[64][kMaxDegree + 1];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
    int g = cache[dev][pmax].load(std::memory_order_relaxed);
    if (g > 0) return g;
    int cus = 0, per = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per, reinterpret_cast<const void *>(&batch_prec_kernel<PMAX, STEP>), 256, lds) != hipSuccess)
        per = 0;
    g = (cus > 0 ? cus : 1) * (per > 0 ? per : 1);
    cache[dev][pmax].store(g, std::memory_order_relaxed);
    return g;
}

template <int PMAX, bool STEP>
int launch_prec_kernel(const batch_groups &G, int pmax, int max_items, double *R, const double *AP, const double *B,
                       double *Zq, double *Pv, const batch_inst *inst, const int2 *item_range,
                       item_sum part, double *item_rr, double *item_rz, cg_state *states, int slot, hipStream_t s) {
    const int tiles = prec_tiles_upto(pmax);
    const size_t lds = (size_t)(tiles + linv_at(pmax + 1)) * sizeof(double);
    const dim3 grid(std::min(max_items, resident_prec_groups<PMAX, STEP>(pmax, lds)));
    hipLaunchKernelGGL((batch_prec_kernel<PMAX, STEP>), grid, dim3(256), lds, s, G, tiles, R, AP, B, Zq, Pv,
                       inst, item_range, part, item_rr, item_rz, states, slot);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

template <bool STEP, class... A>
int launch_prec_any(const batch_groups &G, int max_items, A... args) {
    int pmax = 0;
    for (int g = 0; g < G.n; ++g) {
        if (G.g[g].p < 1 || G.g[g].p > kMaxDegree) return SIPG_ERR_UNSUPPORTED;
        pmax = std::max(pmax, G.g[g].p);
    }
    if (max_items <= 0 || pmax == 0) return SIPG_OK;
    if (pmax <= 8) return launch_prec_kernel<8, STEP>(G, pmax, max_items, args...);
    if (pmax <= 12) return launch_prec_kernel<12, STEP>(G, pmax, max_items, args...);
    return launch_prec_kernel<16, STEP>(G, pmax, max_items, args...);
}

// For the listed chunks of instances whose r is to be replaced: x += z +
// alpha p, z = 0 (the increments since the last true residual, this
// iteration's included, folded as one); marks the instance.
__global__ __launch_bounds__(VT) void batch_pcg_fold_kernel(double *__restrict__ X, double *__restrict__ Z,
                                                            const double *__restrict__ Pv,
                                                            const batch_chunk *__restrict__ chunks,
                                                            const int *__restrict__ count,
                                                            const int2 *__restrict__ chunk_range,
                                                            const int2 *__restrict__ item_range, item_sum part,
                                                            cg_state *states, int slot) {
    const int n = *count;
    for (int k = blockIdx.x; k < n; k += gridDim.x) {
        const batch_chunk c = chunks[k];
        cg_state *st = states + c.inst;
        if (st->s[slot].done | st->err) continue;
        const double pAp = instance_sum(part, item_range, c.inst, threadIdx.x & 63);
        const double alpha = st->s[slot].rz / pAp;
        if (!(pAp > 0.0) || !isfinite(alpha)) continue;
        if (k == chunk_range[c.inst].x && threadIdx.x == 0) {
            st->s[slot].flags |= kSlotReplaced;
            st->nrep += 1;
        }
        for (int64_t i = c.begin + threadIdx.x; i < c.end; i += VT) {
            const double z = Z[i] + alpha * Pv[i];
            X[i] += z;
            Z[i] = 0.0;
        }
    }
}

// beta = r.z(new) / r.z(old) per instance from the preconditioner's item
// sums; z += alpha p (unless r was replaced: it is folded then) and p = zq +
// beta p over the listed chunks; the first chunk's workgroup writes the next
// slot with r.r (stopping test, host decisions) and r.z.  Flag rules as in
// batch_beta_kernel.  An instance that was not stepped (finished, or err)
// carries its slot forward.
//
// Five passes over memory; 16 bytes to a lane, four of them in flight for
// each stream (37 us an iteration on average in the same solve).
__global__ __launch_bounds__(VT) void batch_pcg_update_kernel(double *__restrict__ Z, double *__restrict__ Pv,
                                                              const double *__restrict__ Zq,
                                                              const batch_chunk *__restrict__ chunks,
                                                              const int *__restrict__ count,
                                                              const int2 *__restrict__ chunk_range,
                                                              const int2 *__restrict__ item_range,
                                                              item_sum rr, item_sum rz, cg_state *states, int slot) {
    const int n = *count;
    for (int k = blockIdx.x; k < n; k += gridDim.x) {
        const batch_chunk c = chunks[k];
        cg_state *st = states + c.inst;
        const cg_slot cur = st->s[slot];
        const bool lead = k == chunk_range[c.inst].x && threadIdx.x == 0;
        const bool bad = !(cur.pAp > 0.0) || !isfinite(cur.alpha);
        if (cur.done || !(cur.flags & kSlotStepped) || bad) {
            if (lead) {
                if (!cur.done && (cur.flags & kSlotStepped)) st->err = isfinite(cur.pAp) ? 2 : 3;
                cg_slot nx = cur;
                nx.flags &= ~kSlotStepped;
                st->s[slot ^ 1] = nx;
            }
            continue;
        }
        const int lane = threadIdx.x & 63;
        const double rr_new = instance_sum(rr, item_range, c.inst, lane);
        const double rz_new = instance_sum(rz, item_range, c.inst, lane);
        const double alpha = cur.alpha, beta = rz_new / cur.rz;
        const bool replaced = (cur.flags & kSlotReplaced) != 0;
        if (lead) {
            const bool met = !(sqrt(rr_new) > st->stop);
            const bool need_true = st->true_stop && !replaced;
            cg_slot nx{};
            nx.rr = rr_new;
            nx.rz = rz_new;
            nx.beta = beta;
            nx.it = cur.it + 1;
            nx.done = ((met && !need_true) || nx.it >= st->maxit) ? 1 : 0;
            nx.checked = replaced ? 1 : 0;
            nx.flags = (met && need_true) ? kSlotWantCheck : 0;
            st->s[slot ^ 1] = nx;
            if (replaced) st->rr_ref = rr_new;
            if (!isfinite(rr_new) || !isfinite(rz_new)) st->err = 3;
            else if (!(rz_new > 0.0) && rr_new > 0.0) st->err = 2;
        }
        constexpr int U = 4;
        const int64_t len = c.end - c.begin, nvec = len / 2;
        double *z = Z + c.begin, *p = Pv + c.begin;
        const double *q = Zq + c.begin;
        auto one = [&](int64_t i) {
            const double pv = p[i];
            if (!replaced) z[i] = z[i] + alpha * pv;
            p[i] = q[i] + beta * pv;
        };
        int64_t v0 = 0;
        for (; v0 + U * VT <= nvec; v0 += U * VT) {
            double pv[U][2], qv[U][2], zv[U][2];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t o = 2 * (v0 + u * VT + threadIdx.x);
                load_vec<double, 2>(p + o, pv[u]);
                load_vec<double, 2>(q + o, qv[u]);
                if (!replaced) load_vec<double, 2>(z + o, zv[u]);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t o = 2 * (v0 + u * VT + threadIdx.x);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    if (!replaced) zv[u][h] = zv[u][h] + alpha * pv[u][h];
                    pv[u][h] = qv[u][h] + beta * pv[u][h];
                }
                if (!replaced) store_vec<double, 2>(z + o, zv[u]);
                store_vec<double, 2>(p + o, pv[u]);
            }
        }
        for (int64_t i = 2 * v0 + threadIdx.x; i < len; i += VT) one(i);
    }
}

}  // namespace

bool batch_prec_supported(int p, double pen, int shape) {
    return batch_shape_supported(p, shape) && pen == 5.0 * (p + 1) * (p + 1);
}

int launch_batch_prec_groups(const batch_groups &G, int max_items, const double *R, double *Zq, double *Pv,
                             const batch_inst *inst, double *item_rr, double *item_rz, hipStream_t s) {
    const double *none = nullptr;
    const int2 *nor = nullptr;
    cg_state *nos = nullptr;
    return launch_prec_any<false>(G, max_items, const_cast<double *>(R) /* read only without STEP */, none, none, Zq,
                                  Pv, inst, nor, item_sum{}, item_rr, item_rz, nos, 0, s);
}

int launch_batch_totals(const int *list, const int *count, int max_inst, const int2 *item_range, item_sum a,
                        item_sum b, hipStream_t s) {
    const dim3 grid(std::max(1, std::min(max_inst, 2048)));
    if (b.part)
        hipLaunchKernelGGL(batch_totals_kernel<2>, grid, dim3(VT), 0, s, list, count, item_range, a, b);
    else
        hipLaunchKernelGGL(batch_totals_kernel<1>, grid, dim3(VT), 0, s, list, count, item_range, a, b);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

int launch_batch_pcg_step(const batch_groups &G, int max_items, double *R, const double *AP, const double *B,
                          double *Zq, const batch_inst *inst, const int2 *item_range, item_sum pAp, double *item_rr,
                          double *item_rz, cg_state *states, int slot, hipStream_t s) {
    double *nop = nullptr;
    return launch_prec_any<true>(G, max_items, R, AP, B, Zq, nop, inst, item_range, pAp, item_rr, item_rz, states,
                                 slot, s);
}

int launch_batch_pcg_fold(double *X, double *Z, const double *Pv, const batch_chunk *chunks, const int *count,
                          int max_chunks, const int2 *chunk_range, const int2 *item_range, item_sum pAp,
                          cg_state *states, int slot, hipStream_t s) {
    hipLaunchKernelGGL(batch_pcg_fold_kernel, dim3(std::max(1, std::min(max_chunks, 2048))), dim3(VT), 0, s, X, Z, Pv,
                       chunks, count, chunk_range, item_range, pAp, states, slot);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

int launch_batch_pcg_update(double *Z, double *Pv, const double *Zq, const batch_chunk *chunks, const int *count,
                            int max_chunks, const int2 *chunk_range, const int2 *item_range, item_sum rr,
                            item_sum rz, cg_state *states, int slot, hipStream_t s) {
    hipLaunchKernelGGL(batch_pcg_update_kernel, dim3(std::max(1, std::min(max_chunks, 2048))), dim3(VT), 0, s, Z, Pv,
                       Zq, chunks, count, chunk_range, item_range, rr, rz, states, slot);
    SIPG_HIP_TRY(hipGetLastError());
    return SIPG_OK;
}

}  // namespace sipg_internal
