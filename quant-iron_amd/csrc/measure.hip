// measure.hip — State::measure / measure_n on the device (state.rs:525-784):
// FP64 outcome histogram over the measured qubits, FP64 cumulative scan in
// the reference's sequential order, per-shot search with injected uniforms,
// and collapse + renormalisation into a destination state.
#include <algorithm>

#include "qi_internal.h"
#include "reduce_util.h"

namespace qi {

namespace {

__device__ __forceinline__ uint64_t insert_zeros(uint64_t k, uint64_t fixed) {
    while (fixed) {
        unsigned p = __builtin_ctzll(fixed);
        k = ((k >> p) << (p + 1)) | (k & ((uint64_t(1) << p) - 1));
        fixed &= fixed - 1;
    }
    return k;
}

// Spread the low bits of `o` onto the set bits of `mask` (ascending).
__device__ __host__ __forceinline__ uint64_t deposit(uint64_t o, uint64_t mask) {
    uint64_t r = 0;
    for (int b = 0; mask; b++) {
        uint64_t low = mask & (~mask + 1);
        if ((o >> b) & 1) r |= low;
        mask &= mask - 1;
    }
    return r;
}

template <typename T> __device__ __forceinline__ double nsq(T a) {
    double re = a.x, im = a.y;
    return re * re + im * im;
}

// One thread per bin: sum over the 2^rest indices of the bin, in order.
template <typename T>
__global__ __launch_bounds__(256) void k_hist_thread(const T *__restrict__ psi, uint64_t dmask, uint64_t bins,
                                                     uint64_t rest_items, double *__restrict__ probs) {
    uint64_t o = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (o >= bins) return;
    uint64_t base = deposit(o, dmask);
    DD v = dd_zero();
    for (uint64_t r = 0; r < rest_items; r++) dd_acc(v, nsq(psi[insert_zeros(r, dmask) | base]));
    probs[o] = v.s + v.c;
}

// Gather the bits of x at the set bits of `mask` (ascending), the inverse of
// deposit.
__device__ __host__ __forceinline__ uint64_t extract(uint64_t x, uint64_t mask) {
    uint64_t r = 0;
    for (int b = 0; mask; b++) {
        r |= uint64_t((x & mask & (~mask + 1)) != 0) << b;
        mask &= mask - 1;
    }
    return r;
}

// Index bits inside a wave's 1 KiB row: 16-byte units of 64 lanes.
template <typename T> constexpr int kRowBits = sizeof(T) == 8 ? 7 : 6;

// Rows: one wave sums the bins of one setting of the measured qubits at bit
// kRowBits and above, over `per` settings (from chunk * per) of the unmeasured
// ones there. A lane keeps a sum per amplitude of its unit, so every load is a
// full 1 KiB row whatever the measured set, eight rows in flight; the
// unmeasured qubits of the row are folded across lanes at the end. part == 0:
// the bins go straight to probs, else chunk c's sums to part[(c, bin)].
// Bound by HBM: 28 qubits complex64, the low 20 measured, 0.41 ms (5.2 TB/s)
// against 1.69 ms with one thread per bin (one 8-byte load in flight, its index
// rebuilt bit by bit), which states smaller than a row keep.
template <typename T>
__global__ __launch_bounds__(256) void k_hist_rows(const T *__restrict__ psi, uint64_t outer, uint32_t row_mask,
                                                   uint64_t free_outer, uint64_t settings, uint64_t per, uint64_t waves,
                                                   uint64_t bins, double *__restrict__ probs, double *__restrict__ part) {
    constexpr int RB = kRowBits<T>, U = sizeof(T) == 8 ? 2 : 1, D = 8;
    typedef float F4 __attribute__((ext_vector_type(4)));
    const uint32_t lane = threadIdx.x & 63;
    const uint64_t w0 = uint64_t(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (uint64_t w = w0; w < waves; w += uint64_t(gridDim.x) * 4) {
        const uint64_t o = w & (settings - 1), chunk = w >> __builtin_ctzll(settings);
        const uint64_t hi = deposit(o, outer);
        DD v[U];
#pragma unroll
        for (int k = 0; k < U; k++) v[k] = dd_zero();
        // the free outer qubits' settings in ascending order: add 1 through the others' bits
        uint64_t f = deposit(chunk * per, free_outer);
        const T *row = psi + lane * U;
        for (uint64_t r = 0; r < per; r += D) {
            F4 x[D];
#pragma unroll
            for (int d = 0; d < D; d++) {
                if (per >= D || d < (int)per) x[d] = __builtin_nontemporal_load(reinterpret_cast<const F4 *>(row + ((hi | f) << RB)));
                f = ((f | ~free_outer) + 1) & free_outer;
            }
#pragma unroll
            for (int d = 0; d < D; d++) {
                if (!(per >= D || d < (int)per)) break;
                const T *a = reinterpret_cast<const T *>(&x[d]);
#pragma unroll
                for (int k = 0; k < U; k++) dd_acc(v[k], nsq(a[k]));
            }
        }
        uint32_t mine = 0;  // row bits not measured: this lane writes where they are 0
        if (U == 2 && !(row_mask & 1)) {
            v[0] = dd_add(v[0], v[U - 1]);
            mine |= 1;
        }
#pragma unroll
        for (int b = 0; b < 6; b++) {
            if ((row_mask >> (b + U - 1)) & 1) continue;
#pragma unroll
            for (int k = 0; k < U; k++) v[k] = dd_add(v[k], dd_shfl_xor(v[k], 1 << b));
            mine |= 1u << (b + U - 1);
        }
#pragma unroll
        for (int k = 0; k < U; k++) {
            const uint32_t e = lane * U + k;
            if (e & mine) continue;
            const uint64_t bin = (o << __popc(row_mask)) | extract(e, row_mask);
            if (!part) probs[bin] = v[k].s + v[k].c;
            else { part[(chunk * bins + bin) * 2] = v[k].s; part[(chunk * bins + bin) * 2 + 1] = v[k].c; }
        }
    }
}

// Fold the chunks of each bin: many bins, one thread per bin in chunk order;
// few bins (bins < kFoldBlockBins), one workgroup per bin in a fixed tree.
constexpr uint64_t kFoldBlockBins = 1024;
__global__ __launch_bounds__(256) void k_fold_bins(const double *__restrict__ part, uint64_t bins, uint64_t chunks,
                                                   double *__restrict__ probs) {
    const uint64_t o = uint64_t(blockIdx.x) * 256 + threadIdx.x;
    if (o >= bins) return;
    DD v = dd_zero();
    for (uint64_t c = 0; c < chunks; c++) v = dd_add(v, DD{part[(c * bins + o) * 2], part[(c * bins + o) * 2 + 1]});
    probs[o] = v.s + v.c;
}
__global__ __launch_bounds__(256) void k_fold_bins_block(const double *__restrict__ part, uint64_t bins, uint64_t chunks,
                                                         double *__restrict__ probs) {
    __shared__ double sh[2 * 4];
    const uint64_t o = blockIdx.x;
    DD v[1] = {dd_zero()};
    for (uint64_t c = threadIdx.x; c < chunks; c += 256)
        v[0] = dd_add(v[0], DD{part[(c * bins + o) * 2], part[(c * bins + o) * 2 + 1]});
    block_reduce_dd<1>(v, sh);
    if (threadIdx.x == 0) probs[o] = v[0].s + v[0].c;
}

// Expand a histogram over the distinct measured qubits to the 2^m outcomes of
// the listed qubits (duplicates allowed); inconsistent outcomes get 0.
struct ExpandSlots {
    uint8_t s[64];  // of each listed qubit among the distinct ones, ascending
};
// The value of outcome o of the m listed qubits.
__device__ __forceinline__ double expanded(const double *__restrict__ hd, uint64_t o, const ExpandSlots &slot, int m) {
    uint64_t d = 0, seen = 0;
    bool ok = true;
    for (int b = 0; b < m; b++) {
        int s = slot.s[b];
        uint64_t bit = (o >> b) & 1;
        if ((seen >> s) & 1) { if (((d >> s) & 1) != bit) ok = false; }
        else { seen |= uint64_t(1) << s; d |= bit << s; }
    }
    return ok ? hd[d] : 0.0;
}
__global__ __launch_bounds__(256) void k_expand(const double *__restrict__ hd, double *__restrict__ hm, uint64_t bins_m,
                                                ExpandSlots slot, int m) {
    uint64_t o = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (o < bins_m) hm[o] = expanded(hd, o, slot, m);
}

// Sequential scan (state.rs:590-606): total = sum p_i in index order, then
// C_i = C_{i-1} + p_i / total in index order, with the reference's rounding,
// as three launches: the chain of the total, the quotients (in parallel), the
// chain of the cumulative sum. A chain is one lane's dependent FP64 additions:
// the rest of the workgroup stages the values in LDS a block ahead, the lane
// reads them sixteen ahead of their additions. Up to a block of values, one
// launch does the three.
constexpr int kChainBlock = 2048;  // values staged at a time
struct Group16 {
    double2 x[8];
};
__device__ __forceinline__ Group16 group_at(const double *lds) {
    Group16 r;
#pragma unroll
    for (int j = 0; j < 8; j++) r.x[j] = reinterpret_cast<const double2 *>(lds)[j];
    return r;
}
// cum + lds[0] + ... + lds[cnt - 1] by one lane; with CDF every partial sum goes
// to cdf[i]. lds holds kChainBlock values.
template <bool CDF>
__device__ __forceinline__ double chain_block(const double *lds, int cnt, double cum, double *__restrict__ cdf) {
    Group16 nxt = group_at(lds);
    int i = 0;
    for (; i + 16 <= cnt; i += 16) {
        const Group16 cur = nxt;
        nxt = group_at(lds + (i + 32 <= kChainBlock ? i + 16 : i));
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (CDF) {
            double2 v[8];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                v[j].x = (j ? v[j - 1].y : cum) + cur.x[j].x;
                v[j].y = v[j].x + cur.x[j].y;
            }
            cum = v[7].y;
#pragma unroll
            for (int j = 0; j < 8; j++) *reinterpret_cast<double2 *>(cdf + i + 2 * j) = v[j];
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++) { cum += cur.x[j].x; cum += cur.x[j].y; }
        }
    }
    for (; i < cnt; i++) {
        cum += lds[i];
        if constexpr (CDF) cdf[i] = cum;
    }
    return cum;
}
// cum + p[lo] + ... + p[hi - 1]; with CDF every partial sum goes to cdf[i].
// 256 threads; buf: 2 blocks. The result is valid in thread 0.
template <bool CDF>
__device__ __forceinline__ double chain(const double *__restrict__ p, uint64_t lo, uint64_t hi, double cum,
                                        double *__restrict__ cdf, double (*buf)[kChainBlock]) {
    const int tid = threadIdx.x;
    auto stage = [&](int b, uint64_t at, int first, int threads) {  // the block at `at`, zeros past hi
        for (int i = tid - first; i < kChainBlock / 2 && i >= 0; i += threads) {
            const uint64_t k = at + 2 * i;
            double2 v = make_double2(0.0, 0.0);
            if (k + 1 < hi) v = *reinterpret_cast<const double2 *>(p + k);
            else if (k < hi) v.x = p[k];
            reinterpret_cast<double2 *>(buf[b])[i] = v;
        }
    };
    stage(0, lo, 0, 256);
    __syncthreads();
    int b = 0;
    for (uint64_t at = lo; at < hi; at += kChainBlock, b ^= 1) {
        if (tid >= 64 && at + kChainBlock < hi) stage(b ^ 1, at + kChainBlock, 64, 192);
        if (tid == 0) {
            const int cnt = hi - at < kChainBlock ? int(hi - at) : kChainBlock;
            cum = chain_block<CDF>(buf[b], cnt, cum, CDF ? cdf + at : nullptr);
        }
        __syncthreads();
    }
    return cum;
}
// At most one block of values: total, quotients and cumulative sums in one
// launch, each value by the same operations as in three; m > 0: of the listed
// qubits' outcomes, p a histogram over the distinct ones. A measurement of a few
// qubits is a handful of launches and one read-back: one of 4 qubits 37 us
// with one launch here, 63 with three.
__global__ __launch_bounds__(256) void k_chain_small(const double *__restrict__ p, uint32_t bins, ExpandSlots slot, int m,
                                                     double *__restrict__ cdf, double *__restrict__ total_out) {
    __shared__ __attribute__((aligned(16))) double buf[kChainBlock];
    __shared__ double total;
    for (uint32_t i = threadIdx.x; i < kChainBlock; i += 256)
        buf[i] = i >= bins ? 0.0 : m ? expanded(p, i, slot, m) : p[i];
    __syncthreads();
    if (threadIdx.x == 0) *total_out = total = chain_block<false>(buf, (int)bins, 0.0, nullptr);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < bins; i += 256) buf[i] = buf[i] / total;
    __syncthreads();
    if (threadIdx.x == 0) (void)chain_block<true>(buf, (int)bins, 0.0, cdf);
}
__global__ __launch_bounds__(256) void k_chain_total(const double *__restrict__ p, uint64_t bins, double *__restrict__ total_out) {
    __shared__ __attribute__((aligned(16))) double buf[2][kChainBlock];
    const double total = chain<false>(p, 0, bins, 0.0, nullptr, buf);
    if (threadIdx.x == 0) *total_out = total;
}
__global__ __launch_bounds__(256) void k_quotients(double *__restrict__ p, uint64_t bins, const double *__restrict__ total) {
    const uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i < bins) p[i] = p[i] / *total;
}
__global__ __launch_bounds__(256) void k_chain_cdf(const double *__restrict__ q, uint64_t bins, double *__restrict__ cdf) {
    __shared__ __attribute__((aligned(16))) double buf[2][kChainBlock];
    (void)chain<true>(q, 0, bins, 0.0, cdf, buf);
}

// Large histograms: chunk totals, their sequential prefix, then each chunk is
// scanned sequentially from its prefix, one workgroup per chunk. Agrees with the
// sequential rule up to rounding of the chunk prefixes.
constexpr uint64_t kScanChunk = 1024;
__global__ __launch_bounds__(256) void k_scan_chunk_tot(const double *__restrict__ p, uint64_t bins, double *__restrict__ tot) {
    const uint64_t c = uint64_t(blockIdx.x) * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint64_t lo = c * kScanChunk, hi = lo + kScanChunk < bins ? lo + kScanChunk : bins;
    if (lo >= bins) return;  // whole waves
    DD v = dd_zero();
    for (uint64_t i = lo + lane; i < hi; i += 64) dd_acc(v, p[i]);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v = dd_add(v, dd_shfl_xor(v, m));
    if (lane == 0) { tot[2 * c] = v.s; tot[2 * c + 1] = v.c; }
}
// tot[2 c] <- the sum of the chunks before c: each thread sums a run of
// chunks, the runs' sums are scanned in LDS, each thread fills its run.
__global__ __launch_bounds__(256) void k_scan_chunk_prefix(double *__restrict__ tot, uint64_t nchunks, double *__restrict__ total_out) {
    __shared__ double ss[256], sc[256];
    const uint64_t per = (nchunks + 255) / 256, lo = threadIdx.x * per, hi = lo + per < nchunks ? lo + per : nchunks;
    DD run = dd_zero();
    for (uint64_t c = lo; c < hi; c++) run = dd_add(run, DD{tot[2 * c], tot[2 * c + 1]});
    ss[threadIdx.x] = run.s; sc[threadIdx.x] = run.c;
    __syncthreads();
    for (int d = 1; d < 256; d <<= 1) {
        DD left = dd_zero();
        if ((int)threadIdx.x >= d) left = DD{ss[threadIdx.x - d], sc[threadIdx.x - d]};
        __syncthreads();
        run = dd_add(left, run);
        ss[threadIdx.x] = run.s; sc[threadIdx.x] = run.c;
        __syncthreads();
    }
    if (threadIdx.x == 255) *total_out = run.s + run.c;
    DD at = threadIdx.x ? DD{ss[threadIdx.x - 1], sc[threadIdx.x - 1]} : dd_zero();
    for (uint64_t c = lo; c < hi; c++) {
        const DD t{tot[2 * c], tot[2 * c + 1]};
        tot[2 * c] = at.s + at.c;
        at = dd_add(at, t);
    }
}
__global__ __launch_bounds__(256) void k_scan_chunk_fill(const double *__restrict__ q, uint64_t bins, const double *__restrict__ tot,
                                                         const double *__restrict__ total_p, double *__restrict__ cdf) {
    __shared__ __attribute__((aligned(16))) double buf[2][kChainBlock];
    const uint64_t c = blockIdx.x, lo = c * kScanChunk;
    const uint64_t hi = lo + kScanChunk < bins ? lo + kScanChunk : bins;
    (void)chain<true>(q, lo, hi, tot[2 * c] / *total_p, cdf, buf);
}

// Per shot: first i with u < C_i, else the last bin (state.rs:604-619).
__global__ __launch_bounds__(256) void k_sample(const double *__restrict__ cdf, uint64_t bins, const double *__restrict__ u,
                                                uint64_t shots, uint64_t *__restrict__ out) {
    uint64_t s = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (s >= shots) return;
    double x = u[s];
    uint64_t lo = 0, hi = bins;  // first index with x < cdf[i]
    while (lo < hi) {
        uint64_t mid = lo + (hi - lo) / 2;
        if (x < cdf[mid]) hi = mid; else lo = mid + 1;
    }
    out[s] = lo < bins ? lo : bins - 1;
}

// Keep the amplitudes of the sampled outcome, zero the rest; partial sums of
// the kept |a|^2.
template <typename T>
__global__ __launch_bounds__(256) void k_collapse(const T *src, T *dst, uint64_t dim,
                                                  uint64_t dmask, uint64_t want, double *__restrict__ part) {
    __shared__ double sh[2 * 4];
    DD v[1] = {dd_zero()};
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < dim; i += uint64_t(gridDim.x) * blockDim.x) {
        T a = src[i];
        if ((i & dmask) == want) dd_acc(v[0], nsq(a));
        else { a.x = 0; a.y = 0; }
        dst[i] = a;
    }
    block_reduce_dd<1>(v, sh);
    if (threadIdx.x == 0) { part[blockIdx.x * 2] = v[0].s; part[blockIdx.x * 2 + 1] = v[0].c; }
}

// Histogram over `qubits` (bit b = qubits[b]): 2^m FP64 probabilities inside
// ctx.probs. With `later`, a histogram of at most one block is left over the
// distinct qubits (later->m > 0; else it is the result).
struct Unexpanded {
    const double *hd = nullptr;
    ExpandSlots slot{};
    int m = 0;
};
Status histogram(State &s, const uint64_t *qubits, uint32_t m, double **dprobs, Unexpanded *later, hipStream_t st) {
    Ctx &C = *s.ctx;
    // distinct qubits, in ascending order for the bin index
    uint64_t dmask = 0;
    for (uint32_t b = 0; b < m; b++) dmask |= uint64_t(1) << qubits[b];
    const int d = __builtin_popcountll(dmask);
    const uint64_t bins_d = uint64_t(1) << d, bins_m = uint64_t(1) << m;
    const uint64_t rest = uint64_t(1) << (s.n - d);
    // layout in ctx.probs: [hist_d | hist_m | cdf | total]
    size_t need = (bins_d + 2 * bins_m + 64) * sizeof(double);
    Status e = ensure(C.probs, need);
    if (!e.ok()) return e;
    double *hd = (double *)C.probs.p;
    double *hm = hd + bins_d;
    // the listed qubits in ascending order without repeats: the histogram is the result
    bool plain = true;
    ExpandSlots slot{};
    for (uint32_t b = 0; b < m; b++) {
        slot.s[b] = (uint8_t)__builtin_popcountll(dmask & ((uint64_t(1) << qubits[b]) - 1));
        plain = plain && slot.s[b] == b;
    }
    if (plain) hd = hm;
    const int row_bits = s.prec == QI_C128 ? kRowBits<double2> : kRowBits<float2>;
    if ((int)s.n < row_bits) {
        int blocks = (int)((bins_d + 255) / 256);
        if (s.prec == QI_C128)
            hipLaunchKernelGGL(k_hist_thread<double2>, dim3(blocks), dim3(256), 0, st, (const double2 *)s.d, dmask, bins_d, rest, hd);
        else
            hipLaunchKernelGGL(k_hist_thread<float2>, dim3(blocks), dim3(256), 0, st, (const float2 *)s.d, dmask, bins_d, rest, hd);
    } else {
        const uint64_t outer = dmask >> row_bits, all_outer = (uint64_t(1) << (s.n - row_bits)) - 1;
        const uint64_t settings = uint64_t(1) << __builtin_popcountll(outer), frees = (all_outer + 1) / settings;
        // waves to fill the chip, each with eight rows or more to load
        uint64_t chunks = 1;
        while (settings * chunks < 8192 && frees / chunks > 8) chunks *= 2;
        const uint64_t per = frees / chunks, waves = settings * chunks;
        const uint32_t row_mask = uint32_t(dmask & ((uint64_t(1) << row_bits) - 1));
        double *part = nullptr;
        if (chunks > 1) {
            e = ensure(C.red, bins_d * chunks * 2 * sizeof(double));
            if (!e.ok()) return e;
            part = (double *)C.red.p;
        }
        const unsigned blocks = (unsigned)std::min<uint64_t>((waves + 3) / 4, uint64_t(1) << 22);
        if (s.prec == QI_C128)
            hipLaunchKernelGGL(k_hist_rows<double2>, dim3(blocks), dim3(256), 0, st, (const double2 *)s.d, outer, row_mask,
                               all_outer & ~outer, settings, per, waves, bins_d, hd, part);
        else
            hipLaunchKernelGGL(k_hist_rows<float2>, dim3(blocks), dim3(256), 0, st, (const float2 *)s.d, outer, row_mask,
                               all_outer & ~outer, settings, per, waves, bins_d, hd, part);
        if (chunks > 1 && bins_d >= kFoldBlockBins)
            hipLaunchKernelGGL(k_fold_bins, dim3((unsigned)((bins_d + 255) / 256)), dim3(256), 0, st, (const double *)part, bins_d, chunks, hd);
        else if (chunks > 1)
            hipLaunchKernelGGL(k_fold_bins_block, dim3((unsigned)bins_d), dim3(256), 0, st, (const double *)part, bins_d, chunks, hd);
    }
    if (later) *later = Unexpanded{hd, slot, 0};
    if (!plain && later && bins_m <= kChainBlock) later->m = (int)m;
    else if (!plain)
        hipLaunchKernelGGL(k_expand, dim3((unsigned)((bins_m + 255) / 256)), dim3(256), 0, st, hd, hm, bins_m, slot, (int)m);
    QI_HIP_TRY(hipGetLastError());
    *dprobs = hm;
    return Status{};
}

}  // namespace

Status measure_probs_device(State &s, const uint64_t *qubits, uint32_t m, double **dprobs, hipStream_t st) {
    return histogram(s, qubits, m, dprobs, nullptr, st);
}

// Keep the amplitudes whose measured bits spell `outcome` (bit b of the
// outcome = qubit qubits[b]), renormalise by sqrt(sum |a|^2) when that sum
// exceeds f64::EPSILON (state.rs:622-654). `dst` may be `s`.
Status collapse_outcome(State &s, State &dst, const uint64_t *qubits, uint32_t m, uint64_t outcome, hipStream_t st) {
    Ctx &C = *s.ctx;
    uint64_t dmask = 0, want = 0;
    for (uint32_t b = 0; b < m; b++) {
        dmask |= uint64_t(1) << qubits[b];
        if ((outcome >> b) & 1) want |= uint64_t(1) << qubits[b];
    }
    uint64_t dim = uint64_t(1) << s.n;
    int blocks = (int)std::min<uint64_t>(2048, (dim + 2047) / 2048);
    Status e = ensure(C.red, size_t(blocks) * 2 * sizeof(double));
    if (!e.ok()) return e;
    e = ensure(C.red_out, 64 * sizeof(double));
    if (!e.ok()) return e;
    if (s.prec == QI_C128)
        hipLaunchKernelGGL(k_collapse<double2>, dim3(blocks), dim3(256), 0, st, (const double2 *)s.d, (double2 *)dst.d, dim,
                           dmask, want, (double *)C.red.p);
    else
        hipLaunchKernelGGL(k_collapse<float2>, dim3(blocks), dim3(256), 0, st, (const float2 *)s.d, (float2 *)dst.d, dim,
                           dmask, want, (double *)C.red.p);
    hipLaunchKernelGGL(k_reduce_partials<1>, dim3(1), dim3(256), 0, st, (const double *)C.red.p, blocks, (double *)C.red_out.p);
    QI_HIP_TRY(hipGetLastError());
    QI_HIP_TRY(hipMemcpyAsync(C.host_pinned, C.red_out.p, sizeof(double), hipMemcpyDeviceToHost, st));
    QI_HIP_TRY(hipStreamSynchronize(st));
    double ns = C.host_pinned[0];
    if (ns > 2.220446049250313e-16) {  // state.rs:649-654
        e = launch_div_real(dst, std::sqrt(ns), st);
        if (!e.ok()) return e;
    }
    return Status{};
}

Status measure_sample_collapse(State &s, State &dst, const uint64_t *qubits, uint32_t m, const double *uniforms,
                               size_t shots, uint64_t *outcomes_host, bool collapse, hipStream_t st) {
    Ctx &C = *s.ctx;
    double *hm = nullptr;
    Unexpanded hist;
    Status e = histogram(s, qubits, m, &hm, &hist, st);
    if (!e.ok()) return e;
    const uint64_t bins = uint64_t(1) << m;
    double *cdf = hm + bins;
    double *tot = cdf + bins;  // 64 doubles reserved; chunk totals go to ctx.red
    // total and cdf
    const double *q = hm;  // the quotients p_i / total replace the histogram (of more than one block)
    const unsigned qblocks = (unsigned)((bins + 255) / 256);
    if (bins <= kChainBlock) {
        hipLaunchKernelGGL(k_chain_small, dim3(1), dim3(256), 0, st, hist.m ? hist.hd : (const double *)hm, (uint32_t)bins, hist.slot,
                           hist.m, cdf, tot);
    } else if (bins <= (uint64_t(1) << 16)) {
        hipLaunchKernelGGL(k_chain_total, dim3(1), dim3(256), 0, st, (const double *)hm, bins, tot);
        hipLaunchKernelGGL(k_quotients, dim3(qblocks), dim3(256), 0, st, hm, bins, (const double *)tot);
        hipLaunchKernelGGL(k_chain_cdf, dim3(1), dim3(256), 0, st, q, bins, cdf);
    } else {
        uint64_t nch = (bins + kScanChunk - 1) / kScanChunk;
        e = ensure(C.red, nch * 2 * sizeof(double));
        if (!e.ok()) return e;
        double *ct = (double *)C.red.p;
        hipLaunchKernelGGL(k_scan_chunk_tot, dim3((unsigned)((nch + 3) / 4)), dim3(256), 0, st, (const double *)hm, bins, ct);
        hipLaunchKernelGGL(k_scan_chunk_prefix, dim3(1), dim3(256), 0, st, ct, nch, tot);
        hipLaunchKernelGGL(k_quotients, dim3(qblocks), dim3(256), 0, st, hm, bins, (const double *)tot);
        hipLaunchKernelGGL(k_scan_chunk_fill, dim3((unsigned)nch), dim3(256), 0, st, q, bins, (const double *)ct,
                           (const double *)tot, cdf);
    }
    // uniforms and outcomes through ctx.aux: [outcomes | uniforms]
    e = ensure(C.aux, shots * (sizeof(uint64_t) + sizeof(double)) + 64);
    if (!e.ok()) return e;
    uint64_t *dout = (uint64_t *)C.aux.p;
    double *du = (double *)(dout + shots);
    QI_HIP_TRY(hipMemcpyAsync(du, uniforms, shots * sizeof(double), hipMemcpyHostToDevice, st));
    // total < EPSILON -> UnknownError (state.rs:593-595)
    QI_HIP_TRY(hipMemcpyAsync(C.host_pinned, tot, sizeof(double), hipMemcpyDeviceToHost, st));
    hipLaunchKernelGGL(k_sample, dim3((unsigned)((shots + 255) / 256)), dim3(256), 0, st, cdf, bins, du, (uint64_t)shots, dout);
    QI_HIP_TRY(hipGetLastError());
    QI_HIP_TRY(hipMemcpyAsync(outcomes_host, dout, shots * sizeof(uint64_t), hipMemcpyDeviceToHost, st));
    QI_HIP_TRY(hipStreamSynchronize(st));
    if (C.host_pinned[0] < 2.220446049250313e-16) return make_err(QI_ERR_UNKNOWN);
    if (!collapse) return Status{};
    return collapse_outcome(s, dst, qubits, m, outcomes_host[0], st);
}

}  // namespace qi
