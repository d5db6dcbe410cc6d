// expect.hip — SumOp::expectation_value (pauli_string.rs:485-507).
//
// k_expect_tiles reads the state in tiles (expect_plan.h) and evaluates every
// term whose X and Y factors lie inside the tile's qubits from that one read:
// the tile is staged in LDS, a thread takes the 16 amplitudes of a register
// set into FP64 registers and forms w = conj(a) b once per pair and x mask.
// Every pair's product is added by two-sum.
// Terms that no tile holds (X support too wide) stream the state, one read per
// x mask (k_expect_far).
#include <algorithm>
#include <cmath>

#include "expect_plan.h"
#include "qi_internal.h"
#include "reduce_util.h"

namespace qi {

namespace {

#pragma clang fp contract(off)

// XOR-linear LDS slot of tile-local index e. complex64: bits 1-3 take the
// bits above them in (pairs stay 16-byte units), complex128: bits 0-2.
template <typename T> __device__ __forceinline__ uint32_t exp_slot(uint32_t e) {
    if constexpr (sizeof(T) == 8) return e ^ ((((e >> 4) ^ (e >> 7) ^ (e >> 10)) & 7u) << 1);
    else return e ^ (((e >> 3) ^ (e >> 6) ^ (e >> 9) ^ (e >> 12)) & 7u);
}
__device__ __forceinline__ uint32_t exp_ins0(uint32_t k, uint32_t p) { return ((k >> p) << (p + 1)) | (k & ((1u << p) - 1)); }

// x with its sign flipped when the low bit of `odd` is set
__device__ __forceinline__ double flip_sign(double x, uint32_t odd) {
    const uint64_t b = (uint64_t)__double_as_longlong(x) ^ ((uint64_t)(odd & 1u) << 63);
    return __longlong_as_double((long long)b);
}

// a += x y by two-sum: the rounding error of the sum goes to a.c (one multiply-add
// less than a product and dd_acc, and the product is not rounded by itself).
__device__ __forceinline__ void dd_fma(DD &a, double x, double y) {
    const double s = __builtin_fma(x, y, a.s), bb = s - a.s;
    a.c += (a.s - (s - bb)) + __builtin_fma(x, y, -bb);
    a.s = s;
}

// The index of tile t's first amplitude: t with a zero inserted at each of the
// K tile qubits. (The positions sit in scalar registers: loaded from memory a
// position per trip is a wait per trip.)
struct TilePos {
    uint64_t lo, hi;
    __device__ __forceinline__ explicit TilePos(const uint32_t *pos)
        : lo(pos[0] | uint64_t(pos[1]) << 32), hi(pos[2] | uint64_t(pos[3]) << 32) {}
    __device__ __forceinline__ uint32_t operator()(int k) const { return uint32_t((k < 8 ? lo : hi) >> (8 * (k & 7))) & 255u; }
};
__device__ __forceinline__ uint64_t tile_base(uint64_t t, const TilePos &pos, int K) {
    for (int k = 0; k < K; k++) {
        const uint32_t b = pos(k);
        t = ((t >> b) << (b + 1)) | (t & ((uint64_t(1) << b) - 1));
    }
    return t;
}
// The low `bits` of tid on the qubits of the tile-local bits from `first` on.
__device__ __forceinline__ uint64_t thread_offset(uint32_t tid, const TilePos &pos, int bits, int first) {
    uint64_t at = 0;
    for (int i = 0; i < bits; i++) at |= uint64_t((tid >> i) & 1u) << pos(i + first);
    return at;
}

// u = Re w (IM 0) or Im w (IM 1), w = conj(a) b, of the 8 pairs (s, s ^ M) of
// the register bits, s with the highest bit of M clear, in ascending order of s.
template <int M, int IM>
__device__ __forceinline__ void pair_products(const double (&ar)[kExpSlots], const double (&ai)[kExpSlots], double (&u)[8]) {
    constexpr int P = 31 - __builtin_clz(M);
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int s = ((k >> P) << (P + 1)) | (k & ((1 << P) - 1)), t = s ^ M;
        if (IM) u[k] = __builtin_fma(ar[s], ai[t], -(ai[s] * ar[t]));
        else u[k] = __builtin_fma(ar[s], ar[t], ai[s] * ai[t]);
    }
}

// What bounds it: FP64 issue (VALU busy 66% of the time) and one read of the
// state per pass (3.0 TB/s), neither hidden well behind the other: a CU holds
// 16 waves (125 VGPRs), in two workgroups at 64 KiB tiles, four at 32 KiB. The
// four-bit register sets share the LDS reads (16 per thread and set) and the
// FP64 conversions among the masks of the set; a Heisenberg bond costs a
// multiply-add pair and a compensated product per amplitude pair, whatever its
// number of terms. 29 qubits, complex64, a chain with fields (113 terms, 29 x
// masks): 66 ms with one read of the state per mask, 5.6 ms in four passes (5.0
// with plain FP64 sums inside a register set, which lose what two large
// products that cancel leave between them).
// The imaginary sums (complex coefficients) take registers that cost half the
// waves, so they have an instance of their own.
template <typename T, bool CPLX>
__global__ __launch_bounds__(512, CPLX ? 2 : 4) void k_expect_tiles(const T *__restrict__ psi, const ExpPass *__restrict__ passes,
                                                      const ExpSet *__restrict__ sets, const ExpUnit *__restrict__ units,
                                                      const ExpDiag *__restrict__ diags, int K, uint32_t per_pass,
                                                      uint64_t tiles, double *__restrict__ part) {
    constexpr bool F32 = sizeof(T) == 8;
    extern __shared__ __attribute__((aligned(16))) unsigned char exp_lds[];
    T *const tile = reinterpret_cast<T *>(exp_lds);
    const uint32_t tid = threadIdx.x, nt = 1u << (K - 4);  // threads that hold amplitudes
    const bool act = tid < nt;
    const ExpPass &ps = passes[blockIdx.x / per_pass];
    // Loads: 16-byte units, thread t takes units t, t + nt, ...: the low K - 4
    // unit bits are the thread's, the rest the unit counter's (uniform).
    constexpr int UB = F32 ? 1 : 0, NU = kExpSlots >> UB, JB = 4 - UB;  // local bits in a unit, units per thread, counter bits
    const TilePos pos4(ps.pos);
    const uint64_t at = thread_offset(tid, pos4, K - 4, UB);
    DD acc[2] = {dd_zero(), dd_zero()};
    for (uint64_t t = blockIdx.x % per_pass; t < tiles; t += per_pass) {
        const uint64_t base = tile_base(t, pos4, K);
        if (act) {
            typedef float F4 __attribute__((ext_vector_type(4)));
            F4 u[NU];
#pragma unroll
            for (int j = 0; j < NU; j++) {
                uint64_t o = 0;
#pragma unroll
                for (int b = 0; b < JB; b++)
                    if ((j >> b) & 1) o |= uint64_t(1) << pos4(K - JB + b);
                u[j] = __builtin_nontemporal_load(reinterpret_cast<const F4 *>(psi + (base | at | o)));
            }
            const uint32_t l0 = exp_slot<T>(tid << UB);
#pragma unroll
            for (int j = 0; j < NU; j++)
                *reinterpret_cast<F4 *>(tile + (l0 ^ exp_slot<T>(uint32_t(j) << (K - JB)))) = u[j];
        }
        __syncthreads();
        for (uint32_t si = ps.s0; si < ps.s0 + ps.ns; si++) {
            const ExpSet &st = sets[si];
            if (!act) continue;
            const uint32_t pos = st.pos;
            const uint32_t tl = exp_ins0(exp_ins0(exp_ins0(exp_ins0(tid, pos & 255u), (pos >> 8) & 255u), (pos >> 16) & 255u), pos >> 24);
            const uint32_t ls = exp_slot<T>(tl);
            uint32_t so[4];
#pragma unroll
            for (int j = 0; j < 4; j++) so[j] = exp_slot<T>(1u << ((pos >> (8 * j)) & 255u));
            double ar[kExpSlots], ai[kExpSlots];
#pragma unroll
            for (int s = 0; s < kExpSlots; s++) {
                uint32_t o = ls;
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if ((s >> j) & 1) o ^= so[j];
                const T a = tile[o];
                ar[s] = a.x;
                ai[s] = a.y;
            }
            double u[8] = {0, 0, 0, 0, 0, 0, 0, 0};
            ExpUnit nxt = units[st.u0];
            for (uint32_t ui = st.u0; ui < st.u0 + st.nu; ui++) {
                const ExpUnit un = nxt;
                nxt = units[ui + 1];  // read a unit ahead (the table ends with a spare)
                // (the amplitudes are opaque per trip: the products of all masks
                // would otherwise be hoisted out of the loop and spilled)
#pragma unroll
                for (int s = 0; s < kExpSlots; s++) asm volatile("" : "+v"(ar[s]), "+v"(ai[s]));
                if (!(un.flags() & kExpReuse)) {
                    switch (un.code()) {
#define QI_M(M) case M: pair_products<M, 0>(ar, ai, u); break; case M + 16: pair_products<M, 1>(ar, ai, u); break;
                        QI_M(1) QI_M(2) QI_M(3) QI_M(4) QI_M(5) QI_M(6) QI_M(7) QI_M(8)
                        QI_M(9) QI_M(10) QI_M(11) QI_M(12) QI_M(13) QI_M(14) QI_M(15)
#undef QI_M
                    default: {  // wide: the partner from LDS
                        const uint32_t lx = exp_slot<T>(un.xl()), hi = un.flags() & kExpHigh ? so[3] : 0u;
#pragma unroll
                        for (int k = 0; k < 8; k++) {
                            uint32_t o = ls ^ hi;
#pragma unroll
                            for (int j = 0; j < 3; j++)
                                if ((k >> j) & 1) o ^= so[j];
                            const T a = tile[o], b = tile[o ^ lx];
                            const double xr = a.x, xi = a.y, br = b.x, bi = b.y;
                            u[k] = un.code() ? __builtin_fma(xr, bi, -(xi * br)) : __builtin_fma(xr, br, xi * bi);
                        }
                    } break;
                    }
                }
                // every product by two-sum: first the unit's own sum, whose sign
                // is the same for all eight
                DD v{u[0] * un.h[0], 0.0};
#pragma unroll
                for (int k = 1; k < 8; k++) dd_fma(v, u[k], un.h[k]);
                const uint32_t odd = __popcll(base & un.zo) + __popc(tl & un.zl);
                if (CPLX && (un.flags() & kExpImag)) {
                    dd_acc(acc[1], flip_sign(v.s, odd));
                    acc[1].c += flip_sign(v.c, odd);
                } else {
                    dd_acc(acc[0], flip_sign(v.s, odd));
                    acc[0].c += flip_sign(v.c, odd);
                }
            }
            if (st.diag) {
                // the signed sums of the coefficients by register-bit pattern, then
                // their Walsh transform: the factor of each |a|^2
                double w[kExpSlots], h[kExpSlots], hi[kExpSlots];
#pragma unroll
                for (int s = 0; s < kExpSlots; s++) w[s] = __builtin_fma(ar[s], ar[s], ai[s] * ai[s]);
#pragma unroll
                for (int p = 0; p < kExpSlots; p++) {
                    double cr = 0.0, ci = 0.0;
#pragma unroll 4  // (four terms' scalar loads in flight)
                    for (uint32_t d = st.doff[p]; d < st.doff[p + 1]; d++) {
                        const ExpDiag &t1 = diags[d];
                        const uint32_t odd = __popcll(base & t1.zo) + __popc(tl & t1.zl);
                        cr += flip_sign(t1.re, odd);
                        if (CPLX) ci += flip_sign(t1.im, odd);
                    }
                    h[p] = cr;
                    hi[p] = ci;
                }
#pragma unroll
                for (int b = 1; b < kExpSlots; b <<= 1)
#pragma unroll
                    for (int s = 0; s < kExpSlots; s++)
                        if (!(s & b)) {
                            const double x = h[s], y = h[s | b], z = hi[s], t1 = hi[s | b];
                            h[s] = x + y;
                            h[s | b] = x - y;
                            if (CPLX) { hi[s] = z + t1; hi[s | b] = z - t1; }
                        }
#pragma unroll
                for (int s = 0; s < kExpSlots; s++) {
                    dd_fma(acc[0], w[s], h[s]);
                    if (CPLX) dd_fma(acc[1], w[s], hi[s]);
                }
            }
        }
        __syncthreads();  // the next tile overwrites the LDS copy
    }
    double *sh = reinterpret_cast<double *>(exp_lds);  // 2 values x 2 doubles per wave
    block_reduce_dd<2>(acc, sh);
    if (tid == 0) {
        part[size_t(blockIdx.x) * 4 + 0] = acc[0].s; part[size_t(blockIdx.x) * 4 + 1] = acc[0].c;
        part[size_t(blockIdx.x) * 4 + 2] = acc[1].s; part[size_t(blockIdx.x) * 4 + 3] = acc[1].c;
    }
}

// A term for the streaming kernel, and the terms of one x mask.
struct TermK {
    uint64_t x, z;
    unsigned q0;  // 3 * nY mod 4
    unsigned pad;
    double c[2];
};
struct FarMask {
    uint64_t x;
    uint32_t t0, nt;
};

// Quarter turns of (-i)^{nY} (-1)^{popcount(i & z)}.
__device__ __forceinline__ unsigned quarter(uint64_t i, uint64_t z, unsigned q0) {
    return q0 + 2u * (unsigned)__popcll(i & z);
}
__device__ __forceinline__ uint64_t insert_zero(uint64_t k, unsigned p) {
    return ((k >> p) << (p + 1)) | (k & ((uint64_t(1) << p) - 1));
}

// Expectation of the terms that no tile holds (x masks wider than a tile, states
// of fewer than 4 qubits), one read of the state per x mask:
//   sum_i conj(psi_i) psi_{i^x} h(i),  h(i) = sum_t c_t i^{q_t(i)}.
// FP64 accumulation with two-sum compensation; per_mask blocks of each mask,
// one partial per block. All masks run in one launch: a mask of many has few
// blocks, and a launch of its own would leave the chip to them alone (26
// qubits, 100 random strings: 324 ms in complex64 and 418 in complex128, in one
// launch 14.6 and 23.0). Bound by HBM and, with few terms, by the latency of a
// thread's two loads in flight: one mask of a 28-qubit complex128 state 1.44 ms.
template <typename T>
__global__ __launch_bounds__(256) void k_expect_far(const T *__restrict__ psi, uint64_t dim, const FarMask *__restrict__ masks,
                                                    uint32_t per_mask, const TermK *__restrict__ all_terms, double *__restrict__ part) {
    __shared__ double sh[4 * 4];
    const FarMask &fm = masks[blockIdx.x / per_mask];
    const uint64_t x = fm.x, items = x ? dim / 2 : dim;
    const unsigned pivot = x ? __builtin_ctzll(x) : 0;
    const TermK *__restrict__ terms = all_terms + fm.t0;
    const int nt = (int)fm.nt;
    DD v[2] = {dd_zero(), dd_zero()};
    for (uint64_t k = uint64_t(blockIdx.x % per_mask) * blockDim.x + threadIdx.x; k < items; k += uint64_t(per_mask) * blockDim.x) {
        uint64_t i = x == 0 ? k : insert_zero(k, pivot);
        uint64_t j = i ^ x;
        double ar = psi[i].x, ai = psi[i].y, br = psi[j].x, bi = psi[j].y;
        // w = conj(a) * b for index i; for the partner j it is conj(w)
        double wr = ar * br + ai * bi, wi = ar * bi - ai * br;
        double hr = 0, hi = 0, gr = 0, gi = 0;
        for (int t = 0; t < nt; t++) {
            unsigned qi_ = quarter(i, terms[t].z, terms[t].q0) & 3;
            double cr = terms[t].c[0], ci = terms[t].c[1];
            // c * i^q
            double pr = qi_ == 0 ? cr : qi_ == 1 ? -ci : qi_ == 2 ? -cr : ci;
            double pi = qi_ == 0 ? ci : qi_ == 1 ? cr : qi_ == 2 ? -ci : -cr;
            hr += pr; hi += pi;
            if (x != 0) {
                unsigned qj = quarter(j, terms[t].z, terms[t].q0) & 3;
                double qr = qj == 0 ? cr : qj == 1 ? -ci : qj == 2 ? -cr : ci;
                double qi2 = qj == 0 ? ci : qj == 1 ? cr : qj == 2 ? -ci : -cr;
                gr += qr; gi += qi2;
            }
        }
        // conj(psi_i) psi_j h(i)
        dd_acc(v[0], wr * hr - wi * hi);
        dd_acc(v[1], wr * hi + wi * hr);
        if (x != 0) {  // conj(psi_j) psi_i h(j) = conj(w) h(j)
            dd_acc(v[0], wr * gr + wi * gi);
            dd_acc(v[1], wr * gi - wi * gr);
        }
    }
    block_reduce_dd<2>(v, sh);
    if (threadIdx.x == 0) {
        part[size_t(blockIdx.x) * 4 + 0] = v[0].s; part[size_t(blockIdx.x) * 4 + 1] = v[0].c;
        part[size_t(blockIdx.x) * 4 + 2] = v[1].s; part[size_t(blockIdx.x) * 4 + 3] = v[1].c;
    }
}

// ---------------------------------------------------------- SumOp::apply --
// acc[s] += h[s] part(s) for the real (IM 0) or imaginary parts of a unit's
// coefficients, signed, with fused multiply-adds; part: the partner of slot s.
__device__ __forceinline__ float flip_sign(float x, uint32_t odd) {
    return __uint_as_float(__float_as_uint(x) ^ (odd << 31));
}

template <bool IM, typename T, typename R, int NS>
__device__ __forceinline__ void apply_part(T (&acc)[NS], const R *__restrict__ h, uint32_t odd, const T (&b)[NS]) {
    R c[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) c[s] = h[s];  // one run of scalar loads
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const R k = flip_sign(c[s], odd);
        if (IM) {
            acc[s].x = fma(-k, b[s].y, acc[s].x);
            acc[s].y = fma(k, b[s].x, acc[s].y);
        } else {
            acc[s].x = fma(k, b[s].x, acc[s].x);
            acc[s].y = fma(k, b[s].y, acc[s].y);
        }
    }
}

// One tile of one pass (expect_plan.h): the input tile goes to LDS, each thread
// keeps the results of its loads' places in registers and takes a partner
// per unit and slot from LDS, or from memory for remote masks. FIRST: the pass
// starts the result, later passes add to it.
// Bound by HBM (a pass moves two or three states: 146 us per later pass of a
// 256 MiB state, 5.5 TB/s) and, where the diagonal terms run, by the latency of
// their scalar loads. 24 qubits, complex128, a 4 x 6 lattice (138 terms, 38
// masks): 0.65 ms in four passes, 1.86 ms as 138 gathers per amplitude.
template <typename T, typename R, bool FIRST, bool CPLX>
__global__ __launch_bounds__(512, 4) void k_apply_tiles(const T *__restrict__ psi, T *__restrict__ res, ApplyPass ps,
                                                     const ApplyUnit<R> *__restrict__ units, const ExpDiag *__restrict__ diags, int K) {
    constexpr bool F32 = sizeof(T) == 8;
    constexpr int SB = apply_slot_bits(!F32), NS = 1 << SB, UB = F32 ? 1 : 0, NU = NS >> UB, JB = SB - UB, U = 1 << UB;
    typedef float F4 __attribute__((ext_vector_type(4)));
    extern __shared__ __attribute__((aligned(16))) unsigned char exp_lds[];
    T *const tile = reinterpret_cast<T *>(exp_lds);
    const uint32_t tid = threadIdx.x;
    const TilePos pos4(ps.pos);
    const uint64_t base = tile_base(blockIdx.x, pos4, K), at = base | thread_offset(tid, pos4, K - SB, UB);
    // the slot bits' steps in memory and in LDS
    uint64_t go[JB];
    uint32_t so[SB];
#pragma unroll
    for (int b = 0; b < JB; b++) {
        go[b] = uint64_t(1) << pos4(K - JB + b);
        so[UB + b] = exp_slot<T>(1u << (K - JB + b));
    }
    if (F32) so[0] = exp_slot<T>(1u);
    const uint32_t tl = tid << UB, ls = exp_slot<T>(tl);
    T acc[NS];
    {
        F4 u[NU];
#pragma unroll
        for (int j = 0; j < NU; j++) {
            uint64_t g = at;
#pragma unroll
            for (int b = 0; b < JB; b++)
                if ((j >> b) & 1) g |= go[b];
            u[j] = *reinterpret_cast<const F4 *>(psi + g);
            if (!FIRST) {
                const F4 r = __builtin_nontemporal_load(reinterpret_cast<const F4 *>(res + g));
                if constexpr (F32) {
                    acc[2 * j].x = r.x; acc[2 * j].y = r.y;
                    acc[2 * j + 1].x = r.z; acc[2 * j + 1].y = r.w;
                } else {
                    acc[j] = __builtin_bit_cast(T, r);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < NU; j++) {
            uint32_t o = ls;
#pragma unroll
            for (int b = 0; b < JB; b++)
                if ((j >> b) & 1) o ^= so[UB + b];
            *reinterpret_cast<F4 *>(tile + o) = u[j];
        }
    }
    if (FIRST)
#pragma unroll
        for (int s = 0; s < NS; s++) { acc[s].x = 0; acc[s].y = 0; }
    __syncthreads();
    for (uint32_t ui = ps.u0; ui < ps.u0 + ps.nu; ui++) {
        const ApplyUnit<R> &un = units[ui];
        const uint32_t flags = un.flags, odd = (__popcll(base & un.zo) + __popc(tl & un.zl)) & 1u;
        T b[NS];
        if (flags & kApplyRemote) {
            const uint64_t x = un.x;
#pragma unroll
            for (int j = 0; j < NU; j++) {
                uint64_t g = at;
#pragma unroll
                for (int k = 0; k < JB; k++)
                    if ((j >> k) & 1) g |= go[k];
                const F4 v = *reinterpret_cast<const F4 *>(psi + ((g ^ x) & ~uint64_t(U - 1)));
                if constexpr (F32) {
                    const bool odd_x = x & 1;
                    b[2 * j].x = odd_x ? v.z : v.x; b[2 * j].y = odd_x ? v.w : v.y;
                    b[2 * j + 1].x = odd_x ? v.x : v.z; b[2 * j + 1].y = odd_x ? v.y : v.w;
                } else {
                    b[j] = __builtin_bit_cast(T, v);
                }
            }
        } else {
            const uint32_t lx = ls ^ exp_slot<T>(un.xl);
#pragma unroll
            for (int s = 0; s < NS; s++) {
                uint32_t o = lx;
#pragma unroll
                for (int k = 0; k < SB; k++)
                    if ((s >> k) & 1) o ^= so[k];
                b[s] = tile[o];
            }
        }
        if (flags & kApplyRe) apply_part<false>(acc, un.re, odd, b);
        if (flags & kApplyIm) apply_part<true>(acc, un.im, odd, b);
    }
    if (ps.diag) {
        // the signed sums of the coefficients by slot-bit pattern, then their
        // Walsh transform: the factor of each slot
        double dr[NS], di[NS];
#pragma unroll
        for (int p = 0; p < NS; p++) {
            double cr = 0.0, ci = 0.0;
#pragma unroll 4  // (four terms' scalar loads in flight)
            for (uint32_t d = ps.doff[p]; d < ps.doff[p + 1]; d++) {
                const ExpDiag &t = diags[d];
                const uint32_t odd = (__popcll(base & t.zo) + __popc(tl & t.zl)) & 1u;
                cr += flip_sign(t.re, odd);
                if (CPLX) ci += flip_sign(t.im, odd);
            }
            dr[p] = cr;
            di[p] = ci;
        }
#pragma unroll
        for (int b = 1; b < NS; b <<= 1)
#pragma unroll
            for (int s = 0; s < NS; s++)
                if (!(s & b)) {
                    const double x = dr[s], y = dr[s | b], z = di[s], w = di[s | b];
                    dr[s] = x + y; dr[s | b] = x - y;
                    if (CPLX) { di[s] = z + w; di[s | b] = z - w; }
                }
#pragma unroll
        for (int s = 0; s < NS; s++) {
            uint32_t o = ls;
#pragma unroll
            for (int b = 0; b < SB; b++)
                if ((s >> b) & 1) o ^= so[b];
            const T b = tile[o];
            const R hr = R(dr[s]), hi = R(di[s]);
            acc[s].x = fma(hr, b.x, acc[s].x);
            acc[s].y = fma(hr, b.y, acc[s].y);
            if (CPLX) {
                acc[s].x = fma(-hi, b.y, acc[s].x);
                acc[s].y = fma(hi, b.x, acc[s].y);
            }
        }
    }
    // A complex product with a coefficient of one part adds zero times the other
    // part: no matter, unless that is infinite or NaN.
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const bool fx = __builtin_isfinite(acc[s].x), fy = __builtin_isfinite(acc[s].y);
        if (fy && !fx) acc[s].y = __builtin_nan("");
        if (fx && !fy) acc[s].x = __builtin_nan("");
    }
#pragma unroll
    for (int j = 0; j < NU; j++) {
        uint64_t g = at;
#pragma unroll
        for (int b = 0; b < JB; b++)
            if ((j >> b) & 1) g |= go[b];
        F4 r;
        if constexpr (F32) r = F4{acc[2 * j].x, acc[2 * j].y, acc[2 * j + 1].x, acc[2 * j + 1].y};
        else r = __builtin_bit_cast(F4, acc[j]);
        __builtin_nontemporal_store(r, reinterpret_cast<F4 *>(res + g));
    }
}

// ------------------------------------------------------------- host side --
// Workgroups: a pass takes up to kExpBlocks / passes of them, a streamed mask
// up to kExpBlocks / 4 / masks, neither fewer than kExpBlocksMin (for at most
// 512 passes and masks: at most 2 kExpBlocksMin * 512 partials).
constexpr uint64_t kExpBlocks = 4096, kExpBlocksMin = 16;

size_t up16(size_t b) { return (b + 15) & ~size_t(15); }

struct ExpLaunch {
    size_t sets, units, diags, far, masks, bytes;  // offsets in the device tables (passes first), their size
    uint32_t per_pass, per_far;
    uint64_t tiles;
    size_t blocks;  // partials of the whole call
};

TermK far_term(const qi_pauli_term &p) {
    TermK t{};
    t.x = p.x_mask; t.z = p.z_mask;
    t.q0 = (3u * (unsigned)__builtin_popcountll(p.x_mask & p.z_mask)) & 3u;
    t.c[0] = p.c_re; t.c[1] = p.c_im;
    return t;
}

// Plans into `arena` (exp_plan_bytes(nt, units)).
ExpLaunch plan_launch(const State &s, const qi_pauli_term *terms, size_t nt, void *arena, size_t units, ExpPlan &p) {
    exp_plan_carve(p, arena, nt, units);
    plan_expect(s.n, s.prec == QI_C128, terms, nt, p);
    size_t nf = 0;
    for (size_t g = 0; g < p.nfar; g++)
        for (uint32_t t = p.far_head[g]; t != UINT32_MAX; t = p.next[t]) nf++;
    ExpLaunch L{};
    L.sets = up16(p.npasses * sizeof(ExpPass));
    L.units = L.sets + up16(p.nsets * sizeof(ExpSet));
    L.diags = L.units + up16((p.nunits + 1) * sizeof(ExpUnit));
    L.far = L.diags + up16(p.ndiags * sizeof(ExpDiag));
    L.masks = L.far + up16(nf * sizeof(TermK));
    L.bytes = L.masks + up16(p.nfar * sizeof(FarMask));
    const uint64_t dim = uint64_t(1) << s.n;
    if (p.npasses) {
        L.tiles = dim >> p.K;
        L.per_pass = (uint32_t)std::min<uint64_t>(L.tiles, std::max<uint64_t>(kExpBlocksMin, kExpBlocks / p.npasses));
    }
    if (p.nfar) L.per_far = (uint32_t)std::min<uint64_t>((dim + 2047) / 2048, std::max<uint64_t>(kExpBlocksMin, kExpBlocks / 4 / p.nfar));
    L.blocks = p.npasses * L.per_pass + p.nfar * L.per_far;
    return L;
}

// Device tables in the order of ExpLaunch's offsets.
void pack_tables(const ExpPlan &p, const ExpLaunch &L, const qi_pauli_term *terms, unsigned char *dst) {
    memcpy(dst, p.passes, p.npasses * sizeof(ExpPass));
    memcpy(dst + L.sets, p.sets, p.nsets * sizeof(ExpSet));
    if (p.npasses) memcpy(dst + L.units, p.units, (p.nunits + 1) * sizeof(ExpUnit));
    memcpy(dst + L.diags, p.diags, p.ndiags * sizeof(ExpDiag));
    TermK *const f = reinterpret_cast<TermK *>(dst + L.far);
    FarMask *const m = reinterpret_cast<FarMask *>(dst + L.masks);
    uint32_t k = 0;
    for (size_t g = 0; g < p.nfar; g++) {
        m[g] = FarMask{p.far[g], k, 0};
        for (uint32_t t = p.far_head[g]; t != UINT32_MAX; t = p.next[t]) f[k++] = far_term(terms[t]);
        m[g].nt = k - m[g].t0;
    }
}

template <typename T>
Status launch_all(const State &s, const ExpPlan &p, const ExpLaunch &L, const unsigned char *tab, double *part, double *out,
                  hipStream_t st) {
    if (p.npasses) {
        const unsigned threads = std::max(64u, 1u << (p.K - 4));
        auto *const kernel = p.complex_out ? k_expect_tiles<T, true> : k_expect_tiles<T, false>;
        hipLaunchKernelGGL(kernel, dim3(L.per_pass * (unsigned)p.npasses), dim3(threads),
                           std::max<size_t>(sizeof(T) << p.K, 512), st, (const T *)s.d, (const ExpPass *)tab,
                           (const ExpSet *)(tab + L.sets), (const ExpUnit *)(tab + L.units),
                           (const ExpDiag *)(tab + L.diags), p.K, L.per_pass, L.tiles, part);
    }
    if (p.nfar)
        hipLaunchKernelGGL(k_expect_far<T>, dim3(L.per_far * (unsigned)p.nfar), dim3(256), 0, st, (const T *)s.d, uint64_t(1) << s.n,
                           (const FarMask *)(tab + L.masks), L.per_far, (const TermK *)(tab + L.far),
                           part + size_t(L.per_pass) * p.npasses * 4);
    hipLaunchKernelGGL(k_reduce_partials<2>, dim3(1), dim3(256), 0, st, (const double *)part, (int)L.blocks, out);
    QI_HIP_TRY(hipGetLastError());
    return Status{};
}

// Uploads the packed tables and runs the launches; the result lands in the
// context's pinned words.
Status expect_run(State &s, const qi_pauli_term *terms, const ExpPlan &p, const ExpLaunch &L, Staging &stage, void *dtab, double *part,
                  double *re, double *im, hipStream_t st) {
    Ctx &C = *s.ctx;
    pack_tables(p, L, terms, stage.p);
    Status e = send_tables(stage, dtab, L.bytes, st);
    if (e.ok())
        e = s.prec == QI_C128 ? launch_all<double2>(s, p, L, (const unsigned char *)dtab, part, C.host_pinned, st)
                              : launch_all<float2>(s, p, L, (const unsigned char *)dtab, part, C.host_pinned, st);
    const hipError_t done = hipStreamSynchronize(st);
    if (!e.ok()) return e;
    QI_HIP_TRY(done);
    *re = C.host_pinned[0];
    *im = C.host_pinned[1];
    // (tiles of real coefficients form no imaginary part: it is zero, or unknown with the real one)
    if (std::isnan(*re) && !p.complex_out) *im = *re;
    return Status{};
}

}  // namespace

namespace {
template <typename T, typename R>
Status apply_tiles(const State &in, State &out, const qi_pauli_term *terms, size_t nt, hipStream_t st) {
    Ctx &C = *in.ctx;
    ApplyPlan<R> p;
    plan_apply<R>(in.n, terms, nt, p);
    const size_t diags = up16(p.units.size() * sizeof(ApplyUnit<R>)), bytes = diags + p.diags.size() * sizeof(ExpDiag);
    Staging tab;
    Status s = ensure(C.ops, bytes);
    if (s.ok()) s = stage_tables(C, bytes, tab);
    if (!s.ok()) return s;
    if (!p.units.empty()) memcpy(tab.p, p.units.data(), p.units.size() * sizeof(ApplyUnit<R>));
    if (!p.diags.empty()) memcpy(tab.p + diags, p.diags.data(), p.diags.size() * sizeof(ExpDiag));
    if (!(s = send_tables(tab, C.ops.p, bytes, st)).ok()) return s;
    const uint64_t tiles = (uint64_t(1) << in.n) >> p.K;
    const unsigned threads = 1u << (p.K - apply_slot_bits(sizeof(R) == 8));  // one slot set each: 512
    for (size_t k = 0; k < p.passes.size(); k++) {
        // (the diagonal terms run in the first pass)
        auto *const kernel = k ? k_apply_tiles<T, R, false, false>
                               : p.complex_diag ? k_apply_tiles<T, R, true, true> : k_apply_tiles<T, R, true, false>;
        hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(threads), sizeof(T) << p.K, st, (const T *)in.d, (T *)out.d,
                           p.passes[k], (const ApplyUnit<R> *)C.ops.p, (const ExpDiag *)((const unsigned char *)C.ops.p + diags), p.K);
    }
    const hipError_t launched = hipGetLastError(), done = hipStreamSynchronize(st);  // the next call reuses the tables and the staging buffer
    QI_HIP_TRY(launched);
    QI_HIP_TRY(done);
    return Status{};
}
}  // namespace

Status sumop_apply_tiles(const State &in, State &out, const qi_pauli_term *terms, size_t nt, hipStream_t st) {
    return in.prec == QI_C128 ? apply_tiles<double2, double>(in, out, terms, nt, st)
                              : apply_tiles<float2, float>(in, out, terms, nt, st);
}

size_t expect_arena_bytes(size_t nt) { return exp_plan_bytes(nt); }
size_t expect_table_bytes(size_t nt) {
    return nt * (sizeof(ExpPass) + sizeof(ExpSet) + 4 * sizeof(ExpUnit) + sizeof(ExpDiag) + sizeof(TermK) + sizeof(FarMask)) + 512;
}

Status sumop_expectation(State &s, const qi_pauli_term *terms, size_t nt, double *re, double *im, hipStream_t st) {
    Ctx &C = *s.ctx;
    const size_t units = exp_max_units(terms, nt);
    std::vector<unsigned char> own;
    unsigned char *arena = nullptr;
    Status e = plan_memory(C, exp_plan_bytes(nt, units), own, &arena);
    if (!e.ok()) return e;
    ExpPlan p;
    Staging stage;
    const ExpLaunch L = plan_launch(s, terms, nt, arena, units, p);
    if (!(e = stage_tables(C, L.bytes, stage)).ok()) return e;
    if (!(e = ensure(C.ops, L.bytes)).ok()) return e;
    if (!(e = ensure(C.red, L.blocks * 4 * sizeof(double))).ok()) return e;
    return expect_run(s, terms, p, L, stage, C.ops.p, (double *)C.red.p, re, im, st);
}

// ---------------------------------------------------- no-allocation variant --
// qi_sumop_expectation_noalloc keeps its tables and block partials in this
// fixed device array instead of the context's growable buffers (the host
// arena and staging buffer of the context hold kNoAllocMaxTerms terms from its
// creation): no allocation on any call. Each device that the library runs on
// holds its own copy until the process ends. Every location a call reads is
// written earlier in the same call, so nothing needs clearing; calls that
// overlap on one device (different contexts, or threads without the context's
// lock) race on it.
namespace {
struct NoAllocScratch {
    unsigned char tab[kNoAllocMaxTerms * (sizeof(ExpPass) + sizeof(ExpSet) + 4 * sizeof(ExpUnit) + sizeof(ExpDiag) +
                                          sizeof(TermK) + sizeof(FarMask)) + 512];  // expect_table_bytes(kNoAllocMaxTerms)
    double part[(kExpBlocks + 2 * kExpBlocksMin * kNoAllocMaxTerms) * 4];
};
}  // namespace

static __device__ __align__(256) unsigned char scratch[sizeof(NoAllocScratch)];

Status noalloc_scratch(int device, void **out) {
    static std::mutex mu;
    static void *ptrs[64] = {nullptr};
    if (device < 0 || device >= 64) return make_err(QI_ERR_INVALID_ARGUMENT, 0, 0, 0, 0, "device index");
    std::lock_guard<std::mutex> lk(mu);
    if (!ptrs[device]) {
        // the host-side name of `scratch` is not a device address: take the
        // address of this device's copy once, with the device current
        void *p = nullptr;
        QI_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        ptrs[device] = p;
    }
    *out = ptrs[device];
    return Status{};
}

Status sumop_expectation_noalloc(State &s, const qi_pauli_term *terms, size_t nt, double *re, double *im, hipStream_t st) {
    void *base = s.ctx->noalloc;
    if (!base) return make_err(QI_ERR_DEVICE, 0, 0, 0, 0, "no scratch address for this device");
    if (nt > (size_t)kNoAllocMaxTerms)
        return make_err(QI_ERR_INVALID_ARGUMENT, nt, kNoAllocMaxTerms, 0, 0, "more terms than the no-allocation maximum (512)");
    *re = 0.0; *im = 0.0;
    if (nt == 0) return Status{};
    NoAllocScratch *sc = reinterpret_cast<NoAllocScratch *>(base);
    Ctx &C = *s.ctx;
    const size_t units = exp_max_units(terms, nt);
    if (exp_plan_bytes(nt, units) > C.plan_arena.size()) return make_err(QI_ERR_DEVICE, 0, 0, 0, 0, "expectation planning memory");
    ExpPlan p;
    const ExpLaunch L = plan_launch(s, terms, nt, C.plan_arena.data(), units, p);
    if (L.bytes > sizeof sc->tab || L.bytes > C.stage_bytes || L.blocks * 4 * sizeof(double) > sizeof sc->part)
        return make_err(QI_ERR_DEVICE, 0, 0, 0, 0, "expectation scratch");
    Staging stage;
    stage.p = C.stage;
    return expect_run(s, terms, p, L, stage, sc->tab, sc->part, re, im, st);
}

}  // namespace qi
