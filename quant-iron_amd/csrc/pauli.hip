// pauli.hip — PauliString / SumOp kernels (pauli_string.rs:139-287, 453-507).
//
// A Pauli string with masks (x, z) (Y where both are set) acts as
//     (P psi)_i = (-i)^{nY} (-1)^{popcount(i & z)} psi_{i ^ x},
// the product of the single-qubit X/Y/Z actions of operator.rs:474-606 in any
// order. The phase is a whole number of quarter turns, applied exactly by
// swapping and negating parts, so the result equals the reference's
// op-by-op application. The coefficient multiply, cosh/sinh mix and term sums
// then follow the reference's complex operations one for one.
#include "expect_plan.h"
#include "qi_internal.h"

#pragma clang fp contract(off)

namespace qi {

namespace {

template <typename R> struct V2;
template <> struct V2<float> { using T = float2; };
template <> struct V2<double> { using T = double2; };

template <typename T> __device__ __forceinline__ T cmul(T a, T b) {
    T r; r.x = a.x * b.x - a.y * b.y; r.y = a.x * b.y + a.y * b.x; return r;
}
template <typename T> __device__ __forceinline__ T cadd(T a, T b) { T r; r.x = a.x + b.x; r.y = a.y + b.y; return r; }

// Multiply by i^q exactly.
template <typename T> __device__ __forceinline__ T rot(T a, unsigned q) {
    T r;
    switch (q & 3) {
    case 0: r = a; break;
    case 1: r.x = -a.y; r.y = a.x; break;
    case 2: r.x = -a.x; r.y = -a.y; break;
    default: r.x = a.y; r.y = -a.x; break;
    }
    return r;
}

// Quarter turns of (-i)^{nY} (-1)^{popcount(i & z)}.
__device__ __forceinline__ unsigned quarter(uint64_t i, uint64_t z, unsigned q0) {
    return q0 + 2u * (unsigned)__popcll(i & z);
}

__device__ __forceinline__ uint64_t insert_zero(uint64_t k, unsigned p) {
    return ((k >> p) << (p + 1)) | (k & ((uint64_t(1) << p) - 1));
}

struct TermK {
    uint64_t x, z;
    unsigned q0;     // 3 * nY mod 4
    unsigned pivot;  // lowest bit of x (pair kernels)
    double c[2];     // coefficient
    double ch[2], sh[2];
};

// out = (P in) * c. Pairs (i, i ^ x) with the pivot bit of i clear, so the
// same kernel is correct in place.
template <typename R>
__global__ __launch_bounds__(256) void k_pauli_apply(const typename V2<R>::T *in, typename V2<R>::T *out,
                                                     uint64_t items, TermK t) {
    using T = typename V2<R>::T;
    T c; c.x = R(t.c[0]); c.y = R(t.c[1]);
    for (uint64_t k = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; k < items; k += uint64_t(gridDim.x) * blockDim.x) {
        if (t.x == 0) {
            T a = in[k];
            out[k] = cmul(rot(a, quarter(k, t.z, t.q0)), c);
        } else {
            uint64_t i = insert_zero(k, t.pivot), j = i ^ t.x;
            T a = in[i], b = in[j];
            out[i] = cmul(rot(b, quarter(i, t.z, t.q0)), c);
            out[j] = cmul(rot(a, quarter(j, t.z, t.q0)), c);
        }
    }
}

// psi <- psi * cosh(alpha) + (P psi) * sinh(alpha)   (pauli_string.rs:250-261)
template <typename R>
__global__ __launch_bounds__(256) void k_pauli_exp(typename V2<R>::T *psi, uint64_t items, TermK t) {
    using T = typename V2<R>::T;
    T ch, sh;
    ch.x = R(t.ch[0]); ch.y = R(t.ch[1]); sh.x = R(t.sh[0]); sh.y = R(t.sh[1]);
    for (uint64_t k = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; k < items; k += uint64_t(gridDim.x) * blockDim.x) {
        if (t.x == 0) {
            T a = psi[k];
            psi[k] = cadd(cmul(a, ch), cmul(rot(a, quarter(k, t.z, t.q0)), sh));
        } else {
            uint64_t i = insert_zero(k, t.pivot), j = i ^ t.x;
            T a = psi[i], b = psi[j];
            psi[i] = cadd(cmul(a, ch), cmul(rot(b, quarter(i, t.z, t.q0)), sh));
            psi[j] = cadd(cmul(b, ch), cmul(rot(a, quarter(j, t.z, t.q0)), sh));
        }
    }
}

// out_i = sum_t (P_t in)_i * c_t, folded in term order (SumOp::apply of states
// up to 20 qubits, and of a few wide terms).
template <typename R>
__global__ __launch_bounds__(256) void k_sumop_apply(const typename V2<R>::T *__restrict__ in,
                                                     typename V2<R>::T *__restrict__ out, uint64_t dim,
                                                     const TermK *__restrict__ terms, int nt) {
    using T = typename V2<R>::T;
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < dim; i += uint64_t(gridDim.x) * blockDim.x) {
        T acc;
        for (int k = 0; k < nt; k++) {
            T c; c.x = R(terms[k].c[0]); c.y = R(terms[k].c[1]);
            T v = cmul(rot(in[i ^ terms[k].x], quarter(i, terms[k].z, terms[k].q0)), c);
            acc = k == 0 ? v : cadd(acc, v);
        }
        out[i] = acc;
    }
}

// A run of diagonal Pauli terms (x = 0) applied in one pass: amplitude i is
// multiplied by T_b[bits of i on the qubits of table b] for each table b, a
// product over the run's terms of cosh(a_t) + (-1)^{popcount(i & z_t)} sinh(a_t)
// computed on the host in FP64 (apply_exp_factor of a diagonal string,
// pauli_string.rs:237-262). Tables live in LDS for the whole launch.
template <typename R>
__global__ __launch_bounds__(256) void k_diag_tables(typename V2<R>::T *psi, uint64_t dim, DiagPass p,
                                                     const double2 *__restrict__ tables) {
    using T = typename V2<R>::T;
    extern __shared__ double2 lut[];  // p.entries of them
    for (int e = threadIdx.x; e < p.entries; e += blockDim.x) lut[e] = tables[e];
    __syncthreads();
    for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < dim; i += uint64_t(gridDim.x) * blockDim.x) {
        const T a = psi[i];
        double re = a.x, im = a.y;
        for (int b = 0; b < p.ntab; b++) {
            uint32_t idx = 0;
            for (int k = 0; k < p.tab[b].bits; k++) idx |= uint32_t((i >> p.tab[b].pos[k]) & 1u) << k;
            const double2 f = lut[p.tab[b].off + idx];
            const double nr = re * f.x - im * f.y, ni = re * f.y + im * f.x;
            re = nr; im = ni;
        }
        T r; r.x = R(re); r.y = R(im);
        psi[i] = r;
    }
}

TermK make_term(const qi_pauli_term &p) {
    TermK t{};
    t.x = p.x_mask; t.z = p.z_mask;
    unsigned ny = (unsigned)__builtin_popcountll(p.x_mask & p.z_mask);
    t.q0 = (3u * ny) & 3u;
    t.pivot = p.x_mask ? (unsigned)__builtin_ctzll(p.x_mask) : 0;
    t.c[0] = p.c_re; t.c[1] = p.c_im;
    return t;
}

}  // namespace

Status launch_pauli_apply(const State &in, State &out, const qi_pauli_term &p, hipStream_t st) {
    TermK t = make_term(p);
    uint64_t dim = uint64_t(1) << in.n;
    uint64_t items = t.x ? dim / 2 : dim;
    int blocks = pick_blocks(items, 256);
    if (in.prec == QI_C128)
        hipLaunchKernelGGL(k_pauli_apply<double>, dim3(blocks), dim3(256), 0, st, (const double2 *)in.d, (double2 *)out.d, items, t);
    else
        hipLaunchKernelGGL(k_pauli_apply<float>, dim3(blocks), dim3(256), 0, st, (const float2 *)in.d, (float2 *)out.d, items, t);
    QI_HIP_TRY(hipGetLastError());
    return Status{};
}

Status launch_pauli_exp(State &s, const qi_pauli_term &p, double ch_re, double ch_im, double sh_re, double sh_im,
                        hipStream_t st) {
    TermK t = make_term(p);
    t.ch[0] = ch_re; t.ch[1] = ch_im; t.sh[0] = sh_re; t.sh[1] = sh_im;
    uint64_t dim = uint64_t(1) << s.n;
    uint64_t items = t.x ? dim / 2 : dim;
    int blocks = pick_blocks(items, 256);
    if (s.prec == QI_C128)
        hipLaunchKernelGGL(k_pauli_exp<double>, dim3(blocks), dim3(256), 0, st, (double2 *)s.d, items, t);
    else
        hipLaunchKernelGGL(k_pauli_exp<float>, dim3(blocks), dim3(256), 0, st, (float2 *)s.d, items, t);
    QI_HIP_TRY(hipGetLastError());
    return Status{};
}

Status launch_diag_tables(State &s, const DiagPass &p, const double2 *dtables, hipStream_t st) {
    uint64_t dim = uint64_t(1) << s.n;
    int blocks = pick_blocks(dim, 256 * 4);
    const size_t lds = size_t(p.entries) * sizeof(double2);
    if (p.entries < 1 || p.entries > (kDiagTabMax << kDiagTabBits) || p.ntab < 1 || p.ntab > kDiagTabMax)
        return make_err(QI_ERR_INVALID_ARGUMENT, 0, 0, 0, 0, "diagonal table pass");
    if (s.prec == QI_C128)
        hipLaunchKernelGGL(k_diag_tables<double>, dim3(blocks), dim3(256), lds, st, (double2 *)s.d, dim, p, dtables);
    else
        hipLaunchKernelGGL(k_diag_tables<float>, dim3(blocks), dim3(256), lds, st, (float2 *)s.d, dim, p, dtables);
    QI_HIP_TRY(hipGetLastError());
    return Status{};
}

Status launch_sumop_apply(const State &in, State &out, const qi_pauli_term *terms, size_t nt, hipStream_t st) {
    // Gathers of a state that the caches hold are cheaper than tile passes of few
    // workgroups; the crossover lies between 20 and 21 qubits in both precisions
    // (us, one chain or lattice of each size): 4 x 5 qubits 112 / 145 (complex64),
    // 125 / 136 (complex128), 3 x 7: 198 / 156 and 224 / 162.
    // Above, a few terms that no tile holds are gathers too.
    if (in.n > 20 && !apply_as_gathers(in.n, in.prec == QI_C128, terms, nt)) return sumop_apply_tiles(in, out, terms, nt, st);
    Ctx &C = *in.ctx;
    std::vector<TermK> h(nt);
    for (size_t k = 0; k < nt; k++) h[k] = make_term(terms[k]);
    Status s = ensure(C.ops, nt * sizeof(TermK));
    if (!s.ok()) return s;
    QI_HIP_TRY(hipMemcpyAsync(C.ops.p, h.data(), nt * sizeof(TermK), hipMemcpyHostToDevice, st));
    uint64_t dim = uint64_t(1) << in.n;
    int blocks = pick_blocks(dim, 256);
    if (in.prec == QI_C128)
        hipLaunchKernelGGL(k_sumop_apply<double>, dim3(blocks), dim3(256), 0, st, (const double2 *)in.d, (double2 *)out.d,
                           dim, (const TermK *)C.ops.p, (int)nt);
    else
        hipLaunchKernelGGL(k_sumop_apply<float>, dim3(blocks), dim3(256), 0, st, (const float2 *)in.d, (float2 *)out.d,
                           dim, (const TermK *)C.ops.p, (int)nt);
    QI_HIP_TRY(hipGetLastError());
    QI_HIP_TRY(hipStreamSynchronize(st));  // the term table is reused by the next call
    return Status{};
}

}  // namespace qi
