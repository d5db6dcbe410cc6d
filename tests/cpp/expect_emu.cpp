// CPU model of k_expect_tiles and k_apply_tiles (expect.hip): plans random
// SumOps with plan_expect and plan_apply and evaluates the plan's tables on a random state the way the
// kernel does, against the direct sum over terms. Exit code 0 when every case
// agrees; prints the worst difference.
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "../../quant-iron_amd/csrc/expect_plan.h"

using cd = std::complex<double>;
using namespace qi;

static int pc(uint64_t x) { return __builtin_popcountll(x); }

static cd direct(const std::vector<cd> &psi, const qi_pauli_term &t) {
    static const cd ph[4] = {{1, 0}, {0, -1}, {-1, 0}, {0, 1}};  // (-i)^ny
    cd s = 0;
    for (uint64_t i = 0; i < psi.size(); i++)
        s += std::conj(psi[i]) * psi[i ^ t.x_mask] * (pc(i & t.z_mask) & 1 ? -1.0 : 1.0);
    return s * ph[pc(t.x_mask & t.z_mask) & 3] * cd(t.c_re, t.c_im);
}

static cd planned(const std::vector<cd> &psi, uint32_t n, const ExpPlan &p) {
    cd total = 0;
    for (size_t ip = 0; ip < p.npasses; ip++) {
        const ExpPass &ps = p.passes[ip];
        auto global = [&](uint64_t base, uint32_t l) {
            for (int k = 0; k < p.K; k++) base |= uint64_t((l >> k) & 1u) << exp_pos(ps.pos, k);
            return base;
        };
        for (uint64_t t = 0; t < (psi.size() >> p.K); t++) {
            uint64_t base = t;
            for (int k = 0; k < p.K; k++)
                base = ((base >> exp_pos(ps.pos, k)) << (exp_pos(ps.pos, k) + 1)) | (base & ((uint64_t(1) << exp_pos(ps.pos, k)) - 1));
            for (uint32_t si = ps.s0; si < ps.s0 + ps.ns; si++) {
                const ExpSet &st = p.sets[si];
                for (uint32_t tid = 0; tid < (1u << (p.K - 4)); tid++) {
                    uint32_t tl = tid;
                    for (int j = 0; j < 4; j++) {
                        const uint32_t b = exp_pos(&st.pos, j);
                        tl = ((tl >> b) << (b + 1)) | (tl & ((1u << b) - 1));
                    }
                    auto slot = [&](uint32_t s) {
                        uint32_t l = tl;
                        for (int j = 0; j < 4; j++) l |= ((s >> j) & 1u) << exp_pos(&st.pos, j);
                        return l;
                    };
                    for (uint32_t ui = st.u0; ui < st.u0 + st.nu; ui++) {
                        const ExpUnit &un = p.units[ui];
                        const uint32_t xm = un.code() & 15;
                        if ((un.flags() & kExpReuse) && (ui == st.u0 || p.units[ui - 1].code() != un.code() || p.units[ui - 1].xl() != un.xl() ||
                                                       ((p.units[ui - 1].flags() ^ un.flags()) & kExpHigh)))
                            return cd(1e300, 0);
                        const int pivot = xm ? 31 - __builtin_clz(xm) : -1;
                        for (uint32_t k = 0; k < 8; k++) {
                            const uint32_t s = xm ? ((k >> pivot) << (pivot + 1)) | (k & ((1u << pivot) - 1))
                                                  : k + ((un.flags() & kExpHigh) ? 8u : 0u);
                            const uint32_t la = slot(s), lb = xm ? slot(s ^ xm) : la ^ un.xl();
                            const cd w = std::conj(psi[global(base, la)]) * psi[global(base, lb)];
                            double v = (un.code() & 16 ? w.imag() : w.real()) * un.h[k];
                            if ((pc(base & un.zo) + pc(tl & un.zl)) & 1) v = -v;
                            total += un.flags() & kExpImag ? cd(0, v) : cd(v, 0);
                        }
                    }
                    if (st.diag)
                        for (uint32_t pat = 0; pat < 16; pat++)
                            for (uint32_t d = st.doff[pat]; d < st.doff[pat + 1]; d++)
                                for (uint32_t s = 0; s < 16; s++) {
                                    const int odd = pc(base & p.diags[d].zo) + pc(tl & p.diags[d].zl) + pc(s & pat);
                                    total += std::norm(psi[global(base, slot(s))]) * ((odd & 1) ? -1.0 : 1.0) *
                                             cd(p.diags[d].re, p.diags[d].im);
                                }
                }
            }
        }
    }
    (void)n;
    return total;
}

// The result of the SumOp's product by the apply plan's tables.
template <typename R> static std::vector<cd> applied(const std::vector<cd> &psi, const ApplyPlan<R> &p) {
    std::vector<cd> out(psi.size(), cd(0, 0));
    const uint32_t slots = apply_slots(p.K, sizeof(R) == 8);
    for (const ApplyPass &ps : p.passes)
        for (uint64_t i = 0; i < psi.size(); i++) {
            const uint64_t base = i & ~ps.qmask;
            uint32_t l = 0, s = 0, tl;
            for (int k = 0; k < p.K; k++) l |= uint32_t((i >> exp_pos(ps.pos, k)) & 1u) << k;
            tl = l;
            for (int j = 0; j < apply_slot_bits(sizeof(R) == 8); j++) {
                s |= ((l >> exp_pos(&slots, j)) & 1u) << j;
                tl &= ~(1u << exp_pos(&slots, j));
            }
            for (uint32_t u = ps.u0; u < ps.u0 + ps.nu; u++) {
                const ApplyUnit<R> &un = p.units[u];
                uint64_t j = base;
                if (un.flags & kApplyRemote) j = i ^ un.x;
                else
                    for (int k = 0; k < p.K; k++) j |= uint64_t(((l ^ un.xl) >> k) & 1u) << exp_pos(ps.pos, k);
                const cd h(un.flags & kApplyRe ? un.re[s] : 0, un.flags & kApplyIm ? un.im[s] : 0);
                out[i] += ((pc(base & un.zo) + pc(tl & un.zl)) & 1 ? -h : h) * psi[j];
            }
            if (ps.diag)
                for (uint32_t pat = 0; pat < 16; pat++)
                    for (uint32_t d = ps.doff[pat]; d < ps.doff[pat + 1]; d++) {
                        const cd c(p.diags[d].re, p.diags[d].im);
                        out[i] += ((pc(base & p.diags[d].zo) + pc(tl & p.diags[d].zl) + pc(s & pat)) & 1 ? -c : c) * psi[i];
                    }
        }
    return out;
}
static std::vector<cd> direct_apply(const std::vector<cd> &psi, const std::vector<qi_pauli_term> &terms) {
    static const cd ph[4] = {{1, 0}, {0, -1}, {-1, 0}, {0, 1}};
    std::vector<cd> out(psi.size(), cd(0, 0));
    for (auto &t : terms)
        for (uint64_t i = 0; i < psi.size(); i++)
            out[i] += psi[i ^ t.x_mask] * ph[pc(t.x_mask & t.z_mask) & 3] * cd(t.c_re, t.c_im) * (pc(i & t.z_mask) & 1 ? -1.0 : 1.0);
    return out;
}
template <typename R> static double apply_error(uint32_t n, const std::vector<cd> &psi, const std::vector<qi_pauli_term> &terms, int &remote) {
    ApplyPlan<R> p;
    plan_apply<R>(n, terms.data(), terms.size(), p);
    for (auto &u : p.units) remote += (u.flags & kApplyRemote) != 0;
    const auto a = applied(psi, p), b = direct_apply(psi, terms);
    double d = 0, s = 0;
    for (size_t i = 0; i < a.size(); i++) { d += std::norm(a[i] - b[i]); s += std::norm(b[i]); }
    return std::sqrt(d / s);
}

int main(int argc, char **argv) {
    std::mt19937_64 rng(argc > 1 ? strtoull(argv[1], nullptr, 10) : 1);
    std::normal_distribution<double> nd;
    double worst = 0;
    int wide = 0, far = 0, passes = 0, remote = 0;
    for (uint32_t n = 4; n <= 16; n++)
        for (int c128 = 0; c128 < 2; c128++)
            for (int kind = 0; kind < 4; kind++) {  // chain, random of low weight, random of any weight, diagonal
                std::vector<cd> psi(size_t(1) << n);
                double ns = 0;
                for (auto &a : psi) { a = cd(nd(rng), nd(rng)); ns += std::norm(a); }
                for (auto &a : psi) a /= std::sqrt(ns);
                std::vector<qi_pauli_term> terms;
                const uint64_t all = (uint64_t(1) << n) - 1;
                const int count = 1 + int(rng() % (kind == 0 ? 1 : 40));
                if (kind == 0)
                    for (uint32_t q = 0; q + 1 < n; q++) {
                        const uint64_t b = uint64_t(3) << q;
                        terms.push_back({b, 0, nd(rng), 0}); terms.push_back({b, b, nd(rng), 0}); terms.push_back({0, b, nd(rng), 0});
                        terms.push_back({0, uint64_t(1) << q, nd(rng), 0});
                    }
                else
                    for (int k = 0; k < count; k++) {
                        uint64_t x = kind == 3 ? 0 : rng() & all, z = rng() & all;
                        if (kind == 1) { x &= rng() & rng(); z &= rng(); }
                        if (kind == 2 && k == 0) x = all;
                        terms.push_back({x, z, nd(rng), (rng() & 1) ? nd(rng) : 0.0});
                        if (rng() % 3 == 0) terms.push_back({x, rng() & all, nd(rng), 0.0});  // a group of two
                    }
                std::vector<uint64_t> arena(exp_plan_bytes(terms.size()) / 8 + 2);
                ExpPlan p;
                exp_plan_carve(p, arena.data(), terms.size());
                plan_expect(n, c128 != 0, terms.data(), terms.size(), p);
                cd want = 0;
                double scale = 0;
                for (auto &t : terms) { want += direct(psi, t); scale += std::abs(cd(t.c_re, t.c_im)); }
                cd got = planned(psi, n, p);
                for (size_t f = 0; f < p.nfar; f++)
                    for (auto &t : terms)
                        if (t.x_mask == p.far[f]) got += direct(psi, t);
                const double d = std::abs(got - want) / scale;
                if (!(d < 1e-13) || p.npasses > terms.size() || p.nsets > terms.size() || p.nunits > 4 * terms.size()) {
                    printf("n %u c128 %d kind %d: difference %g\n", n, c128, kind, d);
                    return 1;
                }
                worst = std::max(worst, d);
                const double da = c128 ? apply_error<double>(n, psi, terms, remote) : apply_error<float>(n, psi, terms, remote);
                if (!(da < (c128 ? 1e-13 : 1e-6))) {  // (complex64 tables hold float coefficients)
                    printf("apply n %u c128 %d kind %d: difference %g\n", n, c128, kind, da);
                    return 1;
                }
                for (size_t g = 0; g < p.nunits; g++) wide += !(p.units[g].code() & 15);
                far += (int)p.nfar;
                passes = std::max(passes, (int)p.npasses);
            }
    printf("worst relative difference %.2e, wide units %d, streamed masks %d, passes up to %d\n", worst, wide, far, passes);
    return wide && far && remote && passes > 1 ? 0 : 1;
}
