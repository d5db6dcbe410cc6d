// Long SumOps through the planners of expect_plan.cpp: more distinct x masks
// than the greedy search looks through, and thousands of terms on one x mask
// (their units found through the table), against the direct sums; the planning
// time of 65536 terms on one mask. Uses the model in expect_emu.cpp.
#define main emu_main
#include "expect_emu.cpp"
#undef main

#include <chrono>

static double seconds() {
    return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

int main() {
    std::mt19937_64 rng(11);
    std::normal_distribution<double> nd;
    for (uint32_t n : {9u, 14u})
        for (int c128 = 0; c128 < 2; c128++)
            for (int kind = 0; kind < 3; kind++) {  // many masks of any weight, many of low weight, many Z supports on three masks
                const uint64_t all = (uint64_t(1) << n) - 1;
                std::vector<cd> psi(size_t(1) << n);
                double ns = 0;
                for (auto &a : psi) { a = cd(nd(rng), nd(rng)); ns += std::norm(a); }
                for (auto &a : psi) a /= std::sqrt(ns);
                std::vector<qi_pauli_term> terms;
                for (int k = 0; k < 320; k++) {
                    uint64_t x = 1 + rng() % all;
                    if (kind == 1) x = (x & rng() & rng()) | uint64_t(1) << rng() % n;
                    if (kind == 2) x = uint64_t(1) << rng() % 3;
                    terms.push_back({x, rng() & all, nd(rng), (k & 1) ? nd(rng) : 0.0});
                }
                const size_t nt = terms.size(), most = exp_max_units(terms.data(), nt);
                std::vector<uint64_t> arena(exp_plan_bytes(nt, most) / 8 + 2);  // the exact capacity: the sanitizer sees an overrun
                ExpPlan p;
                exp_plan_carve(p, arena.data(), nt, most);
                plan_expect(n, c128 != 0, terms.data(), nt, p);
                cd want = 0;
                double scale = 0;
                for (auto &t : terms) { want += direct(psi, t); scale += std::abs(cd(t.c_re, t.c_im)); }
                cd got = planned(psi, n, p);
                size_t streamed = 0;
                for (size_t f = 0; f < p.nfar; f++)
                    for (uint32_t t = p.far_head[f]; t != UINT32_MAX; t = p.next[t]) {
                        if (terms[t].x_mask != p.far[f]) return 2;
                        got += direct(psi, terms[t]);
                        streamed++;
                    }
                int remote = 0;
                const double d = std::abs(got - want) / scale;
                const double da = c128 ? apply_error<double>(n, psi, terms, remote) : apply_error<float>(n, psi, terms, remote);
                printf("n %u c128 %d kind %d: expectation %.1e, product %.1e, units %zu of %zu, streamed terms %zu\n", n, c128, kind, d, da,
                       p.nunits, most, streamed);
                // FP64 sums of 320 terms; complex64 tables hold float coefficients
                if (!(d < 1e-13) || !(da < (c128 ? 1e-13 : 1e-6)) || p.nunits > most) return 1;
            }
    // 65536 Z supports on one mask: a fraction of a second also under the sanitizers
    std::vector<qi_pauli_term> terms;
    for (uint64_t z = 0; z < 65536; z++) terms.push_back({3, z << 4, nd(rng), 0.0});
    const size_t most = exp_max_units(terms.data(), terms.size());
    std::vector<uint64_t> arena(exp_plan_bytes(terms.size(), most) / 8 + 2);
    ExpPlan p;
    const double t0 = seconds();
    exp_plan_carve(p, arena.data(), terms.size(), most);
    plan_expect(24, true, terms.data(), terms.size(), p);
    const double t1 = seconds();
    ApplyPlan<double> a;
    plan_apply<double>(24, terms.data(), terms.size(), a);
    const double t2 = seconds();
    printf("65536 terms on one mask: planned in %.2f s, product %.2f s, units %zu\n", t1 - t0, t2 - t1, p.nunits);
    return t2 - t0 < 5.0 ? 0 : 3;
}
