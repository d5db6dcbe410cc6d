// Which term lists go to tile passes and which are streamed, on both sides of
// each limit in expect_plan.cpp. Exit code 0 when all agree.
#include <cstdio>
#include <vector>

#include "../../quant-iron_amd/csrc/expect_plan.h"

using namespace qi;

static int wrong = 0;
static void streamed(const char *what, uint32_t n, bool c128, const std::vector<qi_pauli_term> &t, bool want) {
    std::vector<uint64_t> arena(exp_plan_bytes(t.size()) / 8 + 2);
    ExpPlan p;
    exp_plan_carve(p, arena.data(), t.size());
    plan_expect(n, c128, t.data(), t.size(), p);
    size_t listed = 0;
    for (size_t f = 0; f < p.nfar; f++)
        for (uint32_t k = p.far_head[f]; k != UINT32_MAX; k = p.next[k]) listed += t[k].x_mask == p.far[f];
    const bool all = p.npasses == 0 && listed == t.size(), none = p.nfar == 0 && p.npasses > 0;
    if (!(want ? all : none)) {
        printf("%s: %u qubits, %zu terms: %zu passes, %zu streamed\n", what, n, t.size(), p.npasses, listed);
        wrong = 1;
    }
}

int main() {
    const qi_pauli_term z{0, 1 << 9, 0.5, 0.0}, zz{0, 3 << 4, 0.25, 1.0}, xx{3 << 5, 0, 0.5, 0.0}, xy{3 << 5, 1 << 5, 0.5, 0.0};
    for (uint32_t n : {10u, 12u, 21u, 22u, 23u, 24u, 25u, 30u})
        for (int c128 = 0; c128 < 2; c128++) {
            const bool few = c128 && n >= 22 && n <= 24;
            streamed("Z", n, c128, {z}, few);
            streamed("X X", n, c128, {xx}, few);
            streamed("two of one mask", n, c128, {xx, xy}, few);
            streamed("two diagonal", n, c128, {z, zz}, few);
            streamed("two masks", n, c128, {xx, z}, false);
            streamed("three terms", n, c128, {z, zz, z}, false);
        }
    for (uint32_t n : {1u, 2u, 3u}) streamed("no tiles", n, true, {{0, 1, 0.5, 0.0}, {1, 1, 0.5, 0.0}, {0, 1, 0.5, 0.0}}, true);
    // products: few terms, all wider than a tile (13 qubits in complex64, 12 in complex128, the low ones among them)
    for (int c128 = 0; c128 < 2; c128++) {
        const uint64_t full = (1 << 22) - 1, wide = full & ~uint64_t(0xff0), fits = c128 ? 0xff8 : 0x1ff0;
        const size_t most = c128 ? 4 : 3;
        for (size_t count = 1; count <= 5; count++) {
            std::vector<qi_pauli_term> t(count, {wide, 3, 0.5, 0.0});
            if (apply_as_gathers(22, c128, t.data(), count) != (count <= most)) wrong = 2;
            t.back().x_mask = fits;  // one mask a tile holds, or a diagonal term
            if (apply_as_gathers(22, c128, t.data(), count)) wrong = 3;
            t.back().x_mask = 0;
            if (apply_as_gathers(22, c128, t.data(), count)) wrong = 4;
        }
    }
    return wrong;
}
