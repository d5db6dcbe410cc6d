// expect_plan.cpp — host planner of expect_plan.h. Works in arrays the caller
// owns: no allocation of its own (the no-allocation entry point plans with it).
#include "expect_plan.h"

#include <algorithm>
#include <cstring>

namespace qi {

namespace {

size_t up16(size_t b) { return (b + 15) & ~size_t(15); }
int popc(uint64_t x) { return __builtin_popcountll(x); }

// The tile-local image of a qubit mask inside the tile.
uint32_t local_bits(uint64_t mask, const ExpPass &p, int K) {
    uint32_t r = 0;
    for (int k = 0; k < K; k++) r |= uint32_t((mask >> exp_pos(p.pos, k)) & 1u) << k;
    return r;
}
// The pattern of a tile-local mask on a set's register bits.
uint32_t reg_bits(uint32_t l, const ExpSet &s) {
    uint32_t r = 0;
    for (int j = 0; j < 4; j++) r |= ((l >> exp_pos(&s.pos, j)) & 1u) << j;
    return r;
}

// The qubits of a tile of K: `q`, then the masks that need the fewest new ones
// while they fit; above kGreedyMax masks simply in list order (the search is
// quadratic).
constexpr size_t kGreedyMax = 256;
template <typename F> uint64_t grow_tile(uint64_t q, size_t count, int K, F mask) {
    for (bool grown = true; grown;) {
        grown = false;
        size_t best = SIZE_MAX;
        int least = 64;
        for (size_t g = 0; g < count; g++) {
            const int add = popc(mask(g) & ~q);
            if (!add || popc(q) + add > K || add >= least) continue;
            best = g; least = add;
            if (count > kGreedyMax || add == 1) break;
        }
        if (best != SIZE_MAX) { q |= mask(best); grown = true; }
    }
    return q;
}

// Finds the entry of a list by its key: a few by looking at each, more through
// an open-addressing table, so that a list of any length is planned in linear
// time (one x mask with 16384 Z supports took 0.4 s, its product 3 s).
constexpr size_t kLookAtEach = 16;
size_t exp_table_entries(size_t nt) {
    size_t n = 1;
    while (n < 4 * nt) n <<= 1;
    return n;
}
uint64_t mix(uint64_t a, uint64_t b) {  // (multiply-xorshift, odd constants)
    uint64_t h = a * 0x9E3779B97F4A7C15ull ^ (b + 1) * 0xC2B2AE3D27D4EB4Full;
    h ^= h >> 32;
    h *= 0xD6E8FEB86659FD93ull;
    return h ^ (h >> 32);
}
struct Finder {
    uint32_t *table;
    size_t last = 0;  // table entries - 1 (0: no table)
    // Entries of at most 2 `terms` keys; `table` holds exp_table_entries(terms).
    Finder(uint32_t *table, size_t terms) : table(table) {
        if (terms <= kLookAtEach) return;
        last = exp_table_entries(terms) - 1;
        std::fill(table, table + last + 1, UINT32_MAX);
    }
    // The entry of [first, end) that is(k) accepts; `end` if none, which the caller then adds.
    template <typename F> size_t find(uint64_t hash, size_t first, size_t end, F is) {
        if (!last) {
            while (first < end && !is(first)) first++;
            return first;
        }
        for (size_t at = hash & last;; at = (at + 1) & last) {
            if (table[at] == UINT32_MAX) {
                table[at] = (uint32_t)end;
                return end;
            }
            if (is(table[at])) return table[at];
        }
    }
};

}  // namespace

size_t exp_max_units(const qi_pauli_term *terms, size_t nt) {
    size_t n = 0;
    for (size_t k = 0; k < nt; k++)
        if (terms[k].x_mask) n += (popc(terms[k].x_mask) > 4 ? 2 : 1) * (terms[k].c_im != 0.0 ? 2 : 1);
    return n;
}

size_t exp_plan_bytes(size_t nt, size_t units) {
    return up16(nt * sizeof(ExpPass)) + up16(nt * sizeof(ExpSet)) + up16((units + 1) * sizeof(ExpUnit)) +
           up16(nt * sizeof(ExpDiag)) + up16(nt * sizeof(uint64_t)) + 2 * up16(nt * sizeof(uint32_t)) +
           up16(nt * sizeof(ExpMask)) + up16(exp_table_entries(nt) * sizeof(uint32_t));
}

void exp_plan_carve(ExpPlan &p, void *arena, size_t nt, size_t units) {
    unsigned char *a = (unsigned char *)arena;
    auto take = [&](size_t bytes) { void *r = a; a += up16(bytes); return r; };
    p.passes = (ExpPass *)take(nt * sizeof(ExpPass));
    p.sets = (ExpSet *)take(nt * sizeof(ExpSet));
    p.units = (ExpUnit *)take((units + 1) * sizeof(ExpUnit));
    p.diags = (ExpDiag *)take(nt * sizeof(ExpDiag));
    p.far = (uint64_t *)take(nt * sizeof(uint64_t));
    p.far_head = (uint32_t *)take(nt * sizeof(uint32_t));
    p.next = (uint32_t *)take(nt * sizeof(uint32_t));
    p.masks = (ExpMask *)take(nt * sizeof(ExpMask));
    p.table = (uint32_t *)take(exp_table_entries(nt) * sizeof(uint32_t));
}

int exp_tile_qubits(uint32_t n, bool c128) {
    const int most = c128 ? kExpMaxK - 1 : kExpMaxK;
    return (int)n < most ? (int)n : most;
}

void plan_expect(uint32_t n, bool c128, const qi_pauli_term *terms, size_t nt, ExpPlan &p) {
    const int low = exp_low_qubits(c128);
    p.npasses = p.nsets = p.nunits = p.ndiags = p.nfar = 0;
    p.complex_out = false;
    // One or two terms of one x mask on a complex128 state that about fills the
    // last-level cache are streamed, us per call, tiles -> streamed: 24 qubits Z 83
    // -> 64, XX 77 -> 63; 22 qubits 36.6 -> 34.7. Four Z terms: 86 against 103, 25
    // qubits: 122 against 131, complex64: 54 against 64.
    bool few = c128 && n >= 22 && n <= 24 && nt <= 2;
    for (size_t k = 1; k < nt; k++) few = few && terms[k].x_mask == terms[0].x_mask;
    const bool tiles = n >= 4 && !few;
    // distinct x masks in order of appearance (the zero mask apart, where there are tiles)
    size_t nx = 0;
    ExpMask *const m = p.masks;
    bool diag = false;
    Finder by_mask(p.table, nt);
    for (size_t k = 0; k < nt; k++) {
        const uint64_t x = terms[k].x_mask;
        p.complex_out = p.complex_out || terms[k].c_im != 0.0;
        p.next[k] = UINT32_MAX;
        if (!x && tiles) { diag = true; continue; }
        const size_t g = by_mask.find(mix(x, 0), 0, nx, [&](size_t i) { return m[i].x == x; });
        if (g == nx) {
            m[nx++] = ExpMask{x, (uint32_t)k, (uint32_t)k, 1, 0};
        } else {
            p.next[m[g].tail] = (uint32_t)k;
            m[g].tail = (uint32_t)k;
            m[g].count++;
        }
    }
    const auto stream = [&](const ExpMask &x) { p.far[p.nfar] = x.x; p.far_head[p.nfar++] = x.head; };
    p.K = 0;
    if (!tiles) {
        for (size_t g = 0; g < nx; g++) stream(m[g]);
        return;
    }
    // A complex64 state of more qubits than its widest tile takes tiles of one
    // qubit less, unless a mask needs that one: at half the LDS, four
    // workgroups per CU load and compute out of step instead of two. Tiles of 13
    // -> 12 qubits: 28 qubits, 4 x 7 lattice 4.45 -> 4.01 ms; 24-qubit chain 216 ->
    // 189 us; 29-qubit chain 6.07 -> 5.63 ms (11 qubits: 4.49 ms, 200 us, 5.95 ms;
    // complex128 with 11 instead of 12: 3.03 -> 3.25 ms at 27 qubits).
    int K = exp_tile_qubits(n, c128);
    const bool whole = (int)n == K;
    const uint64_t lowmask = whole ? (uint64_t(1) << n) - 1 : (uint64_t(1) << low) - 1;
    if (!c128 && !whole) {
        K--;
        for (size_t g = 0; g < nx; g++)
            if (popc(m[g].x | lowmask) == K + 1) { K++; break; }
    }
    p.K = K;
    // masks that no tile holds go to the streaming kernel
    size_t nleft = 0;
    for (size_t g = 0; g < nx; g++) {
        if (popc(m[g].x | lowmask) > K) stream(m[g]);
        else m[nleft++] = m[g];
    }
    bool diag_todo = diag;
    size_t at = 0;  // masks [at, nleft) are unplanned; a pass moves its masks to the front
    while (at < nleft || diag_todo) {
        ExpPass &ps = p.passes[p.npasses++];
        memset(&ps, 0, sizeof ps);
        uint64_t q = grow_tile(lowmask, nleft - at, K, [&](size_t g) { return m[at + g].x; });
        for (uint32_t b = 0; b < n && popc(q) < K; b++) q |= uint64_t(1) << b;
        ps.qmask = q;
        for (int k = 0, b = 0; k < K; b++)
            if ((q >> b) & 1) { ps.pos[k >> 2] |= (uint32_t)b << (8 * (k & 3)); k++; }
        ps.s0 = (uint32_t)p.nsets;
        const size_t first = at;
        for (size_t g = at; g < nleft; g++)
            if (!(m[g].x & ~q)) {
                std::swap(m[g], m[at]);
                m[at].xl = local_bits(m[at].x, ps, K);
                at++;
            }
        // register sets over this pass's masks [first, at)
        bool pass_diag = diag_todo;
        diag_todo = false;
        size_t s_at = first;
        while (s_at < at || pass_diag) {
            ExpSet &st = p.sets[p.nsets++];
            memset(&st, 0, sizeof st);
            uint32_t r = 0;
            for (bool grown = true; grown;) {
                grown = false;
                size_t best = SIZE_MAX;
                int least = 64;
                for (size_t g = s_at; g < at; g++) {
                    const int add = popc(m[g].xl & ~r);
                    if (!add || popc(r) + add > 4 || add >= least) continue;
                    best = g; least = add;
                    if (at - s_at > kGreedyMax || add == 1) break;
                }
                if (best != SIZE_MAX) { r |= m[best].xl; grown = true; }
            }
            for (int b = K - 1; b >= 0 && popc(r) < 4; b--) r |= 1u << b;
            for (int j = 0, b = 0; j < 4; b++)
                if ((r >> b) & 1) st.pos |= (uint32_t)b << (8 * j++);
            st.u0 = (uint32_t)p.nunits;
            // the masks inside the set, and (with no set of their own) the ones of more than four bits
            for (size_t g = s_at; g < at; g++) {
                const uint32_t xl = m[g].xl;
                const bool wide = popc(xl) > 4;
                if (!wide && (xl & ~r)) continue;
                const uint32_t xm = wide ? 0 : reg_bits(xl, st);
                const int pivot = xm ? 31 - __builtin_clz(xm) : -1;
                // one run of units per u: Re w or Im w, and for wide masks the two halves of the slots
                for (int run = 0; run < (wide ? 4 : 2); run++) {
                    const int im_w = run & 1, high = run >> 1;
                    const size_t e0 = p.nunits;
                    Finder by_signs(p.table, m[g].count);
                    for (uint32_t t = m[g].head; t != UINT32_MAX; t = p.next[t]) {
                        const qi_pauli_term &tm = terms[t];
                        const int ny = popc(tm.x_mask & tm.z_mask);
                        if ((ny & 1) != im_w) continue;
                        // phi(i) = (-i)^ny (-1)^{popcount(i & z)}: Re(phi w) is s Re w (ny 0: s = 1, ny 2: -1)
                        // or s Im w (ny 1: phi = -i, s = 1; ny 3: phi = i, s = -1)
                        const double s0 = (ny & 3) < 2 ? 1.0 : -1.0;
                        const uint32_t zl = local_bits(tm.z_mask, ps, K), zr = reg_bits(zl, st);
                        for (int part = 0; part < 2; part++) {
                            const double c = part ? tm.c_im : tm.c_re;
                            if (part && c == 0.0) continue;
                            const uint64_t zo = tm.z_mask & ~q;
                            const uint32_t fl = part ? kExpImag : 0u;
                            const size_t e = by_signs.find(mix(zo, uint64_t(zl & ~r) << 1 | part), e0, p.nunits, [&](size_t u) {
                                return p.units[u].zo == zo && p.units[u].zl == (zl & ~r) && (p.units[u].flags() & kExpImag) == fl;
                            });
                            ExpUnit &un = p.units[e];
                            if (e == p.nunits) {
                                memset(&un, 0, sizeof un);
                                un.zo = zo; un.zl = zl & ~r;
                                un.info = (xm + 16u * im_w) | xl << 16 |
                                          (fl | (e > e0 ? kExpReuse : 0u) | (high ? kExpHigh : 0u)) << 8;
                                p.nunits++;
                            }
                            // a pair is visited once (factor 2); a wide mask visits both its members
                            const double f = (xm ? 2.0 : 1.0) * s0 * c;
                            for (uint32_t k = 0; k < 8; k++) {
                                const uint32_t slot =
                                    xm ? ((k >> pivot) << (pivot + 1)) | (k & ((1u << pivot) - 1)) : k + 8u * high;
                                un.h[k] += (popc(slot & zr) & 1) ? -f : f;
                            }
                        }
                    }
                }
                std::swap(m[g], m[s_at]);
                s_at++;
            }
            st.nu = (uint32_t)p.nunits - st.u0;
            if (pass_diag) {  // counting sort by register-bit pattern
                pass_diag = false;
                st.diag = 1;
                uint32_t cnt[kExpSlots + 1] = {0};
                for (size_t k = 0; k < nt; k++)
                    if (!terms[k].x_mask) cnt[reg_bits(local_bits(terms[k].z_mask, ps, K), st) + 1]++;
                for (int b = 0; b < kExpSlots; b++) cnt[b + 1] += cnt[b];
                memcpy(st.doff, cnt, sizeof cnt);
                for (size_t k = 0; k < nt; k++) {
                    if (terms[k].x_mask) continue;
                    const uint32_t zl = local_bits(terms[k].z_mask, ps, K);
                    ExpDiag &d = p.diags[cnt[reg_bits(zl, st)]++];
                    d.zo = terms[k].z_mask & ~q; d.zl = zl & ~r; d.pad = 0;
                    d.re = terms[k].c_re; d.im = terms[k].c_im;
                    p.ndiags++;
                }
            }
        }
        ps.ns = (uint32_t)p.nsets - ps.s0;
    }
    memset(&p.units[p.nunits], 0, sizeof(ExpUnit));
}

// A pass reads and writes the result as well as the input, a remote mask reads
// the input once more: passes of fewer masks than this are not worth it.
constexpr size_t kApplyPassMasks = 3;

bool apply_as_gathers(uint32_t n, bool c128, const qi_pauli_term *terms, size_t nt) {
    if (nt > (c128 ? 4u : 3u)) return false;
    const uint64_t lowmask = (uint64_t(1) << exp_low_qubits(c128)) - 1;
    for (size_t k = 0; k < nt; k++)
        if (!terms[k].x_mask || popc(terms[k].x_mask | lowmask) <= exp_tile_qubits(n, c128)) return false;
    return true;
}

template <typename R> void plan_apply(uint32_t n, const qi_pauli_term *terms, size_t nt, ApplyPlan<R> &p) {
    const bool c128 = sizeof(R) == 8;
    const int K = exp_tile_qubits(n, c128);
    p.K = K;
    const bool whole = (int)n == K;
    const uint64_t lowmask = whole ? (uint64_t(1) << n) - 1 : (uint64_t(1) << exp_low_qubits(c128)) - 1;
    std::vector<ExpMask> m;  // the distinct masks and their terms, as in plan_expect
    std::vector<uint32_t> next(nt, UINT32_MAX), table(exp_table_entries(nt)), unit_of(nt);
    bool diag = false;
    Finder by_mask(table.data(), nt);
    for (size_t k = 0; k < nt; k++) {
        const uint64_t x = terms[k].x_mask;
        if (!x) { diag = true; continue; }
        const size_t g = by_mask.find(mix(x, 0), 0, m.size(), [&](size_t i) { return m[i].x == x; });
        if (g == m.size()) {
            m.push_back(ExpMask{x, (uint32_t)k, (uint32_t)k, 1, 0});
        } else {
            next[m[g].tail] = (uint32_t)k;
            m[g].tail = (uint32_t)k;
            m[g].count++;
        }
    }
    const uint32_t slots = apply_slots(K, c128);
    constexpr int SB = apply_slot_bits(sizeof(R) == 8), NS = 1 << SB;
    uint32_t sm = 0;
    for (int j = 0; j < SB; j++) sm |= 1u << exp_pos(&slots, j);
    auto slot_bits = [&](uint32_t l) {
        uint32_t r = 0;
        for (int j = 0; j < SB; j++) r |= ((l >> exp_pos(&slots, j)) & 1u) << j;
        return r;
    };
    std::vector<std::vector<ExpMask>> local;  // the masks of each pass; the rest (left) are remote
    std::vector<uint64_t> tiles;
    std::vector<ExpMask> left = m;
    for (;;) {
        const uint64_t q0 = grow_tile(lowmask, left.size(), K, [&](size_t g) { return left[g].x; });
        std::vector<ExpMask> in, out;
        for (const ExpMask &x : left) ((x.x & ~q0) ? out : in).push_back(x);
        if (!tiles.empty() && in.size() < kApplyPassMasks) break;
        uint64_t q = q0;
        for (uint32_t b = 0; b < n && popc(q) < K; b++) q |= uint64_t(1) << b;
        tiles.push_back(q);
        local.push_back(in);
        left = out;
        if (left.empty()) break;
    }
    std::vector<double> sums;  // a mask's coefficients: per unit, real then imaginary parts
    for (size_t ip = 0; ip < tiles.size(); ip++) {
        const uint64_t q = tiles[ip];
        ExpPass ps{};  // positions for local_bits
        ps.qmask = q;
        for (int k = 0, b = 0; k < K; b++)
            if ((q >> b) & 1) { ps.pos[k >> 2] |= (uint32_t)b << (8 * (k & 3)); k++; }
        ApplyPass pass{};
        pass.qmask = q;
        memcpy(pass.pos, ps.pos, sizeof ps.pos);
        pass.u0 = (uint32_t)p.units.size();
        const bool last = ip + 1 == tiles.size();  // takes the remote masks
        const size_t nlocal = local[ip].size(), total = nlocal + (last ? left.size() : 0);
        for (size_t g = 0; g < total; g++) {
            const bool remote = g >= nlocal;
            const ExpMask &mask = remote ? left[g - nlocal] : local[ip][g];
            const size_t e0 = p.units.size();
            // the mask's units, and the one of each of its terms
            Finder by_signs(table.data(), mask.count);
            for (uint32_t t = mask.head; t != UINT32_MAX; t = next[t]) {
                const uint32_t zl = local_bits(terms[t].z_mask, ps, K) & ~sm;
                const uint64_t zo = terms[t].z_mask & ~q;
                const size_t e = by_signs.find(mix(zo, zl), e0, p.units.size(),
                                               [&](size_t u) { return p.units[u].zo == zo && p.units[u].zl == zl; });
                if (e == p.units.size()) {
                    ApplyUnit<R> un{};
                    un.zo = zo; un.x = mask.x; un.zl = zl;
                    un.xl = remote ? 0 : local_bits(mask.x, ps, K);
                    un.flags = remote ? (uint32_t)kApplyRemote : 0u;
                    p.units.push_back(un);
                }
                unit_of[t] = (uint32_t)(e - e0);
            }
            // the units' coefficients, summed in FP64: c (-i)^ny (-1)^{popcount(slot & z)}
            sums.assign(2 * NS * (p.units.size() - e0), 0.0);
            for (uint32_t t = mask.head; t != UINT32_MAX; t = next[t]) {
                const qi_pauli_term &tm = terms[t];
                const uint32_t zr = slot_bits(local_bits(tm.z_mask, ps, K));
                double *const hr = sums.data() + 2 * NS * unit_of[t], *const hi = hr + NS;
                double cr = tm.c_re, ci = tm.c_im, r;
                switch (popc(tm.x_mask & tm.z_mask) & 3) {
                case 1: r = cr; cr = ci; ci = -r; break;   // times -i
                case 2: cr = -cr; ci = -ci; break;
                case 3: r = cr; cr = -ci; ci = r; break;   // times i
                default: break;
                }
                for (uint32_t s = 0; s < (uint32_t)NS; s++) {
                    const bool odd = popc(s & zr) & 1;
                    hr[s] += odd ? -cr : cr;
                    hi[s] += odd ? -ci : ci;
                }
            }
            for (size_t e = e0; e < p.units.size(); e++) {
                ApplyUnit<R> &un = p.units[e];
                const double *const hr = sums.data() + 2 * NS * (e - e0), *const hi = hr + NS;
                for (int s = 0; s < NS; s++) {
                    un.re[s] = (R)hr[s];
                    un.im[s] = (R)hi[s];
                    if (hr[s] != 0.0) un.flags |= kApplyRe;
                    if (hi[s] != 0.0) un.flags |= kApplyIm;
                }
                if (!(un.flags & (kApplyRe | kApplyIm))) un.flags |= kApplyRe;  // zero times NaN stays NaN
            }
        }
        pass.nu = (uint32_t)p.units.size() - pass.u0;
        if (ip == 0 && diag) {
            pass.diag = 1;
            uint32_t cnt[kExpSlots + 1] = {0};
            for (size_t k = 0; k < nt; k++)
                if (!terms[k].x_mask) cnt[slot_bits(local_bits(terms[k].z_mask, ps, K)) + 1]++;
            for (int b = 0; b < kExpSlots; b++) cnt[b + 1] += cnt[b];
            memcpy(pass.doff, cnt, sizeof cnt);
            p.diags.resize(cnt[kExpSlots]);
            for (size_t k = 0; k < nt; k++) {
                if (terms[k].x_mask) continue;
                const uint32_t zl = local_bits(terms[k].z_mask, ps, K);
                ExpDiag &d = p.diags[cnt[slot_bits(zl)]++];
                d.zo = terms[k].z_mask & ~q; d.zl = zl & ~sm; d.pad = 0;
                d.re = terms[k].c_re; d.im = terms[k].c_im;
                p.complex_diag = p.complex_diag || d.im != 0.0;
            }
        }
        p.passes.push_back(pass);
    }
}
template void plan_apply<float>(uint32_t, const qi_pauli_term *, size_t, ApplyPlan<float> &);
template void plan_apply<double>(uint32_t, const qi_pauli_term *, size_t, ApplyPlan<double> &);

}  // namespace qi
