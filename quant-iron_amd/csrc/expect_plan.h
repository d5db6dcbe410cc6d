// expect_plan.h — how the expectation of a SumOp is cut into tile passes
// (planned on the host in expect_plan.cpp, run by expect.hip), and a SumOp's
// product with a state on the same tiles.
//
// A tile is the 2^K amplitudes spanned by a set of K qubits. A term whose X
// and Y factors lie inside that set needs only amplitudes of one tile, so one
// read of the state serves every such term, whatever its Z factors. Inside a
// tile the terms with one x mask are a group: P is Hermitian, so the pair
// (i, i ^ x) adds c 2 Re(phi(i) conj(psi_i) psi_{i^x}) with phi(i) a sign or a
// sign times i, and a group's terms share Re w or Im w of each pair.
// A register set is four tile qubits whose 16 amplitudes one thread holds:
// groups inside a set cost no memory traffic.
#pragma once

#include <cstddef>
#include <cstdint>
#include <vector>

#include "../../include/qiron.h"

#ifdef __HIP__
#define QI_HD __host__ __device__
#else
#define QI_HD
#endif

namespace qi {

constexpr int kExpSlots = 16;     // amplitudes per thread: four register bits
constexpr int kExpMaxK = 13;      // tile qubits at most

// One step of a register set: the signed coefficients of one x mask's terms
// that share a Z support outside the register bits and the parity of their
// number of Y factors: adds sign * sum_k h[k] u[k] over the 8 pairs of the
// mask (slots with its highest bit clear), u = Re w or Im w. A mask of more
// than four tile bits ("wide") visits both members of each pair, partners
// read from LDS, in two units of 8 slots.
struct ExpUnit {
    uint64_t zo;      // Z bits outside the tile
    uint32_t zl;      // Z bits inside the tile, outside the register bits (tile-local)
    uint32_t info;    // (dword fields: the kernel reads its tables with scalar loads) byte 0: register-bit pattern
                      // of the mask (1..15), 0: wide; + 16: u = Im w (odd number of Y factors); byte 1: flags
                      // below; bits 16-31: the mask in tile-local bits
    double h[8];
    QI_HD uint32_t code() const { return info & 31u; }
    QI_HD uint32_t flags() const { return (info >> 8) & 255u; }
    QI_HD uint32_t xl() const { return info >> 16; }
};
enum : uint32_t {
    kExpReuse = 1,    // the unit before has the same u
    kExpImag = 2,     // adds to the imaginary part (imaginary parts of the coefficients)
    kExpHigh = 4,     // wide: slots 8..15 (else 0..7)
};
// One diagonal term (x = 0): c (-1)^{popcount(i & z)} |psi_i|^2.
struct ExpDiag {
    uint64_t zo;
    uint32_t zl;
    uint32_t pad;
    double re, im;
};
struct ExpSet {
    uint32_t pos;       // tile-local positions of the four register bits, ascending, a byte each
    uint32_t u0, nu;    // units
    uint32_t diag;      // 1: the diagonal terms run here, sorted by their register-bit pattern
    uint32_t doff[kExpSlots + 1];
};
struct ExpPass {
    uint64_t qmask;     // tile qubits
    uint32_t s0, ns;    // register sets
    uint32_t pos[4];    // qubit of each tile-local bit, ascending, a byte each
};
// Byte k of a packed position list.
QI_HD inline uint32_t exp_pos(const uint32_t *p, int k) { return (p[k >> 2] >> (8 * (k & 3))) & 255u; }

// The distinct x masks of a term list, each with its terms as a list in order.
struct ExpMask {
    uint64_t x;
    uint32_t head, tail, count;  // terms: the first, the last (linked by ExpPlan::next), how many
    uint32_t xl;                 // tile-local bits in the mask's pass
};
// The plan, in arrays the caller owns (capacities for nt terms below).
struct ExpPlan {
    ExpPass *passes;    // <= nt
    ExpSet *sets;       // <= nt
    ExpUnit *units;     // <= exp_max_units + 1 (one spare: the kernel reads a unit ahead)
    ExpDiag *diags;     // <= nt
    uint64_t *far;      // x masks that no tile can hold: <= nt
    uint32_t *far_head; // and the first term of each
    ExpMask *masks;     // scratch: <= nt
    uint32_t *next;     // the next term of the same mask, UINT32_MAX: none
    uint32_t *table;    // scratch: exp_table_entries(nt)
    size_t npasses, nsets, nunits, ndiags, nfar;
    int K;              // tile qubits (0: no tiles, every mask is streamed)
    bool complex_out;   // an imaginary part can be nonzero
};
// Units that a term list can take at most: one per mask and Z support, two for
// masks of more than four qubits, again as many for imaginary coefficients.
size_t exp_max_units(const qi_pauli_term *terms, size_t nt);
// Bytes of the planning arena for nt terms of at most `units` units (any nt
// terms without it).
size_t exp_plan_bytes(size_t nt, size_t units);
inline size_t exp_plan_bytes(size_t nt) { return exp_plan_bytes(nt, 4 * nt); }
// Carves the arrays out of `arena` (exp_plan_bytes bytes, 16-byte aligned).
void exp_plan_carve(ExpPlan &p, void *arena, size_t nt, size_t units);
inline void exp_plan_carve(ExpPlan &p, void *arena, size_t nt) { exp_plan_carve(p, arena, nt, 4 * nt); }
// Widest tile for n qubits (n >= 4): the whole state, at most 13 (complex64) or
// 12 (complex128) qubits of it.
int exp_tile_qubits(uint32_t n, bool c128);
// Qubits 0 .. low-1 are always in a tile: 128-byte runs in memory.
inline int exp_low_qubits(bool c128) { return c128 ? 3 : 4; }
// Without tiles (fewer than 4 qubits, a term or two) every mask is streamed.
void plan_expect(uint32_t n, bool c128, const qi_pauli_term *terms, size_t nt, ExpPlan &p);

// ---- SumOp::apply on the same tiles ----
// A thread owns 16 (complex64) or 8 (complex128) amplitudes of the result
// (slots: the tile-local bits of apply_slots) and adds, per unit, sign * h[slot] * in[i ^ x]: one unit per x
// mask and Z support outside the slot bits. The partner comes from the tile in
// LDS, or from memory for masks the pass's tile does not hold ("remote").
constexpr int apply_slot_bits(bool c128) { return c128 ? 3 : 4; }
template <typename R> struct ApplyUnit {
    uint64_t zo;     // Z bits outside the tile
    uint64_t x;      // the mask
    uint32_t zl;     // Z bits inside the tile, outside the slot bits (tile-local)
    uint32_t xl;     // the mask in tile-local bits (not remote)
    uint32_t flags;  // kApplyRe | kApplyIm | kApplyRemote
    uint32_t pad;
    static constexpr int slots = 1 << apply_slot_bits(sizeof(R) == 8);
    R re[slots], im[slots];
};
enum : uint32_t { kApplyRe = 1, kApplyIm = 2, kApplyRemote = 4 };
struct ApplyPass {
    uint64_t qmask;
    uint32_t u0, nu;
    uint32_t pos[4];     // as ExpPass
    uint32_t diag;       // 1: the diagonal terms run here
    uint32_t doff[kExpSlots + 1];
};
template <typename R> struct ApplyPlan {
    int K = 0;
    std::vector<ApplyPass> passes;
    std::vector<ApplyUnit<R>> units;
    std::vector<ExpDiag> diags;  // sorted by slot-bit pattern
    bool complex_diag = false;   // a diagonal coefficient has an imaginary part
};
// Tile-local positions of the slot bits, ascending, a byte each: the bits a
// thread's loads step over (complex64: bit 0 inside a 16-byte unit, then the top three).
inline uint32_t apply_slots(int K, bool c128) {
    const uint32_t k = (uint32_t)K;
    return c128 ? (k - 3) | (k - 2) << 8 | (k - 1) << 16 : 0u | (k - 3) << 8 | (k - 2) << 16 | (k - 1) << 24;
}
// Whether a product is a few terms whose x masks no tile holds: a tile's copy in
// LDS would be read for nothing, so that each term is cheaper as a gather. 27
// qubits, us, tile passes -> gathers: 1 term 577 -> 380 (complex64), 1185 -> 869
// (complex128); 2 terms 577 -> 476 and 1161 -> 851; 4 terms 602 -> 760 and 1109 ->
// 1024; 3 random terms on 28 qubits in complex64 1912 -> 1602 (complex128 with 8
// terms: between 1.22 and 0.86 times).
bool apply_as_gathers(uint32_t n, bool c128, const qi_pauli_term *terms, size_t nt);
template <typename R> void plan_apply(uint32_t n, const qi_pauli_term *terms, size_t nt, ApplyPlan<R> &p);

}  // namespace qi
