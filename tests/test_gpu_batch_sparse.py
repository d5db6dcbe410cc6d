"""Batched circuits whose tiles reach the state's qubits pass by pass (or never
reach some of them): the arena is not cleared, so what a pass has not written
must read as zero, also on a second run over the first one's leavings."""
import numpy as np
import pytest

import oracle as O
import qiron
from kat_util import gates_array, random_gate, term_array

pytestmark = pytest.mark.gpu


def gates_on(qubits, count, rng):
    out = []
    for _ in range(count):
        d = random_gate(len(qubits), rng, kinds=["H", "RX", "RY", "RZ", "X"] + ["CNOT"] * (len(qubits) > 1), max_controls=0)
        d["targets"] = [qubits[q] for q in d["targets"]]
        d["controls"] = [qubits[q] for q in d["controls"]]
        out.append(d)
    return out


@pytest.mark.parametrize("prec", ["c64", "c128"])
def test_states_grow_from_zero_pass_by_pass(ctx, prec):
    rng = np.random.default_rng(5)
    circuits = []
    for n, groups in ((14, [[0, 1]]), (14, [[13]]), (15, [[2, 14], [5, 7, 9]]), (17, [list(range(0, 12)), list(range(5, 17)), [0, 16]]),
                      (19, [list(range(7, 19)), [3, 4]]), (18, [list(range(18))] * 3), (20, [list(range(0, 9)), list(range(8, 20)), list(range(20))])):
        gates = gates_array([g for q in groups for g in gates_on(q, 6 * len(q), rng)])
        masks = [(1 << i) | (1 << ((i + 1) % n)) for i in range(n)] + [0] * n + [1 << (n - 1), 1]
        terms = term_array([(x, int(rng.integers(1 << n)), float(rng.normal()), 0.0) for x in masks])
        circuits.append((n, gates, terms))
    refs = [O.expectation(O.apply_gates(O.init(n, 0), g), t) for n, g, t in circuits]
    eps = 2.0 ** -24 if prec == "c64" else 2.0 ** -53
    for order in (1, -1):  # the second batch meets other circuits' amplitudes in its arena
        b = qiron.CircuitBatch(prec)
        for n, g, t in circuits[::order]:
            b.add(n, g, t)
        for _ in range(2):
            for e, ref, (n, g, t) in zip(b.run(), refs[::order], circuits[::order]):
                # each gate: four products and sums per component, in bra and ket
                assert abs(e - ref) <= np.sum(np.abs(t["c_re"])) * (8 * g.size * eps + 1e-13), n


@pytest.mark.parametrize("prec", ["c64", "c128"])
def test_a_term_that_only_the_widest_tile_holds(ctx, prec):
    """One term of one circuit spans the widest expectation tile (13 / 12 qubits
    with the low ones): the whole batch takes that width, else one less."""
    rng = np.random.default_rng(8)
    n, low, wide = 15, 4 if prec == "c64" else 3, 13 if prec == "c64" else 12
    span = ((1 << (wide - low)) - 1) << low
    gates = gates_array(gates_on(list(range(n)), 60, rng))
    psi = O.apply_gates(O.init(n, 0), gates)
    eps = 2.0 ** -24 if prec == "c64" else 2.0 ** -53
    for masks in ([span, 3, 0], [span >> 1 & ~((1 << low) - 1), 3, 0]):
        terms = term_array([(x, int(rng.integers(1 << n)), float(rng.normal()), 0.0) for x in masks])
        b = qiron.CircuitBatch(prec)
        b.add(n, gates, terms)
        assert abs(b.run()[0] - O.expectation(psi, terms)) <= np.sum(np.abs(terms["c_re"])) * (8 * 60 * eps + 1e-13)
