"""Tile passes whose ops act across lanes: gates concentrated on the low
qubits (held on lanes when a pass loads and stores), so that one-wave passes
take every lane bit as a pair target, exchange lane and register bits, and
swap register pairs under lane controls; against the CPU oracle."""
import numpy as np
import pytest

import oracle as O
import qiron
from kat_util import gates_array, random_state, random_unitary2
from qiron import _lib as L

pytestmark = pytest.mark.gpu

N = 13
KINDS = ["X", "Y", "H", "RX", "RY", "U2", "Z", "RZ", "P", "CX", "CZ", "CCX", "CRX"]


def low_gates(rng, count):
    """Gates with targets (and half the controls) mostly among qubits 0-5."""
    out = []
    for _ in range(count):
        k = KINDS[rng.integers(len(KINDS))]
        order = [int(q) for q in rng.permutation(6)] + [int(q) for q in 6 + rng.permutation(N - 6)]
        t = order[0] if rng.random() < 0.75 else order[-1]
        rest = [q for q in order if q != t]
        if rng.random() < 0.5:
            rest = rest[::-1]
        kind = {"CX": "X", "CZ": "Z", "CCX": "X", "CRX": "RX"}.get(k, k)
        d = {"kind": kind, "params": [float(rng.uniform(0, 2 * np.pi)) for _ in range(3)], "targets": [t],
             "controls": rest[:{"CX": 1, "CZ": 1, "CRX": 1, "CCX": 2}.get(k, 0)]}
        if kind == "U2":
            d["matrix"] = [[z.real, z.imag] for z in random_unitary2(rng).reshape(-1)]
        out.append(d)
    return gates_array(out)


# every gate is at most four products and sums per component of a unit-norm
# state: gates * 4 ulps of 1
@pytest.mark.parametrize("prec,K", [("c64", 10), ("c64", 11), ("c64", 12), ("c128", 10), ("c128", 11), ("c64", 13), ("c128", 12)])
@pytest.mark.parametrize("seed", [1, 2, 3])
def test_low_qubit_gates_match_the_oracle(ctx, prec, K, seed):
    rng = np.random.default_rng([seed, K])
    gates = low_gates(rng, 150)
    psi = random_state(N, rng)
    s = qiron.State.from_vector_unchecked(psi, prec)
    s.apply_gates_inplace(gates, mode=L.EXEC_TILED, tile_qubits=K)
    tol = 150 * 4 * (2.0 ** -24 if prec == "c64" else 2.0 ** -53)
    assert np.max(np.abs(s.state_vector - O.apply_gates(psi, gates))) <= tol


# two registers per thread (one register bit): the smallest tile that the
# options accept, in both precisions
@pytest.mark.parametrize("prec,threads", [("c64", 9), ("c128", 9), ("c64", 8)])
@pytest.mark.parametrize("seed", [1, 2])
def test_tiles_of_few_registers_match_the_oracle(ctx, prec, threads, seed):
    rng = np.random.default_rng([seed, threads, 40])
    gates = low_gates(rng, 150)
    cnots = [{"kind": "X", "targets": [t], "controls": [c]} for c in range(N) for t in range(6) if c != t]
    turns = [{"kind": k, "targets": [q], "params": [float(rng.uniform(0, 2 * np.pi))]} for q in range(N) for k in ("RX", "RY")]
    more = cnots + turns
    gates = np.concatenate([gates, gates_array([more[i] for i in rng.permutation(len(more))])])
    psi = random_state(N, rng)
    s = qiron.State.from_vector_unchecked(psi, prec)
    s.apply_gates_inplace(gates, mode=L.EXEC_TILED, tile_qubits=10, tile_threads_log2=threads)
    tol = gates.size * 4 * (2.0 ** -24 if prec == "c64" else 2.0 ** -53)
    assert np.max(np.abs(s.state_vector - O.apply_gates(psi, gates))) <= tol
