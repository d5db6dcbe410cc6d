"""SumOp expectations and products on the GPU against the oracle at the edges of
the tile passes: states below, at and above a tile, masks wider than a register set and
wider than a tile."""
import numpy as np
import pytest

import oracle as O
import qiron
from kat_util import random_state, random_terms, term_array
from qiron import workloads as W

pytestmark = pytest.mark.gpu


def close(state, psi, terms):
    # every |<P>| <= 1 and each product, sign and sum is FP64 on both sides: 1e-12 of the coefficients' sum
    tol = 1e-12 * float(np.sum(np.hypot(terms["c_re"], terms["c_im"])))
    assert abs(qiron.expectation_terms(state, terms) - O.expectation(psi, terms)) <= tol


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 9, 12, 13, 14, 17])
def test_expectation_matches_oracle(ctx, n, prec):
    rng = np.random.default_rng(100 + n)
    psi = random_state(n, rng)
    if prec == "c64":
        psi = psi.astype(np.complex64).astype(np.complex128)  # the amplitudes the state holds
    s = qiron.State.from_vector_unchecked(psi, prec)
    if n > 1:
        close(s, psi, W.heisenberg_open_1d(n, 0.9, 1.1, 0.7, rng.normal(size=n)))
    close(s, psi, random_terms(n, 40, rng, max_weight=n))
    everywhere = (1 << n) - 1  # X (and Y) on every qubit, Z on every qubit, and a diagonal list
    close(s, psi, term_array([(everywhere, 0, 0.3, 0.1), (everywhere, 1, -0.2, 0.0), (0, everywhere, 0.5, 0.25)]))
    close(s, psi, term_array([(0, int(rng.integers(everywhere + 1)), float(rng.normal()), 0.0) for _ in range(30)]))


def same_product(state, psi, terms, prec):
    out = qiron.SumOp([qiron.PauliString(complex(t["c_re"], t["c_im"]), ops(t)) for t in terms]).apply(state).state_vector
    # amplitudes are at most 1 and each term adds a product and a sum: a few roundings of the coefficients' sum
    scale = float(np.sum(np.hypot(terms["c_re"], terms["c_im"])))
    assert np.max(np.abs(out - O.sumop_apply(psi, terms))) <= (1e-14 if prec == "c128" else 2e-6) * scale


def ops(t):
    x, z = int(t["x_mask"]), int(t["z_mask"])
    return {q: "XZY"[(x >> q & 1) + 2 * (z >> q & 1) - 1] for q in range(64) if (x | z) >> q & 1}


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("n", [1, 5, 20, 21, 22])
def test_sumop_apply_matches_oracle(ctx, n, prec):
    rng = np.random.default_rng(700 + n)
    psi = random_state(n, rng)
    if prec == "c64":
        psi = psi.astype(np.complex64).astype(np.complex128)
    s = qiron.State.from_vector_unchecked(psi, prec)
    if n > 1:
        same_product(s, psi, W.heisenberg_open_1d(n, 0.9, 1.1, 0.7, rng.normal(size=n)), prec)
    same_product(s, psi, random_terms(n, 40, rng, max_weight=n), prec)
    everywhere = (1 << n) - 1
    same_product(s, psi, term_array([(everywhere, 0, 0.3, 0.1), (everywhere, 1, -0.2, 0.0), (0, everywhere, 0.5, 0.25)]), prec)
    same_product(s, psi, term_array([(0, int(rng.integers(everywhere + 1)), float(rng.normal()), 0.0) for _ in range(30)]), prec)
