"""SumOps of many x masks too wide for a tile: every mask streams the state, all
in one launch. Against the oracle where a mask takes all its blocks and where
many share the launch, and no slower per mask than a list of one."""
import time

import numpy as np
import pytest

import oracle as O
import qiron
from kat_util import random_state, term_array

pytestmark = pytest.mark.gpu


def wide_terms(n, masks, per_mask, rng):
    """Strings with X or Y on all but one or two qubits of n, more than a tile of 13 holds."""
    rows, full, seen = [], (1 << n) - 1, set()
    while len(seen) < masks:
        seen.add(full & ~(1 << int(rng.integers(n))) & ~(1 << int(rng.integers(n))))
    for x in sorted(seen):
        rows += [(x, int(rng.integers(full + 1)), float(rng.normal()), float(rng.normal())) for _ in range(per_mask)]
    return term_array([rows[i] for i in rng.permutation(len(rows))])


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("n,masks,per_mask", [(16, 1, 3), (16, 70, 2), (18, 120, 1)])
def test_many_wide_masks_match_the_oracle(ctx, prec, n, masks, per_mask):
    rng = np.random.default_rng([n, masks])
    psi = random_state(n, rng)
    if prec == "c64":
        psi = psi.astype(np.complex64).astype(np.complex128)
    s = qiron.State.from_vector_unchecked(psi, prec)
    terms = wide_terms(n, masks, per_mask, rng)
    # every |<P>| <= 1 and each product, sign and sum is FP64 on both sides: 1e-12 of the coefficients' sum
    tol = 1e-12 * float(np.sum(np.hypot(terms["c_re"], terms["c_im"])))
    assert abs(qiron.expectation_terms(s, terms) - O.expectation(psi, terms)) <= tol


def test_a_list_of_wide_masks_costs_no_more_per_mask_than_one(ctx):
    n, masks = 24, 100
    s = qiron.State.new_plus(n, "c64", ctx)
    many = wide_terms(n, masks, 1, np.random.default_rng(1))

    def seconds(terms):
        best = np.inf
        for _ in range(5):
            t = time.perf_counter()
            qiron.expectation_terms(s, terms)
            best = min(best, time.perf_counter() - t)
        return best

    one = np.ascontiguousarray(many[:1])
    seconds(one), seconds(many)  # buffers and tables are there
    assert seconds(many) < 2 * masks * seconds(one)
