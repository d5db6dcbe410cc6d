"""Products of one to six terms whose x masks no tile holds: up to a few of them
run as gathers in the reference's order, in complex128 to the bit; more run in
tile passes."""
import numpy as np
import pytest

import oracle as O
import qiron
from kat_util import random_state, term_array

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("n", [20, 21, 22])
def test_products_of_a_few_wide_terms(ctx, n, prec):
    rng = np.random.default_rng([n, 3])
    psi = random_state(n, rng)
    if prec == "c64":
        psi = psi.astype(np.complex64).astype(np.complex128)
    s = qiron.State.from_vector_unchecked(psi, prec)
    full = (1 << n) - 1
    for count in range(1, 7):
        rows = [(full & ~(1 << k), int(rng.integers(full + 1)), float(rng.normal()), float(rng.normal())) for k in range(count)]
        terms = term_array(rows)
        ops = [{q: "XZY"[(x >> q & 1) + 2 * (z >> q & 1) - 1] for q in range(n) if (x | z) >> q & 1} for x, z, _r, _i in rows]
        out = qiron.SumOp([qiron.PauliString(complex(r, i), o) for (_x, _z, r, i), o in zip(rows, ops)]).apply(s).state_vector
        want = O.sumop_apply(psi, terms)
        if prec == "c128" and count <= 4:
            np.testing.assert_array_equal(out, want)
        # amplitudes are at most 1 and each term adds a product and a sum: a few roundings of the coefficients' sum
        scale = float(np.sum(np.hypot(terms["c_re"], terms["c_im"])))
        assert np.max(np.abs(out - want)) <= (1e-14 if prec == "c128" else 2e-6) * scale
