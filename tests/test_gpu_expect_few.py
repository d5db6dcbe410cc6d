"""One and two terms of one x mask, streamed where the state about fills the
last-level cache and in tiles beside it, on a product state whose expectations
are known."""
import numpy as np
import pytest

import qiron
from kat_util import term_array

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("n", [21, 22, 24, 25])
def test_few_terms_on_a_product_state(ctx, n, prec):
    angles = np.linspace(0.3, 2.6, n)
    s = qiron.State.new_zero(n, prec, ctx)
    qiron.Circuit(n, [qiron.Gate.ry_gate(q, float(a)) for q, a in enumerate(angles)]).execute_inplace(s)
    z, x = np.cos(angles), np.sin(angles)
    # 25 rotations: FP64 sums of unit norm, or 25 roundings of a 24-bit product
    tol = 1e-13 if prec == "c128" else 25 * 4 * 2.0 ** -24
    for a, b in ((0, n - 1), (3, 5), (n - 2, n - 1)):
        m = 1 << a | 1 << b
        for terms, want in (([(0, 1 << a, 0.5, 0.25)], (0.5 + 0.25j) * z[a]), ([(0, m, 2.0, 0.0)], 2 * z[a] * z[b]),
                            ([(m, 0, 0.5, 0.0)], 0.5 * x[a] * x[b]), ([(m, m, 0.5, 0.0), (m, 0, 1.0, 0.0)], x[a] * x[b]),
                            ([(0, 1 << a, 1.0, 0.0), (0, 1 << b, 0.0, 1.0)], z[a] + 1j * z[b])):
            assert abs(qiron.expectation_terms(s, term_array(terms)) - want) <= tol * 3
