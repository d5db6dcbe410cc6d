"""Expectations add every amplitude's product by two-sum: a contribution of 1
survives between two of 2^60 that cancel, wherever the three lie."""
import itertools

import numpy as np
import pytest

import qiron
from kat_util import term_array

pytestmark = pytest.mark.gpu

BIG = 2.0 ** 30


def state(n, prec, amplitudes):
    v = np.zeros(1 << n, dtype=np.complex128)
    for i, a in amplitudes.items():
        v[i] = a
    return qiron.State.from_vector_unchecked(v, prec)


# all numbers are powers of two below 2^62 and the exact sum is a small integer
@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("n", [3, 4, 9, 14])
def test_cancelling_products_keep_what_lies_between(ctx, n, prec):
    for lo, hi in itertools.permutations(range(n), 2):
        s = state(n, prec, {0: BIG, 1 << lo: 1.0, 1 << hi: BIG})
        for c in (1.0, 1j):
            got = qiron.expectation_terms(s, term_array([(0, 1 << hi, c.real, c.imag)]))  # Z: 2^60 + 1 - 2^60
            assert got == c, (lo, hi)
    for p in range(n):
        q = [b for b in range(n) if b != p]
        for a, b in itertools.permutations(q, 2):
            x = 1 << p
            s = state(n, prec, {0: BIG, x: BIG, 1 << a: 1.0, 1 << a | x: 1.0, 1 << b: BIG, 1 << b | x: -BIG})
            got = qiron.expectation_terms(s, term_array([(x, 0, 1.0, 0.0)]))  # X: twice 2^60 + 1 - 2^60
            assert got == 2.0, (p, a, b)
            if a == q[0]:
                y = qiron.expectation_terms(s, term_array([(x, x, 0.5, 0.0), (x, 0, 1.0, 0.25)]))  # a Y beside it: Im w is 0
                assert y == 2.0 + 0.5j, (p, a, b)


# a sum with a value that is not finite is NaN in both parts, whatever the route
@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("n", [2, 5, 13, 15])
@pytest.mark.parametrize("value", [complex(np.nan, 0), complex(np.inf, 0), complex(0, -np.inf)])
def test_values_that_are_not_finite(ctx, n, prec, value):
    v = np.full(1 << n, 2.0 ** (-n / 2), dtype=np.complex128)
    v[3] = value
    s = qiron.State.from_vector_unchecked(v, prec)
    full = (1 << n) - 1
    for terms in ([(0, 1, 0.5, 0.0)], [(1, 0, 0.5, 0.0)], [(2, 2, 0.5, 0.0)], [(1, 0, 0.5, 0.25)], [(1, 0, 0.0, 0.0)], [(full, 0, 1.0, 0.0)],
                  [(0, 3, 0.2, 0.0), (3, 1, 0.1, 0.0), (full, 2, -0.3, 0.0)]):
        got = qiron.expectation_terms(s, term_array(terms))
        assert np.isnan(got.real) and np.isnan(got.imag), terms
