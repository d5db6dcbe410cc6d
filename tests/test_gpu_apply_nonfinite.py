"""SumOp products of states with an infinite or NaN amplitude: Pauli factors move
and negate parts, a coefficient multiplies as a complex number, and the parts
that are not numbers follow from that, as a gather and in tile passes."""
import numpy as np
import pytest

import qiron
from kat_util import random_state

pytestmark = pytest.mark.gpu


def product(psi, rows):
    i = np.arange(psi.size, dtype=np.uint64)
    re, im = np.zeros(psi.size), np.zeros(psi.size)
    with np.errstate(all="ignore"):
        for x, z, cr, ci in rows:
            j = i ^ np.uint64(x)
            a, b = psi.real[j], psi.imag[j]
            sign = 1.0 - 2.0 * (np.bitwise_count(i & np.uint64(z)) & 1)  # of (-i)^ny (-1)^(i & z)
            for _ in range(bin(x & z).count("1")):
                a, b = b, -a
            a, b = a * sign, b * sign
            re, im = re + (a * cr - b * ci), im + (a * ci + b * cr)
    return re, im


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("n", [13, 21])
@pytest.mark.parametrize("value", [complex(np.nan, 0), complex(np.inf, 0), complex(0, -np.inf), complex(np.nan, np.nan)])
def test_parts_that_are_not_numbers(ctx, n, prec, value):
    psi = random_state(n, np.random.default_rng(n))
    if prec == "c64":
        psi = psi.astype(np.complex64).astype(np.complex128)
    psi[3] = value
    s = qiron.State.from_vector_unchecked(psi, prec)
    full = (1 << n) - 1
    for rows in ([(0, 1, 0.5, 0.0)], [(1, 0, 0.5, 0.0)], [(2, 2, 0.5, 0.0)], [(1, 0, 0.0, 0.0)], [(1, 1, 0.5, 0.25)],
                 [(0, 3, 0.2, 0.0), (3, 1, 0.1, 0.0), (1, 2, -0.3, 0.0), (12, 4, 0.4, 0.0)], [(full, 5, 0.5, 0.0)]):
        ops = [{q: "XZY"[(x >> q & 1) + 2 * (z >> q & 1) - 1] for q in range(n) if (x | z) >> q & 1} for x, z, _r, _i in rows]
        out = qiron.SumOp([qiron.PauliString(complex(r, i), o) for (_x, _z, r, i), o in zip(rows, ops)]).apply(s).state_vector
        for got, want in zip((out.real, out.imag), product(psi, rows)):
            np.testing.assert_array_equal(np.isnan(got), np.isnan(want), str(rows))
            np.testing.assert_array_equal(np.isinf(got), np.isinf(want), str(rows))
            ok = np.isfinite(want)
            # finite parts: a few roundings of amplitudes below 1
            assert np.max(np.abs(got[ok] - want[ok])) <= (1e-14 if prec == "c128" else 2e-6), rows
