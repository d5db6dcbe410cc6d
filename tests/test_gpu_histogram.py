"""Measurement histograms and sampling at the edges of the row kernel: states
below, at and above one row, measured sets inside the row, outside it and
mixed, listed in and out of order and with repeats; cumulative sums on both
sides of the sequential / chunked limit (2^16 outcomes)."""
import numpy as np
import pytest

import qiron
from kat_util import random_state

pytestmark = pytest.mark.gpu


def probs(psi, qubits):
    p = psi.real ** 2 + psi.imag ** 2
    idx = np.arange(psi.size)
    o = np.zeros(psi.size, dtype=np.int64)
    for b, q in enumerate(qubits):
        o |= ((idx >> q) & 1) << b
    # sums of up to 2^17 positive values; longdouble keeps the reference below FP64 rounding
    out = np.zeros(1 << len(qubits), dtype=np.longdouble)
    np.add.at(out, o, p.astype(np.longdouble))
    return out


def held(n, prec, seed):
    psi = random_state(n, np.random.default_rng(seed))
    if prec == "c64":
        psi = psi.astype(np.complex64).astype(np.complex128)
    return psi, qiron.State.from_vector_unchecked(psi, prec)


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("n", [1, 5, 6, 7, 8, 11, 17])
def test_histogram(ctx, n, prec):
    psi, s = held(n, prec, 300 + n)
    rng = np.random.default_rng(n)
    sets = [[0], [n - 1], list(range(n)), list(range(n))[::-1], [0, n - 1, 0] if n > 2 else [0]]
    sets += [sorted(int(q) for q in rng.choice(n, size=max(1, n // 2), replace=False)) for _ in range(4)]
    sets += [list(range(max(0, n - 3), n)), list(range(min(n, 3)))]
    for qs in sets:
        if len(qs) > n:
            continue
        # |a|^2 carries at most 1.5 ulp, the compensated sum and the fold half an ulp each: under 6e-16
        np.testing.assert_allclose(s.measure_probs(qs), probs(psi, qs).astype(np.float64), rtol=1e-15, atol=0)


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("m", [1, 6, 10, 16, 17])
def test_sampled_outcomes_follow_the_cumulative_sums(ctx, m, prec):
    n = 18
    _psi, s = held(n, prec, 900)
    qs = list(range(n - m, n))
    u = np.random.default_rng(m).random(5000)
    p = s.measure_probs(qs)
    total = 0.0
    for x in p:  # sequential, as the reference sums
        total += x
    cdf = np.cumsum(p / total)
    want = np.minimum(np.searchsorted(cdf, u, side="right"), p.size - 1)
    got = s.measure_outcomes(qs, u).astype(np.int64)
    if m <= 16:
        np.testing.assert_array_equal(got, want)
    else:  # chunk prefixes round differently from the sequential sum, by under 1e-12: a draw that close to a step may differ
        for k in np.nonzero(got != want)[0]:
            assert abs(cdf[min(got[k], want[k])] - u[k]) < 1e-12
