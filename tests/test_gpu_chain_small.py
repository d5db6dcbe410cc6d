"""Sampled outcomes on both sides of the limit of one block of outcomes (2^11),
drawn at and beside the steps of the cumulative sums, against the sequential
sums; and the states that have no outcome."""
import numpy as np
import pytest

import qiron
from kat_util import random_state

pytestmark = pytest.mark.gpu


def outcomes(p, u):
    total = 0.0
    for x in p:
        total += x
    cum, cdf = 0.0, []
    for x in p:
        cum += x / total
        cdf.append(cum)
    return np.minimum(np.searchsorted(np.array(cdf), u, side="right"), p.size - 1), np.array(cdf)


@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 7, 10, 11, 12])
def test_outcomes_at_the_steps_of_the_cumulative_sums(ctx, m, prec):
    n = 12
    s = qiron.State.from_vector_unchecked(random_state(n, np.random.default_rng(40 + m)), prec)
    qs = list(range(n - m, n))
    p = s.measure_probs(qs)
    _w, cdf = outcomes(p, np.zeros(0))
    u = np.concatenate([cdf, np.nextafter(cdf, 0), np.nextafter(cdf, 2), np.random.default_rng(m).random(300), [0.0]])
    u = u[(u >= 0) & (u < 1)]
    np.testing.assert_array_equal(s.measure_outcomes(qs, u).astype(np.int64), outcomes(p, u)[0])


@pytest.mark.parametrize("n,m", [(1, 1), (11, 11), (12, 12)])
def test_a_zero_state_is_an_error(ctx, n, m):
    s = qiron.State.from_vector_unchecked(np.zeros(1 << n, dtype=np.complex128), "c128")
    with pytest.raises(qiron.QuantIronError):
        s.measure_outcomes(list(range(m)), [0.5])


# qubits out of order and listed again: an outcome whose bits contradict each other has no weight
@pytest.mark.parametrize("prec", ["c64", "c128"])
@pytest.mark.parametrize("n,qs", [(3, [2, 0]), (3, [1, 1, 1]), (9, [8, 0, 8, 3]), (13, [12, 12]), (14, [5, 3, 5, 9, 13, 0, 0, 1, 2, 7, 11]),
                                  (14, [5, 3, 5, 9, 13, 0, 0, 1, 2, 7, 11, 12])])
def test_lists_out_of_order_and_with_repeats(ctx, n, qs, prec):
    s = qiron.State.from_vector_unchecked(random_state(n, np.random.default_rng([n, len(qs)])), prec)
    p = s.measure_probs(qs)
    for a in range(len(qs)):
        for b in range(a):
            if qs[a] == qs[b]:
                o = np.arange(p.size)
                assert not np.any(p[((o >> a) ^ (o >> b)) & 1 == 1])
    u = np.random.default_rng(n).random(2000)
    got = s.measure_outcomes(qs, u).astype(np.int64)
    np.testing.assert_array_equal(got, outcomes(p, u)[0])
    r = s.measure(qiron.MeasurementBasis.Computational, qs, float(u[0]))
    assert sum(bit << k for k, bit in enumerate(r.outcomes)) == got[0]
