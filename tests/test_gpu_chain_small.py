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
