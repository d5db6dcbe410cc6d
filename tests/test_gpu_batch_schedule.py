"""A schedule that is asked for by its numbers is the schedule: the default one,
set explicitly, gives the default's bits, and so does another batch with the
autotuned one."""
import numpy as np
import pytest

import qiron
from qiron import surrogate as S

pytestmark = pytest.mark.gpu


def batch(prec, seed):
    rng = np.random.default_rng(seed)
    specs = [(n, 3, 2 * np.pi * rng.random(2 * n * 3), 0.5 + rng.random(3)) for n in (9, 13, 14, 15, 16, 16, 17, 17, 18)]
    b = S.ansatz_batch(specs, prec)
    b.set_angles(np.concatenate([s[2] for s in specs]))
    return b


@pytest.mark.parametrize("prec", ["c64", "c128"])
def test_the_default_schedule_by_its_numbers(ctx, prec):
    for seed in range(4):
        b = batch(prec, seed)
        default = b.run()
        k, ks = b.schedule()
        assert k == ks == (12 if prec == "c128" else 13)
        b.set_schedule(k, ks)
        np.testing.assert_array_equal(b.run(), default)


@pytest.mark.parametrize("prec", ["c64", "c128"])
def test_an_autotuned_schedule_carries_over(ctx, prec):
    b, other = batch(prec, 7), batch(prec, 7)
    b.autotune(trials=1)
    other.set_executor(b.executor())
    other.set_schedule(*b.schedule())
    np.testing.assert_array_equal(other.run(), b.run())
