"""Buffers of destroyed states are kept for the next state of the same size:
live states never share one, a reused one holds the new state's amplitudes, and
another context's states take none of them."""
import numpy as np
import pytest

import qiron

pytestmark = pytest.mark.gpu


def ptr(s):
    return s.lib.qi_state_device_ptr(s._h)


@pytest.mark.parametrize("n,prec", [(1, "c64"), (10, "c128"), (20, "c64")])
def test_buffers_are_reused_one_owner_at_a_time(n, prec):
    c = qiron.Context(0)
    states = [qiron.State.new_plus(n, prec, c) for _ in range(5)]
    seen = {ptr(s) for s in states}
    assert len(seen) == 5
    keep = states.pop()
    del states
    again = [qiron.State.new_zero(n, prec, c) for _ in range(4)]
    assert len({ptr(s) for s in again} | {ptr(keep)}) == 5
    assert {ptr(s) for s in again} <= seen  # the four idle ones
    for s in again:
        v = s.state_vector
        assert v[0] == 1 and not np.any(v[1:])
    del s  # every state of a context goes before the context
    np.testing.assert_allclose(keep.state_vector, 2.0 ** (-n / 2), rtol=1e-7)
    other = qiron.Context(0)
    del again
    foreign = qiron.State.new_zero(n, prec, other)
    assert ptr(foreign) not in seen
    copy = keep.clone()
    assert ptr(copy) in seen - {ptr(keep)}
    del copy, keep, foreign
    c.close()
    other.close()


def test_many_small_states_stay_bounded():
    c = qiron.Context(0)
    states = [qiron.State.new_basis_n(4, k % 16, "c64", c) for k in range(100)]  # more than are kept idle
    del states
    states = [qiron.State.new_basis_n(4, k % 16, "c64", c) for k in range(100)]
    for k, s in enumerate(states):
        assert s.state_vector[k % 16] == 1
    del states, s
    c.close()
