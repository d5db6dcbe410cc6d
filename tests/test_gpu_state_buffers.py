"""Buffers of destroyed states are kept for the next state of the same size:
live states never share one, a reused one holds the new state's amplitudes, and
another context's states take none of them."""
import ctypes as C

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


def test_work_on_another_stream_is_done_before_a_buffer_is_reused(ctx):
    n, size = 20, 8 << 20
    hip = qiron.load_library()  # the HIP runtime that the engine runs on

    def call(name, *args):
        assert getattr(hip, name)(*args) == 0, name

    def device(b):
        p = C.c_void_p()
        call("hipMalloc", C.byref(p), C.c_size_t(b))
        return p

    def copy(dst, src, b):  # device to device, on the side stream
        call("hipMemcpyAsync", dst, src, C.c_size_t(b), 3, side)

    side, big = C.c_void_p(), 1 << 30
    call("hipStreamCreateWithFlags", C.byref(side), C.c_uint(1))
    s = qiron.State.new_plus(n, "c64", ctx)
    threes, seen, a, b = device(size), device(size), device(big), device(big)
    call("hipMemcpy", threes, np.full(2 << n, 3.0, np.float32).ctypes.data_as(C.c_void_p), C.c_size_t(size), 1)
    address = ptr(s)
    for _ in range(100):  # tens of milliseconds: what follows is pending when the state goes
        copy(a, b, big)
    copy(seen, C.c_void_p(address), size)
    copy(C.c_void_p(address), threes, size)
    del s
    again = qiron.State.new_zero(n, "c64", ctx)
    assert ptr(again) == address
    v = again.state_vector
    assert v[0] == 1 and not np.any(v[1:])
    call("hipStreamSynchronize", side)
    out = np.empty(2 << n, np.float32)
    call("hipMemcpy", out.ctypes.data_as(C.c_void_p), seen, C.c_size_t(size), 2)
    np.testing.assert_array_equal(out[0::2], np.float32(2.0 ** (-n / 2)))
    assert not np.any(out[1::2])
    assert again.state_vector[0] == 1  # nothing arrived late
    for p in (threes, seen, a, b):
        call("hipFree", p)
    call("hipStreamDestroy", side)
