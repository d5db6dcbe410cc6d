"""Lists whose planning memory or tables are more than a context keeps: they run
from memory of the call's own, and small lists before and after them are right."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
import qiron
from kat_util import gates_array, random_state, random_terms, term_array
from qiron import _lib as L

pytestmark = pytest.mark.gpu


def noalloc(state, terms):
    re, im, err = C.c_double(), C.c_double(), L.QiError()
    rc = state.lib.qi_sumop_expectation_noalloc(state._h, terms.ctypes.data_as(C.c_void_p), terms.size, C.byref(re), C.byref(im),
                                                C.byref(err))
    assert rc == 0
    return complex(re.value, im.value)


def test_long_sumops(ctx):
    n = 16
    rng = np.random.default_rng(5)
    psi = random_state(n, rng)
    s = qiron.State.from_vector_unchecked(psi, "c128")
    few = random_terms(n, 40, rng, max_weight=n)
    want = O.expectation(psi, few)
    # 2^19 Z supports on eight masks: more than 32 MiB of tables, more than 8 MiB to plan in
    z = np.arange(1 << 19, dtype=np.uint64)
    rows = np.zeros(z.size, dtype=L.TERM_DTYPE)
    rows["x_mask"] = 1 << (z % 8)
    rows["z_mask"] = z >> 3
    rows["c_re"] = rng.normal(size=z.size)
    rows = rows[rng.permutation(z.size)]
    tol = 1e-12 * float(np.sum(np.abs(rows["c_re"])))
    parts = sum(qiron.expectation_terms(s, p) for p in np.array_split(rows, 40))  # each within what is kept
    assert abs(qiron.expectation_terms(s, few) - want) <= 1e-12 * float(np.sum(np.hypot(few["c_re"], few["c_im"])))
    whole = qiron.expectation_terms(s, rows)
    assert abs(whole - parts) <= tol
    assert qiron.expectation_terms(s, few) == noalloc(s, few)
    assert abs(noalloc(s, few) - want) <= 1e-12 * float(np.sum(np.hypot(few["c_re"], few["c_im"])))
    assert qiron.expectation_terms(s, rows) == whole


@pytest.mark.parametrize("prec", ["c64", "c128"])
def test_long_gate_lists_on_a_small_state(ctx, prec):
    rng = np.random.default_rng(6)
    n = 5
    psi = random_state(n, rng)
    s = qiron.State.from_vector_unchecked(psi, prec)
    # 2^17 times the same three permutations: 37 MiB of op tables, and an even power of each is the identity
    block = gates_array([{"kind": "X", "targets": [1]}, {"kind": "X", "targets": [3], "controls": [0]}, {"kind": "SWAP", "targets": [2, 4]}])
    before = s.state_vector.copy()
    s.apply_gates_inplace(np.tile(block, 1 << 17))
    np.testing.assert_array_equal(s.state_vector, before)
    s.apply_gates_inplace(block)
    assert np.max(np.abs(s.state_vector - O.apply_gates(before, block))) == 0
