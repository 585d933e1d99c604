"""The addresses that a Weight passes to the library are those of the arrays it holds: as made, after an attribute is
set again, after a copy and a pickle; and numpy refuses to move an array that it holds."""
import copy
import pickle

import numpy as np
import pytest


def test_addresses_follow_the_arrays(pkg):
    w = pkg.Weight(np.arange(64, dtype=np.uint8).reshape(4, 16), np.ones((4, 2), np.uint8), 0.5)

    def holds(x):
        st = x.struct()
        assert st.codes == x.codes.ctypes.data and st.scales == x.scales.ctypes.data
        assert (st.n_out, st.k, st.glob) == (4, 32, 0.5)

    holds(w)
    for other in (copy.copy(w), copy.deepcopy(w), pickle.loads(pickle.dumps(w))):
        holds(other)
        np.testing.assert_array_equal(other.codes, w.codes)
    first = w.codes
    w.codes = w.codes.copy()
    w.scales = w.scales.copy()
    assert w.codes.ctypes.data != first.ctypes.data
    holds(w)
    with pytest.raises(ValueError):
        w.codes.resize((8, 16))
    holds(w)
