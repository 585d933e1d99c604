"""The addresses that a Weight passes to the library are those of the arrays it holds: as made, after an attribute is
set again, after a copy and a pickle; and numpy refuses to move an array that it holds."""
import copy
import pickle
import types
import weakref

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


def test_copies_and_pickles_keep_what_a_program_sets(pkg, monkeypatch):
    """Attributes of its own, and a subclass's slot."""
    named = type("Named", (pkg.Weight,), {"__slots__": ("slot",), "__module__": __name__})
    monkeypatch.setitem(globals(), "Named", named)   # where pickle looks for it
    w = named(np.zeros((4, 16), np.uint8), np.ones((4, 2), np.uint8), 0.5)
    w.name, w.slot = "layers.0.q", 7
    for other in (copy.copy(w), copy.deepcopy(w), pickle.loads(pickle.dumps(w))):
        assert (other.name, other.slot, other.glob) == (w.name, w.slot, 0.5)
        st = other.struct()
        assert st.codes == other.codes.ctypes.data and st.scales == other.scales.ctypes.data
    assert {"codes", "scales", "glob", "n_out", "k", "name"} <= set(vars(w))
    # a state of the arrays alone, as a pickle of an earlier version holds it
    old = pkg.Weight.__new__(pkg.Weight)
    old.__dict__.update(codes=w.codes, scales=w.scales, glob=0.5, n_out=4, k=32)
    assert old.struct().codes == w.codes.ctypes.data
    backend = types.SimpleNamespace(_weights={})
    for ws in ([w], [other, old]):
        arr = pkg.HipBackend._hold(backend, ws)
        assert [(st.codes, st.scales, st.glob, st.n_out, st.k) for st in arr] == [
            (x.codes.ctypes.data, x.scales.ctypes.data, 0.5, 4, 32) for x in ws]
    assert backend._weights == {w.codes.ctypes.data: w, other.codes.ctypes.data: other}


def test_arrays_can_be_let_go(pkg):
    w = pkg.Weight(np.zeros((4, 16), np.uint8), np.ones((4, 2), np.uint8))
    gone = weakref.ref(w.codes)
    w.struct()
    w.codes = None   # its memory goes, and the weight can be used no more
    assert gone() is None
    with pytest.raises(AttributeError):
        w.struct()
    del w.scales
    with pytest.raises(AttributeError):
        w.scales
