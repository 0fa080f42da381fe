"""Host arrays handed to the library: a call sees memory that is still held."""
import ctypes as C
import weakref

import numpy as np
import pytest

from turbulentbl_amd import tbl


class _Lib:
    """stands in for the library: notes whether the array whose address a call
    receives is still there"""

    def __init__(self, live):
        self.live, self.seen = live, []

    def __getattr__(self, name):
        def call(*a):
            self.seen += [self.live[p]() is not None for p in a if isinstance(p, int) and p in self.live]
            return 0
        return call


@pytest.mark.parametrize("method", ["set_field", "apply_operator"])
def test_converted_input_is_held_during_the_call(monkeypatch, method):
    live, f64 = {}, tbl._f64

    class Held(np.ndarray):
        pass

    def converted(a):
        h = f64(a).view(Held)
        live[h.ctypes.data] = weakref.ref(h)
        return h

    monkeypatch.setattr(tbl, "_f64", converted)
    sv = object.__new__(tbl.Solver)
    sv.lib, sv.h, sv.nX, sv.nY, sv.nZ = _Lib(live), C.c_void_p(), 8, 8, 8
    x = np.ones((8, 8, 8), dtype=np.float32)                 # converted: another type and order
    getattr(sv, method)(0, x)
    assert sv.lib.seen == [True]
    sv.h = None
