"""Which densities the pivoted Cholesky factor stands for: the rule on what a finished factorisation found."""
import ctypes
import math

import pytest

INF, NAN = math.inf, math.nan


@pytest.mark.parametrize("dmax,columns,left,want", [
    (2.0, 5, 0.0, 5), (2.0, 5, 1.5e-13, 5), (2.0, 5, 2e-13, -1), (2.0, 5, 1e300, -1),
    (0.0, 0, 0.0, 0),                 # P = 0
    (-1.0, 0, 1.0, -1),               # negative definite
    (INF, 0, INF, -1),                # an infinite diagonal element: no column, and everything is left
    (INF, 0, 3.0, -1), (NAN, 0, 0.0, -1), (2.0, 5, NAN, -1), (2.0, 5, INF, -1)])
def test_rule(dmax, columns, left, want):
    from dftax_amd import _native
    f = _native.lib()["_ZN4dfks15pfactor_columnsEPKdd"]
    f.restype, f.argtypes = ctypes.c_int, [ctypes.POINTER(ctypes.c_double), ctypes.c_double]
    assert f((ctypes.c_double * 4)(dmax, columns, 1.0, left), 1e-14) == want
