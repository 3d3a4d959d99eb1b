"""A column that stores an entry twice takes the last value, as the one-by-one
insertion of the reference does (SparseCSCInterface.jl:112-163): the solution
is bit for bit that of the matrix without the earlier one. The repeat stands
right before the entry or out of order before the whole column, in the first
or last column, with the map built by one host thread or by several (2^18
entries and more)."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

from helpers import csc1
from sparspak_hip import _lib
from sparspak_hip.gallery import laplace2d
from sparspak_hip.symbolic import Graph, SymbolicFactor

pytestmark = pytest.mark.gpu


def _solve_csc(sym, n, colptr, rowval, nzval, b):
    L, I, P = _lib.lib(), _lib.p64, _lib.pd
    h = ctypes.c_void_p()
    _lib.check(L.spkhip_create(ctypes.byref(h), 0), "spkhip_create")
    try:
        _lib.check(L.spkhip_symbolic_upload(
            h, 0, n, sym.nsuper, I(sym.xsuper), I(sym.snode), I(sym.xlindx), I(sym.lindx),
            I(sym.xlnz), I(sym.xunz), I(sym.order.rperm), I(sym.order.rinvp), I(colptr),
            I(rowval)), "spkhip_symbolic_upload")
        _lib.check(L.spkhip_inmatrix(h, P(nzval)), "spkhip_inmatrix")
        _lib.check(L.spkhip_factor(h, 0), "spkhip_factor")
        x = b.copy()
        _lib.check(L.spkhip_solve(h, 1, P(x), n), "spkhip_solve")
    finally:
        L.spkhip_destroy(h)
    return x


@pytest.mark.parametrize("nx", [7, 240])
@pytest.mark.parametrize("col", [0, -1])
@pytest.mark.parametrize("adjacent", [True, False])
def test_last_value_counts(nx, col, adjacent):
    print(f"case repeated entries {nx} {col} {adjacent}", flush=True)
    A = sp.csc_matrix(laplace2d(nx, nx))
    A.sort_indices()
    n, cp, rv, nz = csc1(A)
    sym = SymbolicFactor(n, Graph.from_csc(n, cp, rv), kind="lu")
    sym.findorder()
    sym.symbolicfactor()
    b = np.arange(1.0, n + 1) / n
    want = _solve_csc(sym, n, cp, rv, nz, b)
    col %= n
    last = cp[col + 1] - 2  # the column's last entry
    at = last if adjacent else cp[col] - 1
    cp2 = cp.copy()
    cp2[col + 1:] += 1
    got = _solve_csc(sym, n, cp2, np.insert(rv, at, rv[last]), np.insert(nz, at, 77.0), b)
    assert np.array_equal(got, want)
