"""Refinement with a pattern that stores an entry twice: residual, norms and
factor are those of one matrix, whose entry is the last value stored (the
reference inserts one by one, SparseCSCInterface.jl:112-163). The refined
solution and the backward error are bit for bit those of the matrix without
the earlier entry: LU and SPD (stored whole, the repeat in the lower or in the
upper triangle, which the SPD factor does not read), one and several
right-hand sides, one and two value sets."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

from helpers import csc1
from sparspak_hip import _lib
from sparspak_hip.gallery import laplace2d
from sparspak_hip.symbolic import Graph, SymbolicFactor

pytestmark = pytest.mark.gpu


def _refined(kind, sym, n, colptr, rowval, nzval, b, nrhs, nvs):
    L, I, P = _lib.lib(), _lib.p64, _lib.pd
    h = ctypes.c_void_p()
    _lib.check(L.spkhip_create(ctypes.byref(h), 0), "spkhip_create")
    try:
        xunz = sym.xunz if sym.xunz is not None else np.zeros(n + 1, dtype=np.int64)
        _lib.check(L.spkhip_symbolic_upload(
            h, 0 if kind == "lu" else 1, n, sym.nsuper, I(sym.xsuper), I(sym.snode),
            I(sym.xlindx), I(sym.lindx), I(sym.xlnz), I(xunz), I(sym.order.rperm),
            I(sym.order.rinvp), I(colptr), I(rowval)), "spkhip_symbolic_upload")
        if nvs > 1:
            _lib.check(L.spkhip_set_value_sets(h, nvs), "spkhip_set_value_sets")
        _lib.check(L.spkhip_inmatrix(h, P(nzval)), "spkhip_inmatrix")
        _lib.check(L.spkhip_factor(h, 1), "spkhip_factor")
        x = b.copy()
        _lib.check(L.spkhip_solve_refine(h, nrhs, P(x), n * nvs, 1e-15, 20),
                   "spkhip_solve_refine")
        st = _lib.Stats()
        _lib.check(L.spkhip_stats(h, ctypes.byref(st)), "spkhip_stats")
    finally:
        L.spkhip_destroy(h)
    return x, st.backward_error


@pytest.mark.parametrize("nrhs,nvs", [(1, 1), (3, 1), (2, 2)])
@pytest.mark.parametrize("adjacent", [True, False])
@pytest.mark.parametrize("kind,which", [("lu", -1), ("lu", 0), ("spd", -1), ("spd", 0)])
def test_refined_solution_is_the_last_values(kind, which, adjacent, nrhs, nvs):
    print(f"case repeated refine {kind} {which} {adjacent} {nrhs} {nvs}", flush=True)
    A = sp.csc_matrix(laplace2d(17, 17))
    A.sort_indices()
    n, cp, rv, nz = csc1(A)
    sym = SymbolicFactor(n, Graph.from_csc(n, cp, rv), kind=kind)
    sym.findorder()
    sym.symbolicfactor()
    b = np.tile((np.arange(1.0, n * nvs + 1) / n), nrhs)
    want, eta = _refined(kind, sym, n, cp, rv, np.tile(nz, nvs), b, nrhs, nvs)
    col = n // 2
    e = cp[col + 1] - 2 if which < 0 else cp[col] - 1  # the column's last or first entry
    end = cp[col + 1] - 1
    order = np.r_[0:e, e + 1:end, e, end:len(rv)]  # ... stored last in its column
    cp2 = cp.copy()
    cp2[col + 1:] += 1
    at = end - 1 if adjacent else cp[col] - 1
    got, eta2 = _refined(kind, sym, n, cp2, np.insert(rv[order], at, rv[e]),
                         np.tile(np.insert(nz[order], at, 77.0), nvs), b, nrhs, nvs)
    assert np.array_equal(got, want) and eta == eta2
