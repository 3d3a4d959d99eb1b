"""A symbolic upload that is refused (a piece wider than the kernels take:
-2; an index list that does not nest in its parent's: -4) leaves a handle that
holds no symbolic factor, whatever it held before: every later phase is out of
sequence (-3) until an upload succeeds, and then the handle works as a new
one."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

from helpers import csc1, symbolic
from sparspak_hip import _lib
from sparspak_hip.gallery import laplace2d

pytestmark = pytest.mark.gpu


def _upload(h, kind, n, sym, cp, rv, lindx=None):
    L, I = _lib.lib(), _lib.p64
    return int(L.spkhip_symbolic_upload(
        h, kind, n, sym.nsuper, I(sym.xsuper), I(sym.snode), I(sym.xlindx),
        I(sym.lindx if lindx is None else lindx), I(sym.xlnz), I(sym.xunz), I(sym.order.rperm),
        I(sym.order.rinvp), I(cp), I(rv)))


@pytest.mark.parametrize("why", ["wide", "nested"])
def test_refused_upload_holds_nothing(why):
    print(f"case refused upload {why}", flush=True)
    L, P = _lib.lib(), _lib.pd
    A = laplace2d(9, 9)
    n, cp, rv, nz = csc1(A)
    sym = symbolic(A)
    if why == "wide":  # one piece of 60 columns, more than an LU piece may have
        m = 60
        B = sp.csc_matrix(np.ones((m, m)) + m * np.eye(m))
        bad, lindx = symbolic(B, maxblocksize=m), None
    else:  # the last row of the first front with update rows is no longer its parent's
        m, B, bad = n, A, symbolic(A)
        lindx = bad.lindx.copy()
        J = next(J for J in range(bad.nsuper) if bad.xlindx[J + 1] - bad.xlindx[J]
                 > bad.xsuper[J + 1] - bad.xsuper[J] + 1)
        have = set(lindx[bad.xlindx[J] - 1:bad.xlindx[J + 1] - 1])
        par = bad.snode[lindx[bad.xlindx[J] - 1 + bad.xsuper[J + 1] - bad.xsuper[J]] - 1] - 1
        have |= set(lindx[bad.xlindx[par] - 1:bad.xlindx[par + 1] - 1])
        lindx[bad.xlindx[J + 1] - 2] = next(g for g in range(n, 0, -1) if g not in have)
    _, cpb, rvb, _ = csc1(B)
    b = np.arange(1.0, n + 1)
    h = ctypes.c_void_p()
    _lib.check(L.spkhip_create(ctypes.byref(h), 0), "spkhip_create")
    try:
        assert _upload(h, 0, n, sym, cp, rv) == 0
        _lib.check(L.spkhip_inmatrix(h, P(nz)), "spkhip_inmatrix")
        _lib.check(L.spkhip_factor(h, 0), "spkhip_factor")
        x0 = b.copy()
        _lib.check(L.spkhip_solve(h, 1, P(x0), n), "spkhip_solve")
        assert _upload(h, 0, m, bad, cpb, rvb, lindx) == (-2 if why == "wide" else -4)
        big = np.zeros(max(n, m))
        assert L.spkhip_inmatrix(h, P(np.zeros(len(rv) + len(rvb)))) == -3
        assert L.spkhip_factor(h, 0) == -3
        assert L.spkhip_solve(h, 1, P(big), max(n, m)) == -3
        assert L.spkhip_solve_refine(h, 1, P(big), max(n, m), 1e-15, 5) == -3
        assert L.spkhip_download(h, P(np.zeros(sym.nlnz + bad.nlnz)), None, None) == -3
        assert _upload(h, 0, n, sym, cp, rv) == 0
        _lib.check(L.spkhip_inmatrix(h, P(nz)), "spkhip_inmatrix")
        _lib.check(L.spkhip_factor(h, 0), "spkhip_factor")
        x = b.copy()
        _lib.check(L.spkhip_solve(h, 1, P(x), n), "spkhip_solve")
        assert np.array_equal(x, x0)
    finally:
        L.spkhip_destroy(h)
