"""The bytes that the per-class profile attributes to the fronts' assembly: a
large front's matrix written once and its children's update matrices read
(A's entries are not counted); a small front's panels and update matrix
written and its children's read. One dense front (no children) of each kind,
and two small leaves on a large core."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

from sparspak_hip import SparseSolver, _lib, factor, findorderperm, inmatrix, symbolicfactor

pytestmark = pytest.mark.gpu


def _bytes(A, precision):
    n = A.shape[0]
    s = SparseSolver(A)
    findorderperm(s, np.arange(1, n + 1))
    symbolicfactor(s)
    inmatrix(s)
    dev = s.slvr._dev
    _lib.check(dev.L.spkhip_profile_enable(dev.h, 1), "spkhip_profile_enable")
    factor(s, precision)
    out = {}
    for k, name in enumerate(_lib.KCLASSES):
        st = _lib.KStat()
        _lib.check(dev.L.spkhip_profile_get(dev.h, k, ctypes.byref(st)), "spkhip_profile_get")
        out[name] = st.bytes
    return out, s.slvr.sym


@pytest.mark.parametrize("precision,size", [("fp64", 8), ("fp32", 4)])
def test_assembly_bytes(precision, size):
    print(f"case profile bytes {precision}", flush=True)
    for n in (100, 300):
        out, _ = _bytes(sp.csc_matrix(np.ones((n, n)) + n * np.eye(n)), precision)
        assert out["large_init"] == size * n * n and out["small_front"] == 0
    n = 50
    out, _ = _bytes(sp.csc_matrix(np.ones((n, n)) + n * np.eye(n)), precision)
    assert out["small_front"] == size * n * n and out["large_init"] == 0
    # two leaves of one column and 20 update rows each on a core of 100
    P = np.zeros((102, 102))
    P[2:, 2:] = P[[0, 1], [0, 1]] = 1
    P[:2, 2:22] = P[2:22, :2] = 1
    out, sym = _bytes(sp.csc_matrix(P + 102 * np.eye(102) * (P > 0)), precision)
    assert np.array_equal(sym.xsuper[:3], [1, 2, 3])
    assert np.array_equal(np.diff(sym.xlindx[:4]), [21, 21, 100])
    # a leaf's panels 21^2 - 20^2, its update matrix 20^2
    assert out["small_front"] == size * 2 * 21 * 21
    assert out["large_init"] == size * (100 * 100 + 2 * 20 * 20)
