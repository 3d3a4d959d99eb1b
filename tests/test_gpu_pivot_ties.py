"""The pivot search of the diagonal regions where the leading 32 bits of the
candidates' magnitudes agree: a piece's first column whose entries differ in
the low half of the double only, tie exactly (the smallest position wins), or
tie up to sign. The matrices are diagonal apart from every piece's first
column, so the elimination's other pivots are far apart and the interchanges
do not depend on rounding: they equal the oracle's, in double and in float
(where the low half rounds away and the ties are exact)."""
import numpy as np
import pytest
import scipy.sparse as sp

import oracle.oracle as orc
from helpers import csc1
from sparspak_hip import SparseSolver, factor, findorder, inmatrix, symbolicfactor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", ["low", "equal", "sign", "low_descending"])
@pytest.mark.parametrize("n", [31, 60, 90])
def test_pivot_ties(n, kind, precision):
    print(f"case n={n} {kind} {precision}", flush=True)
    rng = np.random.default_rng(n)
    order = rng.permutation(n).astype(float)
    col = {"low": 16.0 + order * 2.0 ** -40, "equal": np.full(n, 16.0),
           "sign": 16.0 * rng.choice([-1.0, 1.0], n),
           "low_descending": 16.0 - np.arange(n) * 2.0 ** -40}[kind]
    M = np.diag(rng.uniform(1, 2, n))
    # every entry stored (the zeros too): one dense front
    idx = np.tile(np.arange(n), n)
    A = sp.csc_matrix((M.T.ravel(), idx, np.arange(n + 1) * n), shape=(n, n))
    s = SparseSolver(A)
    findorder(s)
    symbolicfactor(s)
    sym = s.slvr.sym
    p = sym.order.rperm - 1
    first = sym.xsuper[:-1] - 1  # first columns of the pieces, new numbering
    Mp = M[np.ix_(p, p)]
    for f, e in zip(first, sym.xsuper[1:] - 1):
        Mp[f:e, f] = col[f:e]
    M[np.ix_(p, p)] = Mp
    A = sp.csc_matrix((M.T.ravel(), idx, np.arange(n + 1) * n), shape=(n, n))
    s._nzval = A.data.copy()
    inmatrix(s)
    s.slvr.set_tuning(small_lmax=0)
    inmatrix(s)
    factor(s, precision)
    _, _, ipiv = s.slvr.download()
    _, cp, rv, nz = csc1(A)
    dt = np.float64 if precision == "fp64" else np.float32
    op = orc.factor_csc(sym, cp, rv, nz, dt)[2]
    assert np.array_equal(ipiv, op)
