"""The off-diagonal solves of factor blocks of at most 64 columns at the edges
of their 16-column sub-blocks and 64-row tiles: dense matrices, one front
each, split into pieces of 5 to 60 columns (blocks of 40, 48, 51, 60 and 64
columns, several pieces per block, last blocks of one column up), with one
row up to a full tile of rows left below the last full tile, pivoting inside
the pieces (LU) or none (SPD).

The factor is multiplied out again in 80 bits, piece by piece from the last,
and held to the componentwise bound of Gaussian elimination by substitution,
|A - L U| <= c n eps |L| |U| (Higham, Accuracy and Stability, 9.3) with c = 4,
which holds whatever the growth (pivoting confined to pieces of five columns
lets these matrices grow by many orders, so entries of two correct factors
need not agree closely). The SPD factor also agrees with the oracle's within
4 n eps of its largest entry (diagonally dominant: no growth)."""
import numpy as np
import pytest
import scipy.sparse as sp

import oracle.oracle as orc
from helpers import csc1, panels_to_dense, spd_meaningful
from sparspak_hip import (SparseSolver, SparseSpdSolver, factor, findorder, inmatrix,
                          symbolicfactor)

pytestmark = pytest.mark.gpu


def _multiply_out(sym, D, ipiv):
    """(L U with every piece's interchanges undone, the same of |L| |U|)."""
    n = sym.n
    S, B = D.copy(), np.abs(D)
    for J in range(sym.nsuper - 1, -1, -1):
        f, l = sym.xsuper[J] - 1, sym.xsuper[J + 1] - 1
        for out, M in ((S, D), (B, np.abs(D))):
            low = np.tril(M[f:, f:l], -1)
            low[np.arange(l - f), np.arange(l - f)] = 1
            up = np.triu(M[f:l, f:])
            new = low @ up
            new[l - f:, l - f:] += out[l:, l:]
            for k in range(l - 1, f - 1, -1):
                kp = int(ipiv[k]) - 1
                new[[k - f, kp]] = new[[kp, k - f]]
            out[f:, f:] = new
    return S, B


@pytest.mark.parametrize("n", [65, 66, 113, 129, 195])
@pytest.mark.parametrize("width", [5, 16, 17, 30, 60])
@pytest.mark.parametrize("spd", [False, True])
def test_offdiag_block_edges(n, width, spd):
    print(f"case n={n} width={width} spd={spd}", flush=True)
    rng = np.random.default_rng(100 * n + width)
    M = rng.uniform(-1, 1, (n, n))
    if spd:
        M = (M + M.T) / 2 + n * np.eye(n)
    else:
        M += 2 * np.eye(n)
    A = sp.csc_matrix(M)
    s = (SparseSpdSolver if spd else SparseSolver)(A)
    if spd or width <= 30:
        s.slvr.sym.maxblocksize = width
    findorder(s)
    symbolicfactor(s)
    inmatrix(s)
    factor(s, "fp64")
    lnz, unz, ipiv = s.slvr.download()
    sym = s.slvr.sym
    p = sym.order.rperm - 1
    Ap = M[np.ix_(p, p)].astype(np.longdouble)
    if spd:
        _, cp, rv, nz = csc1(A)
        ol, _, _ = orc.inmatrix(sym, cp, rv, nz)
        orc.ldltfactor(sym, ol)
        m = spd_meaningful(sym)
        assert np.max(np.abs(lnz - ol)[m]) <= 4 * n * 2.0 ** -53 * np.max(np.abs(ol[m]))
        return
    S, B = _multiply_out(sym, panels_to_dense(sym, lnz, unz).astype(np.longdouble), ipiv)
    assert np.all(np.abs(Ap - S) <= 4 * n * 2.0 ** -53 * B)
