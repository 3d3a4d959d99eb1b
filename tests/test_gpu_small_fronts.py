"""Small fronts (at most 64 rows) at the edges of their thread grids (8 and
16) and of the one-wave limit (32 rows): leaves of W columns and R update
rows on a shared root of 24 columns, natural order, so that every leaf is a
front of W + R rows and the root sums all of their update matrices. LU rows
are a diagonally dominant matrix's with the rows of each leaf's piece
reversed: its steps interchange rows, and the elimination does
not grow (dominant by columns after the interchanges: multipliers at most 1,
entries at most twice the largest of A). Each entry sums at most 64 products
from its own front and 24 x 19 leaves' worth below it, so it differs from the
oracle's (double) by at most about 2 (64 + 19) of its largest terms' roundings:
the bound is 8 x 128 units of the largest entry. One group per front in both
forms: small_wave_min 1 gives every front one wave."""
import numpy as np
import pytest
import scipy.sparse as sp

import oracle.oracle as orc
from helpers import csc1, spd_meaningful
from sparspak_hip import (SparseSolver, SparseSpdSolver, factor, findorderperm, inmatrix,
                          symbolicfactor)

pytestmark = pytest.mark.gpu

ROOT = 24
# (W, R) of the leaves: W + R = 1 .. 64 around 8, 16, 32 and 64 rows
LEAVES = [(1, 1), (1, 24), (2, 5), (7, 1), (8, 0), (5, 4), (8, 8), (9, 8), (16, 15), (8, 24),
          (31, 1), (32, 0), (9, 24), (32, 1), (30, 24), (39, 24), (40, 24), (63, 1), (64, 0)]


def _matrix(spd):
    rng = np.random.default_rng(77)
    n = sum(w for w, _ in LEAVES) + ROOT
    M = np.zeros((n, n))
    c0, r0 = 0, n - ROOT
    M[r0:, r0:] = rng.uniform(-1, 1, (ROOT, ROOT))
    for w, r in LEAVES:
        own = np.arange(c0, c0 + w)
        idx = np.concatenate([own, np.arange(r0, r0 + r)])
        M[np.ix_(own, idx)] = rng.uniform(-1, 1, (w, w + r))
        M[np.ix_(idx, own)] = rng.uniform(-1, 1, (w + r, w))
        c0 += w
    if spd:
        M = (M + M.T) / 2
    np.fill_diagonal(M, 0.0)
    off = np.abs(M).sum(axis=0) + np.abs(M).sum(axis=1)
    np.fill_diagonal(M, (off + 1.0) * (1.0 if spd else 1.5))
    return M


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("wave_min", [16384, 1])
@pytest.mark.parametrize("spd", [False, True])
def test_small_fronts_match_oracle(spd, wave_min, precision):
    print(f"case small fronts spd={spd} wave_min={wave_min} {precision}", flush=True)
    M = _matrix(spd)
    n = M.shape[0]
    cls = SparseSpdSolver if spd else SparseSolver

    def prepared(A):
        s = cls(sp.csc_matrix(A))
        findorderperm(s, np.arange(1, n + 1))
        symbolicfactor(s)
        return s

    s = prepared(M)
    xs = np.asarray(s.slvr.sym.xsuper) - 1
    if not spd:  # the pattern is unchanged: rows of a leaf's piece share it
        P = M.copy()
        old = np.asarray(s.slvr.sym.order.rperm) - 1
        for a, b in zip(xs[:-1], xs[1:]):
            if old[a:b].max() < n - ROOT:
                P[old[a:b]] = M[old[a:b][::-1]]
        s = prepared(P)
        assert np.array_equal(np.asarray(s.slvr.sym.xsuper) - 1, xs)
        M = P
    inmatrix(s)
    s.slvr.set_tuning(small_wave_min=wave_min)
    factor(s, precision)
    lnz, unz, ipiv = s.slvr.download()
    _, cp, rv, nz = csc1(sp.csc_matrix(M))
    tol = 8 * 128 * (2.0 ** -53 if precision == "fp64" else 2.0 ** -24)
    if spd:
        ol, _, _ = orc.inmatrix(s.slvr.sym, cp, rv, nz)
        orc.ldltfactor(s.slvr.sym, ol)
        m = spd_meaningful(s.slvr.sym)
        assert np.max(np.abs(lnz - ol)[m]) <= tol * np.max(np.abs(ol[m]))
    else:
        ol, ou, op, rc, _ = orc.factor_csc(s.slvr.sym, cp, rv, nz)
        assert rc == 0
        assert np.array_equal(ipiv, op)
        assert np.max(np.abs(lnz - ol)) <= tol * np.max(np.abs(ol))
        assert np.max(np.abs(unz - ou)) <= tol * max(np.max(np.abs(ol)), np.max(np.abs(ou)))
