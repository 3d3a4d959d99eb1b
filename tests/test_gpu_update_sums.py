"""The trailing update's products at the edges of its 64 x 64 tiles and of its
chunks of the inner dimension (16, or 32 with 16-bit operands), on matrices
whose updates are as large as their entries: A = L U with L(i, k) = s_i a_k
and U(k, j) = t_j b_k off the diagonals, so that an entry's updates all have
one sign and sum to about 4 min(i, j) / n of its s_i t_j. Dense, one front each;
the magnitudes of s, t, a, b are random (the 16-bit operands are rounded),
the signs of s and t agree, so that pivots stay the diagonal's.

The factor is multiplied out and held, entry by entry, to Gaussian
elimination's bound |A - L U| <= (c n eps + 2 u + u^2) |L| |U| (Higham,
Accuracy and Stability, 9.3) with c = 8 and u the unit rounding of the
update's operands (fronts of more than 256 columns): 2^-8 (bf16), 2^-11
(fp16), and 3 2^-16 in all for split bf16, whose products leave out lo lo.
The CPU test below checks what the bound can see: a factor whose updates skip
one chunk of the inner dimension, its last columns, one row or one column of
an edge tile breaks it in every precision."""
import numpy as np
import pytest
import scipy.sparse as sp

from helpers import csc1, panels_to_dense
from sparspak_hip import (SparseSolver, SparseSpdSolver, factor, findorderperm, inmatrix,
                          symbolicfactor)

PREC = ["fp64", "fp32", "fp32_bf16", "fp32_fp16", "fp32_bf16x3"]
SIZES = [61, 125, 188, 257, 545, 607]


def _matrix(n, spd):
    rng = np.random.default_rng(n)
    sign = rng.choice([-1.0, 1.0], n)

    def mag():
        return rng.uniform(0.6, 1.0, n)

    s, a = sign * mag(), mag() * np.sqrt(6.0 / n)
    t, b = (s, a) if spd else (sign * mag(), mag() * np.sqrt(6.0 / n))
    L = np.tril(np.outer(s, a), -1) + np.eye(n)
    U = np.triu(np.outer(b, t), 1) + np.eye(n)
    return L @ U


def _bound(n, precision):
    u = {"fp32_bf16": 2.0 ** -7 + 2.0 ** -16, "fp32_fp16": 2.0 ** -10 + 2.0 ** -22,
         "fp32_bf16x3": 3 * 2.0 ** -16}.get(precision, 0.0)
    eps = 2.0 ** -53 if precision == "fp64" else 2.0 ** -24
    return 8 * n * eps + (u if n > 256 else 0.0)


def _excess(A, D, precision):
    """Largest |A - L U| over its bound."""
    n = A.shape[0]
    L, U = np.tril(D, -1) + np.eye(n), np.triu(D)
    return np.max(np.abs(A - L @ U) / (np.abs(L) @ np.abs(U))) / _bound(n, precision)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", PREC)
@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("spd", [False, True])
def test_updates_sum_every_product(n, precision, spd):
    print(f"case update sums n={n} {precision} spd={spd}", flush=True)
    A = _matrix(n, spd)
    s = (SparseSpdSolver if spd else SparseSolver)(sp.csc_matrix(A))
    findorderperm(s, np.arange(1, n + 1))
    symbolicfactor(s)
    inmatrix(s)
    factor(s, precision)
    lnz, unz, ipiv = s.slvr.download()
    sym = s.slvr.sym
    assert np.array_equal(sym.order.rperm, np.arange(1, n + 1))
    if spd:
        L = np.tril(panels_to_dense(sym, lnz, None))
        D = L + np.triu(L.T * np.diag(L)[:, None], 1)
    else:
        D = panels_to_dense(sym, lnz, unz)
        assert np.array_equal(ipiv, np.arange(n) - np.repeat(sym.xsuper[:-1] - 1,
                                                             np.diff(sym.xsuper)) + 1)
    assert _excess(A, D, precision) <= 1.0


def _factor(A, skip):
    """LU whose step k updates the trailing matrix but for skip(k, M)."""
    M = A.copy()
    for k in range(A.shape[0] - 1):
        M[k + 1:, k] /= M[k, k]
        P = np.outer(M[k + 1:, k], M[k, k + 1:])
        skip(k, P)
        M[k + 1:, k + 1:] -= P
    return M


@pytest.mark.parametrize("precision", PREC)
@pytest.mark.parametrize("n", [125, 607])
@pytest.mark.parametrize("spd", [False, True])
def test_bound_sees_missing_products(n, precision, spd):
    A = _matrix(n, spd)
    assert _excess(A, _factor(A, lambda k, P: None), precision) <= 1.0

    def missing(rows, cols, ks):
        def skip(k, P):
            if k in ks:
                r, c = rows - k - 1, cols - k - 1
                P[np.ix_(r[r >= 0], c[c >= 0])] = 0.0
        return skip

    every, tail = np.arange(n), np.arange(64 * ((n - 1) // 64), n)
    first = range(0, 60)  # the first block group's columns, or the first block's
    for rows, cols, ks in [
            (np.arange(60, n), np.arange(60, n), range(0, 32)),   # one chunk of 32
            (np.arange(60, n), np.arange(60, n), range(32, 60)),  # a tail of 28
            (every[-1:], np.arange(60, n), first),                # the last row
            (np.arange(60, n), every[-1:], first),                # the last column
            (tail, tail, first)]:                                 # the corner tile
        D = _factor(A, missing(rows, cols, ks))
        assert _excess(A, D, precision) > 1.0
