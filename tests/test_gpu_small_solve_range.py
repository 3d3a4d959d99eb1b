"""Backward solves of small fronts (at most 64 rows) where the reciprocal of a
pivot, or the quotient itself, leaves the type's range: the reference divides
(gtrsm!), so a subnormal pivot whose reciprocal overflows still gives the
finite quotient, and an infinite right-hand side an infinite one. Dense upper
triangular blocks with unit diagonals and a last pivot of 2^-140 (float) or
2^-1050 (double); the right-hand sides are chosen so that every product and
sum is exact, so the solution is known bit for bit. Blocks of 1 to 64 rows
take every form of the kernel (a workgroup, a wave, a part of a wave with 8192
units or more; one, up to four and more right-hand sides)."""
import numpy as np
import pytest
import scipy.sparse as sp

from sparspak_hip import (SparseSolver, factor, findorderperm, inmatrix, symbolicfactor,
                          triangularsolve)

pytestmark = pytest.mark.gpu


def _blocks(n, count, last):
    """count dense upper triangular n x n blocks (all entries stored)."""
    M = np.eye(n)
    M[:-1, -1] = 0.5
    M[-1, -1] = last
    i = np.tile(np.arange(n), n)
    rows = (np.arange(count)[:, None] * n + i).ravel()
    return sp.csc_matrix((np.tile(M.T.ravel(), count), rows, np.arange(n * count + 1) * n),
                         shape=(n * count, n * count))


def _solver(A, precision):
    s = SparseSolver(A)
    findorderperm(s, np.arange(1, A.shape[0] + 1))
    symbolicfactor(s)
    inmatrix(s)
    factor(s, precision)
    return s


# 8192 units (blocks and right-hand sides) take parts of a wave per front
CASES = [(1, 3, 1), (6, 3, 1), (12, 3, 4), (24, 5, 1), (24, 5, 4), (24, 5, 7), (40, 3, 1),
         (40, 3, 4), (64, 2, 9), (6, 2100, 4), (12, 2100, 4)]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n,count,nrhs", CASES)
def test_subnormal_pivot(n, count, nrhs, precision):
    print(f"case subnormal pivot n={n} count={count} nrhs={nrhs} {precision}", flush=True)
    tiny = 2.0 ** (-1050 if precision == "fp64" else -140)
    s = _solver(_blocks(n, count, tiny), precision)
    # x_last = 2 k, the others k + 1 .. from b = x + x_last / 2; and the block
    # before the last with a zero entry there
    X = np.empty((n, count, nrhs))
    X[:] = np.arange(1.0, n + 1)[:, None, None] + np.arange(nrhs)
    X[-1] = 2.0 * (1 + np.arange(count) % 5)[:, None]
    X[-1, -1] = 0.0
    B = X.copy()
    B[:-1] += 0.5 * X[-1]
    B[-1] = X[-1] * tiny
    x = np.asfortranarray(B.transpose(1, 0, 2).reshape(n * count, nrhs))
    triangularsolve(s, x, refine=False)
    assert np.array_equal(x, X.transpose(1, 0, 2).reshape(n * count, nrhs))


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n,count,nrhs", CASES)
def test_infinite_quotients(n, count, nrhs, precision):
    print(f"case infinite quotient n={n} count={count} nrhs={nrhs} {precision}", flush=True)
    s = _solver(_blocks(n, count, 0.25), precision)
    big = 2.0 ** (1023 if precision == "fp64" else 127)
    B = np.ones((count, n, nrhs))
    B[0, -1] = np.inf
    B[1, -1] = -big  # overflows when divided by 1 / 4
    x = np.asfortranarray(B.reshape(n * count, nrhs))
    triangularsolve(s, x, refine=False)
    x = x.reshape(count, n, nrhs)
    assert np.all(x[0, -1] == np.inf) and np.all(x[1, -1] == -np.inf)
    if count > 2:  # the other blocks are not touched
        assert np.all(x[2:, -1] == 4.0) and np.all(x[2:, :-1] == -1.0)
