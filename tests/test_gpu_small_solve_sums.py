"""The order of the sums in the solves of small fronts (at most 64 rows): as
the reference does (SpkLUFactor.jl:269-377), the products of a piece's columns
with a row below it, and of a row with the columns right of its piece, are
summed from zero and subtracted once. Unit triangular blocks whose
off-diagonal entries are half a unit in the last place below one, so that each
product alone leaves an entry of one unchanged and only their sum is felt; all
sums are exact, so the solution is known bit for bit. Blocks split into
pieces, at sizes that take every form of the kernels (a workgroup, a wave, a
part of a wave with 8192 units or more; one, up to four and more right-hand
sides), fronts with update rows among them."""
import numpy as np
import pytest
import scipy.sparse as sp

from sparspak_hip import (SparseSolver, factor, findorderperm, inmatrix, symbolicfactor,
                          triangularsolve)

pytestmark = pytest.mark.gpu

# block size, most columns of a piece, blocks, right-hand sides
CASES = [(8, 4, 3, 1), (8, 4, 3, 3), (16, 8, 3, 1), (16, 6, 3, 6), (32, 16, 3, 1), (32, 10, 3, 4),
         (32, 16, 3, 6), (64, 30, 2, 1), (64, 16, 2, 3), (64, 30, 2, 9), (8, 4, 2100, 4),
         (16, 8, 2100, 4)]


def _solver(M, count, mb, precision):
    n = M.shape[0]
    r, c = np.nonzero(np.ones((n, n)))
    A = sp.csc_matrix((np.tile(M.T.ravel(), count),
                       (np.arange(count)[:, None] * n + np.tile(np.arange(n), n)).ravel(),
                       np.arange(n * count + 1) * n), shape=(n * count, n * count))
    s = SparseSolver(A)
    s.slvr.sym.maxblocksize = mb
    findorderperm(s, np.arange(1, n * count + 1))
    symbolicfactor(s)
    xs = np.asarray(s.slvr.sym.xsuper) - 1
    assert len(xs) > 2 * count  # at least two pieces per block
    inmatrix(s)
    factor(s, precision)
    return s, xs[xs <= n]


def _same(s, n, count, nrhs, want):
    x = np.ones((n * count, nrhs), order="F")
    triangularsolve(s, x, refine=False)
    assert np.array_equal(x, np.tile(want, count)[:, None].repeat(nrhs, 1))


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n,mb,count,nrhs", CASES)
def test_forward_sums_a_piece(n, mb, count, nrhs, precision):
    print(f"case forward sums n={n} mb={mb} count={count} nrhs={nrhs} {precision}", flush=True)
    dt = np.float64 if precision == "fp64" else np.float32
    e = 2.0 ** (-54 if precision == "fp64" else -25)
    M = np.eye(n)
    M[-1, :-1] = e
    s, xs = _solver(M, count, mb, precision)
    want = np.ones(n)
    y = dt(1.0)
    for a, b in zip(xs[:-2], xs[1:-1]):
        y = dt(y - dt((b - a) * e))
    for _ in range(xs[-2], n - 1):  # inside its own piece one by one
        y = dt(y - dt(e))
    want[-1] = y
    assert y != 1.0
    _same(s, n, count, nrhs, want)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n,mb,count,nrhs", CASES)
def test_backward_sums_right_of_a_piece(n, mb, count, nrhs, precision):
    print(f"case backward sums n={n} mb={mb} count={count} nrhs={nrhs} {precision}", flush=True)
    dt = np.float64 if precision == "fp64" else np.float32
    e = 2.0 ** (-54 if precision == "fp64" else -25)
    M = np.eye(n)
    M[0, 1:] = e
    s, xs = _solver(M, count, mb, precision)
    y = dt(dt(1.0) - dt((n - xs[1]) * e))
    for _ in range(1, xs[1]):
        y = dt(y - dt(e))
    want = np.ones(n)
    want[0] = y
    assert y != 1.0
    _same(s, n, count, nrhs, want)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("w,r,nrhs", [(2, 5, 1), (5, 9, 3), (8, 20, 1), (6, 20, 6), (24, 30, 1),
                                      (24, 40, 4), (20, 30, 7)])
def test_backward_sums_update_rows(w, r, nrhs, precision):
    print(f"case backward update rows w={w} r={r} nrhs={nrhs} {precision}", flush=True)
    dt = np.float64 if precision == "fp64" else np.float32
    e = 2.0 ** (-54 if precision == "fp64" else -25)
    n = 2 * w + r
    M = np.zeros((n, n))
    P = np.zeros((n, n), dtype=bool)
    P[2 * w:, 2 * w:] = True
    for a in (0, w):  # two leaves of w columns on a root of r
        P[a:a + w, a:a + w] = P[a:a + w, 2 * w:] = P[2 * w:, a:a + w] = True
    M[0, 2 * w:] = e  # the first leaf: a front of w columns and r update rows
    np.fill_diagonal(M, 1.0)
    c, rows = np.nonzero(P.T)
    A = sp.csc_matrix((M[rows, c], rows, np.r_[0, np.cumsum(P.sum(axis=0))]), shape=(n, n))
    s = SparseSolver(A)
    findorderperm(s, np.arange(1, n + 1))
    symbolicfactor(s)
    sym = s.slvr.sym
    assert sym.xsuper[1] - 1 == w and sym.xlindx[1] - 1 == w + r
    inmatrix(s)
    factor(s, precision)
    x = np.ones((n, nrhs), order="F")
    triangularsolve(s, x, refine=False)
    want = np.ones(n)
    want[0] = dt(dt(1.0) - dt(r * e))
    assert want[0] != 1.0
    assert np.array_equal(x, want[:, None].repeat(nrhs, 1))
