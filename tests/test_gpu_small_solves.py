"""Solves through small fronts (at most 64 rows) at the edges of the one-wave
limit and of the register blocks of right-hand sides (1, 4, 16): the matrices
of test_gpu_small_fronts (fronts of 1 to 64 rows, row interchanges inside
pieces), a general sparse one, and one of many small blocks, whose
right-hand sides change the form that its fronts of at most 16 rows take. The solution of every right-hand side
equals that of its own solve bit for bit, and its backward error is within
that of a substitution with an LU factor that does not grow (entries at most
twice those of A): n eps with a factor of 8 for the two sweeps."""
import numpy as np
import pytest
import scipy.sparse as sp

from helpers import backward_error, random_pattern
from sparspak_hip import (SparseSolver, SparseSpdSolver, factor, findorder, findorderperm,
                          inmatrix, symbolicfactor, triangularsolve)
from sparspak_hip.gallery import uniform
from test_gpu_small_fronts import ROOT, _matrix

pytestmark = pytest.mark.gpu


def _solver(kind):
    if kind in ("sparse", "many"):
        A = random_pattern(160, 0.012, 5, symmetric=False)
        if kind == "many":
            rng = np.random.default_rng(9)
            A = sp.block_diag([np.diag(np.full(w, 2.0 * w)) + rng.uniform(-1, 1, (w, w))
                               for w in [3, 8, 9, 16, 5] * 120], format="csc")
        s = SparseSolver(A)
        findorder(s)
        symbolicfactor(s)
    else:
        M = _matrix(kind == "spd")
        n = M.shape[0]
        cls = SparseSpdSolver if kind == "spd" else SparseSolver
        s = cls(sp.csc_matrix(M))
        findorderperm(s, np.arange(1, n + 1))
        symbolicfactor(s)
        if kind == "lu":
            xs = np.asarray(s.slvr.sym.xsuper) - 1
            old = np.asarray(s.slvr.sym.order.rperm) - 1
            P = M.copy()
            for a, b in zip(xs[:-1], xs[1:]):
                if old[a:b].max() < n - ROOT:
                    P[old[a:b]] = M[old[a:b][::-1]]
            M = P
            s = cls(sp.csc_matrix(M))
            findorderperm(s, np.arange(1, n + 1))
            symbolicfactor(s)
        A = sp.csc_matrix(M)
    inmatrix(s)
    return A, s


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", ["lu", "spd", "sparse", "many"])
def test_small_front_solves(kind, precision):
    A, s = _solver(kind)
    n = A.shape[0]
    factor(s, precision)
    eps = 2.0 ** -53 if precision == "fp64" else 2.0 ** -24
    B = np.asfortranarray(np.stack([uniform(400 + q, n, -1.0, 1.0) for q in range(17)], axis=1))
    single = []
    for q in range(17):
        x = B[:, q].copy()
        triangularsolve(s, x, refine=False)
        assert backward_error(A, x, B[:, q]) <= 8 * n * eps
        single.append(x)
    for nrhs in (2, 4, 5, 16, 17):
        print(f"case small solves {kind} {precision} nrhs={nrhs}", flush=True)
        X = np.array(B[:, :nrhs], order="F")
        triangularsolve(s, X, refine=False)
        for q in range(nrhs):
            assert np.array_equal(X[:, q], single[q]), f"right-hand side {q} of {nrhs}"
