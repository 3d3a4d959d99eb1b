"""The trailing update at the edges of its 64 x 64 tiles and of its chunks of
the inner dimension (16, or 32 with 16-bit operands): dense diagonally
dominant matrices, one front each, whose updates leave remainders of one row,
a full tile and one row less, with one block group (n <= 480) and a second
one. Against the oracle in double: every entry within the rounding of its
products. With |l| <= 1/2 summed over a row (dominance), an update's products
sum to at most the largest entry, so an operand rounding of u per factor and
an accumulation of k terms in eps give at most 2 u + k eps per level of the
elimination, relative to the largest entry."""
import numpy as np
import pytest
import scipy.sparse as sp

import oracle.oracle as orc
from helpers import csc1, spd_meaningful
from sparspak_hip import (SparseSolver, SparseSpdSolver, factor, findorder, inmatrix,
                          symbolicfactor)

pytestmark = pytest.mark.gpu

# unit roundings of the update's operands and accumulation
TOL = {"fp64": lambda n: 4 * n * 2.0 ** -53, "fp32": lambda n: 4 * n * 2.0 ** -24,
       "fp32_bf16": lambda n: 2.0 ** -6 + 4 * n * 2.0 ** -24,
       "fp32_fp16": lambda n: 2.0 ** -9 + 4 * n * 2.0 ** -24,
       "fp32_bf16x3": lambda n: 2.0 ** -14 + 4 * n * 2.0 ** -24}


def _dense(n, spd):
    rng = np.random.default_rng(n)
    M = rng.uniform(-1, 1, (n, n)) / (2 * n)
    if spd:
        M = (M + M.T) / 2
    return sp.csc_matrix(M + np.diag(rng.uniform(1, 2, n)))


@pytest.mark.parametrize("precision", list(TOL))
@pytest.mark.parametrize("n", [61, 125, 188, 257, 545, 607])
@pytest.mark.parametrize("spd", [False, True])
def test_update_tile_edges(n, precision, spd):
    print(f"case n={n} {precision} spd={spd}", flush=True)
    A = _dense(n, spd)
    s = (SparseSpdSolver if spd else SparseSolver)(A)
    findorder(s)
    symbolicfactor(s)
    inmatrix(s)
    factor(s, precision)
    lnz, unz, ipiv = s.slvr.download()
    nn, cp, rv, nz = csc1(A)
    if spd:
        ol, _, _ = orc.inmatrix(s.slvr.sym, cp, rv, nz)
        orc.ldltfactor(s.slvr.sym, ol)
        m = spd_meaningful(s.slvr.sym)
        assert np.max(np.abs(lnz - ol)[m]) <= TOL[precision](n) * np.max(np.abs(ol[m]))
    else:
        ol, ou, op, rc, _ = orc.factor_csc(s.slvr.sym, cp, rv, nz)
        assert rc == 0 and np.array_equal(ipiv, op)
        big = max(np.max(np.abs(ol)), np.max(np.abs(ou)) if ou.size else 0.0)
        assert np.max(np.abs(lnz - ol)) <= TOL[precision](n) * big
        if ou.size:
            assert np.max(np.abs(unz - ou)) <= TOL[precision](n) * big
