"""The pivot search of small fronts (at most 64 rows) where the leading 32
bits of the candidates' magnitudes agree, in each of its thread grids (6 to 64
rows; one wave per front with small_wave_min 1): a piece's first column whose
entries differ in the low half of the double only, tie exactly (the smallest
position wins) or tie up to sign, and a column that holds NaN (a NaN in the
first row keeps the row, others are passed over: the comparisons of ggetrf!,
GenericBlasLapackFragments.jl:56-100, are false). The other columns hold
their diagonal only, so the interchanges do not depend on rounding: they equal
the oracle's (with NaN, which spreads, those of the first column)."""
import numpy as np
import pytest
import scipy.sparse as sp

import oracle.oracle as orc
from helpers import csc1
from sparspak_hip import SparseSolver, factor, findorderperm, inmatrix, symbolicfactor

pytestmark = pytest.mark.gpu

KINDS = ["low", "equal", "sign", "low_descending", "nan_first", "nan_inside"]


def _column(kind, n, rng):
    if kind == "low":
        return 16.0 + rng.permutation(n) * 2.0 ** -40
    if kind == "low_descending":
        return 16.0 - np.arange(n) * 2.0 ** -40
    if kind == "sign":
        return 16.0 * rng.choice([-1.0, 1.0], n)
    col = np.full(n, 16.0)
    if kind == "nan_first":
        col[0] = np.nan
    elif kind == "nan_inside":
        col = 16.0 + np.arange(n)
        col[n // 2:] = np.nan
    return col


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("wave_min", [16384, 1])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n", [6, 12, 24, 31, 40, 64])
def test_small_front_ties(n, kind, wave_min, precision):
    print(f"case small ties n={n} {kind} {wave_min} {precision}", flush=True)
    rng = np.random.default_rng(n)
    M = np.diag(rng.uniform(1, 2, n))
    idx = np.tile(np.arange(n), n)

    def prepared():  # every entry stored: one dense front
        s = SparseSolver(sp.csc_matrix((M.T.ravel(), idx, np.arange(n + 1) * n), shape=(n, n)))
        findorderperm(s, np.arange(1, n + 1))
        symbolicfactor(s)
        return s

    xs = np.asarray(prepared().slvr.sym.xsuper) - 1
    nan = kind.startswith("nan")
    for a, b in list(zip(xs[:-1], xs[1:]))[:1 if nan else None]:
        M[a:b, a] = _column(kind, b - a, rng)
    s = prepared()
    inmatrix(s)
    s.slvr.set_tuning(small_wave_min=wave_min)
    factor(s, precision)
    _, _, ipiv = s.slvr.download()
    _, cp, rv, nz = csc1(sp.csc_matrix((M.T.ravel(), idx, np.arange(n + 1) * n), shape=(n, n)))
    dt = np.float64 if precision == "fp64" else np.float32
    op = orc.factor_csc(s.slvr.sym, cp, rv, nz, dt)[2]
    if nan:
        assert ipiv[0] == op[0] == (1 if kind == "nan_first" else xs[1] // 2)
    else:
        assert np.array_equal(ipiv, op)
