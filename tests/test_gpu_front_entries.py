"""A's entries added by the front assembly of the handle (small fronts, large
fronts' columns summed in LDS or in place) against the drop-ins that factor
assembled lnz/unz (SparseCSCInterface.jl:112-163, then SpkLUFactor.jl:178-302
or SpkLDLtFactor.jl:33-118). Both add the same numbers in the same order, so
factors, pivots and LDL^T entries are equal in every bit. Sizes: one small
front, fronts around the small limit (64 rows), columns on either side of the
one-wave limit (16 KB: 2048 doubles, 4096 floats) and past the LDS limit
(64 KB: 8192 doubles), each with children whose rows coincide; unsymmetric
patterns, explicitly stored zeros and SPD input with both triangles."""
import numpy as np
import pytest
import scipy.sparse as sp

import oracle.oracle as orc
from helpers import csc1, random_pattern
from sparspak_hip import (SparseSolver, SparseSpdSolver, _lib, factor, findorder, findorderperm,
                          inmatrix, symbolicfactor)
from sparspak_hip.gallery import convdiff3d, elasticity3d

pytestmark = pytest.mark.gpu


def _arrow(m, spd):
    """Three leaves on random halves of a core of m columns whose first column
    is full: in natural order one front of m rows with three children."""
    rng = np.random.default_rng(m)
    n = m + 3
    M = sp.lil_matrix((n, n))
    for c in range(4):
        half = np.append(True, rng.random(m - 1) < 0.5)
        rows = np.arange(4, n) if c == 3 else 3 + np.flatnonzero(half)
        M[rows, c] = rng.uniform(-1, 1, (rows.size, 1))
        M[c, rows] = M[rows, c].T if spd else rng.uniform(-1, 1, (1, rows.size))
    return sp.csc_matrix(M + sp.diags(np.full(n, 2.0 * m)))


def _unsym():
    A = random_pattern(90, 0.03, 4, symmetric=False)
    off = np.flatnonzero(A.indices != np.repeat(np.arange(90), np.diff(A.indptr)))
    A.data[off[3::7]] = 0.0  # stored zeros keep their slot
    return A


CASES = {"one_small": (_unsym, SparseSolver, False),
         "convdiff3d_9": (lambda: convdiff3d(9), SparseSolver, False),
         "elasticity3d_5": (lambda: elasticity3d(5), SparseSpdSolver, False),
         "arrow_61": (lambda: _arrow(61, False), SparseSolver, True),
         "arrow_62_spd": (lambda: _arrow(62, True), SparseSpdSolver, True),
         "arrow_2048": (lambda: _arrow(2048, False), SparseSolver, True),
         "arrow_2049_spd": (lambda: _arrow(2049, True), SparseSpdSolver, True),
         "arrow_4097": (lambda: _arrow(4097, False), SparseSolver, True),
         "arrow_8193": (lambda: _arrow(8193, False), SparseSolver, True)}


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("name", list(CASES))
def test_front_entries_match_assembled_panels(name, precision):
    print(f"case front entries {name} {precision}", flush=True)
    gen, cls, natural = CASES[name]
    A = sp.csc_matrix(gen())
    s = cls(A)
    if natural:
        findorderperm(s, np.arange(1, A.shape[0] + 1))
    else:
        findorder(s)
    symbolicfactor(s)
    inmatrix(s)
    factor(s, precision)
    lnz, unz, ipiv = s.slvr.download()
    sym = s.slvr.sym
    n, cp, rv, nz = csc1(A)
    gl, gu, gp = orc.inmatrix(sym, cp, rv, nz)
    dt, P = (np.float64, _lib.pd) if precision == "fp64" else (np.float32, _lib.pf)
    gl = gl.astype(dt)
    L, I = _lib.lib(), _lib.p64
    suffix = "f64" if precision == "fp64" else "f32"
    if cls is SparseSolver:
        gu = gu.astype(dt)
        rc = getattr(L, "spkhip_lufactor_" + suffix)(
            n, sym.nsuper, I(sym.xsuper), I(sym.snode), I(sym.xlindx), I(sym.lindx),
            I(sym.xlnz), P(gl), I(sym.xunz), P(gu), I(gp))
        assert rc == 0
        assert np.array_equal(ipiv, gp)
        assert np.array_equal(np.asarray(unz, dtype=dt), gu)
    else:
        rc = getattr(L, "spkhip_ldltfactor_" + suffix)(
            n, sym.nsuper, I(sym.xsuper), I(sym.snode), I(sym.xlindx), I(sym.lindx),
            I(sym.xlnz), P(gl))
        assert rc == 0
    assert np.array_equal(np.asarray(lnz, dtype=dt), gl)
