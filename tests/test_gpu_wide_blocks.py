"""SPD blocks wider than 64 columns (pieces up to 96) followed by narrower ones
in the same group: the narrower block's diagonal region takes the wide one's
product, all of its columns. Dense matrices, one front each, with pieces of at
most 80 columns: 460 columns split into six blocks of 68 and one of 52, 329
and 333 into blocks of 64 to 75. The matrices and the bound on the factor
multiplied out are those of test_gpu_update_sums."""
import numpy as np
import pytest
import scipy.sparse as sp

from helpers import panels_to_dense
from sparspak_hip import SparseSpdSolver, factor, findorderperm, inmatrix, symbolicfactor
from test_gpu_update_sums import _excess, _matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [329, 333, 460])
def test_wide_block_before_a_narrow_one(n, precision):
    print(f"case wide block n={n} {precision}", flush=True)
    A = _matrix(n, True)
    s = SparseSpdSolver(sp.csc_matrix(A))
    s.slvr.sym.maxblocksize = 80
    findorderperm(s, np.arange(1, n + 1))
    symbolicfactor(s)
    w = np.diff(s.slvr.sym.xsuper)
    assert any(a > 64 and b <= 64 for a, b in zip(w[:-1], w[1:]))
    inmatrix(s)
    factor(s, precision)
    L = np.tril(panels_to_dense(s.slvr.sym, s.slvr.download()[0], None))
    D = L + np.triu(L.T * np.diag(L)[:, None], 1)
    assert _excess(A, D, precision) <= 1.0
