"""The block products of the large fronts' solves with eight rows and eight
right-hand sides per workgroup (launches of at least 8192 rows) against one
row per workgroup: 80 value sets of one pattern whose top front has more than
256 columns, so that blocks end in remainders of eight rows, solved for 1, 7,
8 and 17 right-hand sides. Every set's solution equals that of a handle that
holds the set alone (far fewer rows per launch), bit for bit."""
import numpy as np
import pytest
import scipy.sparse as sp

from sparspak_hip.batch import BatchedSolver
from sparspak_hip.gallery import uniform

pytestmark = pytest.mark.gpu

NSETS = 80


def _sets(kind):
    n, w = 301, 40
    rng = np.random.default_rng(31)
    P = np.ones((n, n), dtype=bool)
    P[:w, w:2 * w] = P[w:2 * w, :w] = False  # two children under a dense front
    out = []
    for _ in range(NSETS):
        M = rng.uniform(-1, 1, (n, n)) * P
        if kind == "spd":
            M = (M + M.T) / 2
        out.append(sp.csc_matrix(M + 2 * n * np.eye(n)))
    return out


@pytest.mark.parametrize("kind", ["lu", "spd"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_row_groups_equal_single_rows(kind, precision):
    mats = _sets(kind)
    n = mats[0].shape[0]
    vs = BatchedSolver(mats, kind=kind)
    assert vs.value_sets
    vs.set_values()
    vs.factor(precision)
    one = {}
    for v in (0, 41, NSETS - 1):
        one[v] = BatchedSolver([mats[v]], kind=kind, value_sets=False)
        one[v].set_values()
        one[v].factor(precision)
    for nrhs in (1, 7, 8, 17):
        print(f"case block gemv {kind} {precision} nrhs={nrhs}", flush=True)
        rhs = [np.stack([uniform(50 * v + q, n, -1, 1) for q in range(nrhs)], axis=1)
               for v in range(NSETS)]
        xs = vs.solve(rhs, refine=False)
        for v, s in one.items():
            assert np.array_equal(xs[v], s.solve([rhs[v]], refine=False)[0]), f"set {v}"
