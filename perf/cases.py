"""The work that users of this library have it do, as measurable cases.

Every case solves sparse systems A x = b whose solution is known exactly: the
entries of A, of x and so every product and partial sum of A x are multiples
of small powers of two that a double holds without rounding, so b = A x is
exact and x is the 64-bit answer of the solve.

Modes of a case:
  refactor  new values of a kept pattern, resident on the device (a Newton or
            time step assembled there): spkhip_inmatrix_device, spkhip_factor,
            then the solve (refined in double for the float precisions)
  solve     the factor is kept, new right-hand sides only (linear time steps)
  host      the Python interface on host arrays: sparspaklu_refactor with a
            scipy matrix, then triangularsolve
  batch     many uneven systems in one BatchedSolver: values from the host,
            factor, solve of right-hand sides resident on the device
  sets      many value sets of one pattern in one handle (resident values)

Matrices: "grid" is a 2D (nz = 1: 5-point) or 3D (7-point) diffusion operator
with a diffusivity per cell (log-uniform over `contrast`, drawn from the
seed) and, for the LU solver, upwind convection; "elasticity" is Q1 linear
elasticity (3 dof per node, nx elements per side) plus a diagonal mass term
drawn from the seed.
"""
import ctypes
import math
import os
import random
import sys
from collections import OrderedDict

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "sparspak.jl_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "sparspak.jl_amd"))

from sparspak_hip import (findorder, sparspaklu, sparspaklu_refactor, symbolicfactor,  # noqa: E402
                          triangularsolve)
from sparspak_hip import _lib  # noqa: E402
from sparspak_hip.batch import BatchedSolver  # noqa: E402
from sparspak_hip.gallery import convdiff3d, elasticity3d, laplace2d  # noqa: E402
from sparspak_hip.symbolic import Graph, SymbolicFactor  # noqa: E402

PRECISION = {"fp64": 0, "fp32": 1, "fp32_bf16": 2, "fp32_bf16x3": 4}


def _case(mode, nx, ny=1, nz=1, matrix="grid", solver="lu", precision="fp64", nrhs=1, count=1,
          contrast=2.0, **name):
    return dict(name, mode=mode, matrix=matrix, nx=nx, ny=ny, nz=nz, solver=solver,
                precision=precision, nrhs=nrhs, count=count, contrast=float(contrast))


def listed():
    return [
        # a small nonlinear 2D problem inside a Newton loop: launches and
        # latency are all of it
        _case("refactor", 24, 17, name="newton_2d_24x17"),
        # the 2D 5-point SPD configuration, n = 10 000
        _case("refactor", 100, 100, solver="spd", name="diffusion_2d_100_spd"),
        # the drop-in use from Python: sparspaklu! with a new scipy matrix,
        # then ldiv on a host vector; an odd 2D grid
        _case("host", 193, 171, name="host_2d_193x171"),
        # an odd, ragged 3D grid, float factor with refinement, three loads
        _case("refactor", 31, 23, 17, precision="fp32", nrhs=3, name="convdiff_31x23x17_fp32"),
        # ordinary 3D convection-diffusion step in double
        _case("refactor", 32, 32, 32, name="convdiff_32_fp64"),
        # the headline configuration in double and in its mixed precision
        _case("refactor", 64, 64, 64, name="convdiff_64_fp64"),
        _case("refactor", 64, 64, 64, precision="fp32_bf16x3", name="convdiff_64_bf16x3"),
        # implicit dynamics of an elastic body: an ordinary mesh in double,
        # the large mixed-precision configuration
        _case("refactor", 20, matrix="elasticity", solver="spd", name="elasticity_20_spd"),
        _case("refactor", 40, matrix="elasticity", solver="spd", precision="fp32_bf16x3",
              name="elasticity_40_spd_bf16x3"),
        # uneven 2D systems (sides 8..96) factored together, four loads each
        _case("batch", 8, 96, solver="spd", count=128, nrhs=4, name="batch_128_uneven_spd"),
        # value sets of one 32^3 pattern with strongly varying diffusivity
        # (parameter studies), 16 right-hand sides each
        _case("sets", 32, 32, 32, precision="fp32_bf16x3", nrhs=16, count=32, contrast=100.0,
              name="sets_32_of_convdiff_32"),
        # linear time steps: the factor is kept, one right-hand side a step
        _case("solve", 56, 48, 41, name="timestep_56x48x41_solve"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above; none costs more than the largest listed."""
    kind = rng.choice(["grid2", "grid2", "grid3", "grid3", "grid3", "elasticity", "batch", "sets",
                       "solve", "host"])
    precision = rng.choice(["fp64", "fp64", "fp32", "fp32_bf16x3"])
    solver = rng.choice(["lu", "lu", "spd"])
    if kind == "grid2":
        return _case("refactor", _log(rng, 16, 300), _log(rng, 16, 300), solver=solver,
                     precision=precision, nrhs=rng.choice([1, 1, 2, 5]))
    if kind == "grid3":
        return _case("refactor", _log(rng, 6, 60), _log(rng, 6, 60), _log(rng, 6, 60),
                     solver=solver, precision=precision, nrhs=rng.choice([1, 1, 3]))
    if kind == "elasticity":
        return _case("refactor", _log(rng, 4, 30), matrix="elasticity",
                     solver=rng.choice(["spd", "spd", "lu"]), precision=precision)
    if kind == "batch":
        lo = rng.randint(4, 24)
        return _case("batch", lo, rng.randint(lo + 8, 96), solver=solver, count=_log(rng, 8, 128),
                     precision=rng.choice(["fp64", "fp32"]), nrhs=rng.randint(1, 6))
    if kind == "sets":
        return _case("sets", _log(rng, 8, 30), _log(rng, 8, 30), _log(rng, 8, 30),
                     precision=precision, count=_log(rng, 2, 32), nrhs=rng.randint(1, 16),
                     contrast=rng.choice([2.0, 100.0]))
    if kind == "solve":
        return _case("solve", _log(rng, 10, 56), _log(rng, 10, 56), _log(rng, 10, 56),
                     solver=solver, precision=precision, nrhs=rng.choice([1, 1, 2, 8, 16]))
    return _case("host", _log(rng, 16, 240), _log(rng, 16, 240),
                 precision=rng.choice(["fp64", "fp32"]), nrhs=rng.choice([1, 1, 4]))


# -- patterns: what does not change from one step to the next -----------------

class _Pattern:
    """A pattern's scipy matrix, its entries' rows and columns on the device,
    and its host symbolic factor (ordering and panel structure)."""

    def __init__(self, matrix, nx, ny, nz):
        if matrix == "elasticity":
            A = elasticity3d(nx) * float(nx)  # entries of order one
            # multiples of 2^-28, so that products with x are exact
            A.data = np.round(A.data * 2.0 ** 28) * 2.0 ** -28
        else:
            A = laplace2d(nx, ny) if nz == 1 else convdiff3d(nx, ny, nz)
        A.sort_indices()
        self.A = A
        self.n = A.shape[0]
        self.shape = (nx, ny, nz)
        self.matrix = matrix
        cols = np.repeat(np.arange(self.n, dtype=np.int64), np.diff(A.indptr))
        self.rows = torch.from_numpy(A.indices.astype(np.int64)).cuda()
        self.cols = torch.from_numpy(cols).cuda()
        self.base = torch.from_numpy(A.data.copy()).cuda() if matrix == "elasticity" else None
        self.colptr = A.indptr.astype(np.int64) + 1
        self.rowval = A.indices.astype(np.int64) + 1
        self.nnz = int(A.nnz)
        self.sym = {}

    def symbolic(self, solver):
        if solver not in self.sym:
            s = SymbolicFactor(self.n, Graph.from_csc(self.n, self.colptr, self.rowval), kind=solver)
            s.findorder()
            s.symbolicfactor()
            self.sym[solver] = s
        return self.sym[solver]

    def values(self, g, solver, contrast):
        """One step's values (CSC order, double, on the device)."""
        diag = self.rows == self.cols
        if self.matrix == "elasticity":
            mass = torch.randint(0, 1024, (self.n,), generator=g, device="cuda").double() * 2.0 ** -20
            v = self.base.clone()
            v[diag] += mass[self.rows[diag]]
            return v
        # diffusivity per cell; a face takes the harmonic mean of its two
        # cells, a boundary face its own cell's; multiples of 2^-20
        u = torch.rand((self.n,), generator=g, device="cuda", dtype=torch.float64)
        k = torch.exp((2.0 * u - 1.0) * math.log(contrast))
        ki, kj = k[self.rows], k[self.cols]
        off = -torch.round(2.0 * ki * kj / (ki + kj) * 2.0 ** 20) * 2.0 ** -20
        off[diag] = 0.0
        d = torch.zeros(self.n, dtype=torch.float64, device="cuda")
        d.index_add_(0, self.rows, -off)
        faces = torch.zeros(self.n, dtype=torch.float64, device="cuda")
        faces.index_add_(0, self.rows, (~diag).double())
        d += (4 if self.shape[2] == 1 else 6) - faces  # Dirichlet sides
        if solver == "lu":  # upwind convection along +x, +y, +z
            nx, ny, _ = self.shape
            step = self.rows - self.cols
            for stride, vel in ((1, 1.0), (nx, 0.5), (nx * ny, 0.25)):
                if stride < nx * ny * self.shape[2]:
                    off -= vel * (step == stride).double()
                    d += vel
        off[diag] = d[self.rows[diag]]
        return off

    def product(self, v, x):
        """A x for x (nrhs, n), exact."""
        b = torch.zeros_like(x)
        for q in range(x.shape[0]):
            b[q].index_add_(0, self.rows, v * x[q][self.cols])
        return b


_patterns = OrderedDict()


def _pattern(matrix, nx, ny, nz):
    key = (matrix, nx, ny, nz)
    if key not in _patterns:
        _patterns[key] = _Pattern(*key)
        if len(_patterns) > 2:
            _patterns.popitem(last=False)
    _patterns.move_to_end(key)
    return _patterns[key]


def _sides(case):
    """Sides of a batch's square grids: spread over [nx, ny], the same for
    every seed (they are the pattern)."""
    r = random.Random(4)
    return [r.randint(case["nx"], case["ny"]) for _ in range(case["count"])]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _solution(g, nrhs, n):
    """x in [-1, 1], multiples of 2^-16, (nrhs, n): column-major n x nrhs."""
    x = torch.randint(-2 ** 16, 2 ** 16 + 1, (nrhs, n), generator=g, device="cuda")
    return x.double() * 2.0 ** -16


def _problem(case, seed):
    """The step's values (one tensor per system or set) and its exact x and
    b, both (nrhs, n of all systems)."""
    g = _generator(seed)
    if case["mode"] == "batch":
        pats = [_square(s) for s in _sides(case)]
        n = sum(p.n for p in pats)
        x = _solution(g, case["nrhs"], n)
        vals, bs, at = [], [], 0
        for p in pats:
            vals.append(p.values(g, case["solver"], case["contrast"]))
            bs.append(p.product(vals[-1], x[:, at:at + p.n]))
            at += p.n
        return pats, vals, x, torch.cat(bs, dim=1)
    p = _pattern(case["matrix"], case["nx"], case["ny"], case["nz"])
    x = _solution(g, case["nrhs"], p.n * case["count"])
    vals, bs = [], []
    for v in range(case["count"]):
        vals.append(p.values(g, case["solver"], case["contrast"]))
        bs.append(p.product(vals[-1], x[:, v * p.n:(v + 1) * p.n]))
    return p, vals, x, torch.cat(bs, dim=1)


_squares = {}


def _square(side):
    if side not in _squares:
        _squares[side] = _Pattern("grid", side, side, 1)
    return _squares[side]


class _Handle:
    """A device handle of the C interface with its symbolic factor."""

    def __init__(self, p, solver, count):
        self.L = _lib.lib()
        self.h = ctypes.c_void_p()
        _lib.check(self.L.spkhip_create(ctypes.byref(self.h), 0), "spkhip_create")
        s, p64 = p.symbolic(solver), _lib.p64
        xunz = s.xunz if s.xunz is not None else np.zeros(p.n + 1, dtype=np.int64)
        _lib.check(self.L.spkhip_symbolic_upload(
            self.h, 0 if solver == "lu" else 1, p.n, s.nsuper, p64(s.xsuper), p64(s.snode),
            p64(s.xlindx), p64(s.lindx), p64(s.xlnz), p64(xunz), p64(s.order.rperm),
            p64(s.order.rinvp), p64(p.colptr), p64(p.rowval)), "spkhip_symbolic_upload")
        if count > 1:
            _lib.check(self.L.spkhip_set_value_sets(self.h, count), "spkhip_set_value_sets")

    def __del__(self):
        if self.h:
            self.L.spkhip_destroy(self.h)

    def inmatrix(self, vals):
        _lib.check(self.L.spkhip_inmatrix_device(self.h, ctypes.c_void_p(vals.data_ptr())),
                   "spkhip_inmatrix_device")

    def factor(self, precision):
        _lib.check(self.L.spkhip_factor(self.h, PRECISION[precision]), "spkhip_factor")

    def solve(self, x, precision):
        nrhs, n = x.shape
        ptr = ctypes.c_void_p(x.data_ptr())
        if precision == "fp64":
            _lib.check(self.L.spkhip_solve_device(self.h, nrhs, ptr, n), "spkhip_solve_device")
        else:
            rc = self.L.spkhip_solve_refine_device(self.h, nrhs, ptr, n, 1e-14, 10)
            if rc != -5:  # -5: the tolerance was not met, x is still the best found
                _lib.check(rc, "spkhip_solve_refine_device")


def prepare(case, seed):
    p, vals, x, b = _problem(case, seed)
    st = {"case": case, "b": b}
    if case["mode"] == "host":
        m = p.A.copy()
        m.data = vals[0].cpu().numpy()
        lu = sparspaklu(p.A, factorize=False)
        findorder(lu)
        symbolicfactor(lu)
        st.update(lu=lu, m=m, b=np.asfortranarray(b.cpu().numpy().T))
        return st
    st["x"] = torch.empty_like(b)
    if case["mode"] == "batch":
        values = [v.cpu().numpy() for v in vals]
        mats = []
        for q, v in zip(p, values):
            m = q.A.copy()
            m.data = v
            mats.append(m)
        st.update(batch=BatchedSolver(mats, kind=case["solver"], value_sets=False), values=values)
        st["batch"].upload()
        return st
    st["handle"] = _Handle(p, case["solver"], case["count"])
    st["vals"] = torch.cat(vals)
    if case["mode"] == "solve":
        st["handle"].inmatrix(st["vals"])
        st["handle"].factor(case["precision"])
    return st


def run(st):
    c = st["case"]
    if c["mode"] == "host":
        sparspaklu_refactor(st["lu"], st["m"], precision=c["precision"])
        x = st["b"].copy(order="F")
        triangularsolve(st["lu"], x)
        return x
    x = st["x"]
    if c["mode"] == "batch":
        st["batch"].set_values(st["values"])
        st["batch"].factor(c["precision"])
        x.copy_(st["b"])
        st["batch"].solve_device(x, c["nrhs"])
        return x
    h = st["handle"]
    if c["mode"] != "solve":
        h.inmatrix(st["vals"])
        h.factor(c["precision"])
    x.copy_(st["b"])
    h.solve(x, c["precision"])
    return x


def exact(case, seed):
    x = _problem(case, seed)[2]
    return x.cpu().numpy().T if case["mode"] == "host" else x


def work(case):
    """A pass reads the values and right-hand sides and writes the factor and
    the solutions once (a kept factor is read once instead); operations are
    the factorisation's and the solve's own, from the column counts."""
    item = 8 if case["precision"] == "fp64" else 4
    if case["mode"] == "batch":
        pats = [_square(s) for s in _sides(case)]
    else:
        pats = [_pattern(case["matrix"], case["nx"], case["ny"], case["nz"])] * case["count"]
    flops = nbytes = 0.0
    for p in pats:
        s = p.symbolic(case["solver"])
        entries = float(np.sum(s.colcnt)) * (2 if case["solver"] == "lu" else 1)
        nbytes += entries * item + 16.0 * p.n * case["nrhs"]
        flops += 4.0 * float(np.sum(s.colcnt)) * case["nrhs"]
        if case["mode"] != "solve":
            nbytes += 8.0 * p.nnz
            flops += s.flops()
    return {"bytes": nbytes, "flops": flops}
