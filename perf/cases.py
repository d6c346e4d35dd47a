"""The work that a program has this framework do, through its public entry
points, for timing one state of the code against another.

A case is a dict of plain values.  ``prepare`` makes what a program holds
before the call (a matrix on the device, its preconditioner, a set-up
solver, right-hand sides), ``run`` is one call and returns its whole result,
``work`` says what that call cannot do without, and ``exact`` gives the
result in 64 bits from the definition alone.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from faspxx_amd import fx
from faspxx_amd.autograd import SolveOptions, SparsePattern, sparse_solve

RESTART = 30  # GMRES / FGMRES restart length (SOLParams default)
SWEEPS = 50   # weighted-Jacobi sweeps, omega = 2/3


# ---- systems ------------------------------------------------------------------
def _stencil(n, cols, vals, mask):
    """CSR (row pointers, columns, values) of the masked (n, s) candidates."""
    rp = np.zeros(n + 1, dtype=np.uint32)
    np.cumsum(mask.sum(axis=1), out=rp[1:])
    return rp, cols[mask].astype(np.uint32), np.ascontiguousarray(vals[mask])


def _grid2(m):
    i = np.arange(m * m, dtype=np.int64)
    ix, iy = i % m, i // m
    cols = np.stack([i - m, i - 1, i, i + 1, i + m], axis=1)
    mask = np.stack([iy > 0, ix > 0, np.ones(m * m, bool), ix < m - 1, iy < m - 1], axis=1)
    return cols, mask


@functools.lru_cache(maxsize=2)
def _poisson2d(m):
    """5-point Laplacian on m x m interior points."""
    cols, mask = _grid2(m)
    return _stencil(m * m, cols, np.tile([-1.0, -1.0, 4.0, -1.0, -1.0], (m * m, 1)), mask)


@functools.lru_cache(maxsize=2)
def _poisson3d(m):
    """7-point Laplacian on m x m x m interior points."""
    n = m * m * m
    i = np.arange(n, dtype=np.int64)
    ix, iy, iz = i % m, (i // m) % m, i // (m * m)
    cols = np.stack([i - m * m, i - m, i - 1, i, i + 1, i + m, i + m * m], axis=1)
    mask = np.stack([iz > 0, iy > 0, ix > 0, np.ones(n, bool), ix < m - 1, iy < m - 1,
                     iz < m - 1], axis=1)
    return _stencil(n, cols, np.tile([-1.0] * 3 + [6.0] + [-1.0] * 3, (n, 1)), mask)


@functools.lru_cache(maxsize=2)
def _convdiff2d(m):
    """-eps Lap u + w . grad u, first-order upwind, eps = 1e-2, w = (1, 0.5)."""
    h = 1.0 / (m + 1)
    e = 1e-2 / (h * h)
    cols, mask = _grid2(m)
    vals = np.tile([-e - 0.5 / h, -e - 1.0 / h, 4 * e + 1.5 / h, -e, -e], (m * m, 1))
    return _stencil(m * m, cols, vals, mask)


def _varcoef2d(m, seed):
    """-div(kappa grad u) by finite volumes on m x m cells, kappa lognormal
    (another one for each seed), harmonic-mean faces, Dirichlet zero."""
    kap = np.exp(0.5 * np.random.default_rng([seed, 7]).standard_normal((m, m)))
    def face(a, b):
        return 2.0 * a * b / (a + b)
    south, west = 2.0 * kap, 2.0 * kap
    east, north = 2.0 * kap, 2.0 * kap
    south[1:], north[:-1] = face(kap[1:], kap[:-1]), face(kap[:-1], kap[1:])
    west[:, 1:], east[:, :-1] = face(kap[:, 1:], kap[:, :-1]), face(kap[:, :-1], kap[:, 1:])
    diag = south + west + east + north
    cols, mask = _grid2(m)
    vals = np.stack([-south, -west, diag, -east, -north], axis=-1).reshape(m * m, 5)
    return _stencil(m * m, cols, vals, mask)


@functools.lru_cache(maxsize=2)
def _powerlaw(n):
    """Symmetric irregular M-matrix: row i picks k_i ~ k^-2.2 (2 .. 2048)
    uniform columns, both triangles get the entry, the diagonal dominates."""
    rng = np.random.default_rng([n, 3])
    ks = np.arange(2, 2049, dtype=np.float64)
    cdf = np.cumsum(ks ** -2.2)
    k = 2 + np.searchsorted(cdf / cdf[-1], rng.random(n))
    k = np.minimum(k, max(1, n // 2))
    r = np.repeat(np.arange(n, dtype=np.int64), k)
    c = rng.integers(0, n, r.shape[0])
    lo, hi = np.minimum(r, c), np.maximum(r, c)
    key = np.unique(lo[lo < hi] * n + hi[lo < hi])
    v = -rng.random(key.shape[0])
    lo, hi = key // n, key % n
    diag = 1.0 + np.bincount(lo, -v, n) + np.bincount(hi, -v, n)
    key = np.concatenate([key, hi * n + lo, np.arange(n, dtype=np.int64) * (n + 1)])
    order = np.argsort(key)
    rp = np.zeros(n + 1, dtype=np.uint32)
    np.cumsum(np.bincount(key // n, minlength=n), out=rp[1:])
    return rp, (key[order] % n).astype(np.uint32), np.concatenate([v, v, diag])[order]


def _system(case, seed):
    kind, size = case["system"], case["size"]
    if kind == "poisson2d":
        return _poisson2d(size)
    if kind == "poisson3d":
        return _poisson3d(size)
    if kind == "convdiff2d":
        return _convdiff2d(size)
    if kind == "varcoef2d":
        return _varcoef2d(size, seed)
    return _powerlaw(size)


def _order(case):
    """Rows of the case's system, and about how many entries it stores."""
    kind, m = case["system"], case["size"]
    if kind == "poisson3d":
        return m ** 3, 7 * m ** 3 - 6 * m * m
    if kind == "powerlaw":
        return m, 13 * m
    return m * m, 5 * m * m - 4 * m


def _apply(A, x):
    """A x in 64 bits."""
    rp, ci, va = A
    return np.add.reduceat(va * x[ci], rp[:-1].astype(np.int64))


def _apply_t(A, x):
    rp, ci, va = A
    rows = np.repeat(np.arange(rp.shape[0] - 1), np.diff(rp.astype(np.int64)))
    return np.bincount(ci, va * x[rows], rp.shape[0] - 1)


def _uniform(seed, stream, n):
    return np.random.default_rng([seed, stream]).uniform(-1.0, 1.0, n)


# ---- the cases ------------------------------------------------------------------
def listed():
    return [
        # the size of the reference's own data files and unit tests: launch
        # and synchronisation latency is all there is
        {"name": "pcg_poisson2d_32", "op": "pcg", "system": "poisson2d", "size": 32},
        # the headline solve: FP64 Jacobi-PCG to 1e-8 on the 3D Poisson system
        {"name": "pcg_poisson3d_128", "op": "pcg", "system": "poisson3d", "size": 128},
        # the same system by the f32-inner / f64-refined solver, to 1e-12
        {"name": "ir_poisson3d_128", "op": "ir", "system": "poisson3d", "size": 128},
        # the headline SpMV and the residual with it, MAT::Apply and
        # MAT::Residual, as a program's own loop calls them
        {"name": "spmv_poisson3d_128", "op": "spmv", "system": "poisson3d", "size": 128,
         "dtype": "f64"},
        # SpMV on an irregular matrix, scattered columns, long and short rows
        {"name": "spmv_powerlaw_1048576", "op": "spmv", "system": "powerlaw", "size": 1048576,
         "dtype": "f64"},
        # weighted Jacobi as a smoother: a fixed number of sweeps
        {"name": "jacobi_poisson3d_128", "op": "jacobi", "system": "poisson3d", "size": 128},
        # BiCGStab to 1e-13 on an odd-sized system (its iterates follow every
        # rounding, so only a tight solution can be compared)
        {"name": "bicgstab_poisson3d_95", "op": "bicgstab", "system": "poisson3d", "size": 95},
        # GMRES(30) and FGMRES(30) on upwind convection-diffusion, each with
        # a budget of iterations, large and ordinary
        {"name": "gmres_convdiff2d_1024", "op": "gmres", "system": "convdiff2d", "size": 1024,
         "iters": 240},
        {"name": "fgmres_convdiff2d_256", "op": "fgmres", "system": "convdiff2d", "size": 256,
         "iters": 240},
        # forward and adjoint solve of the differentiable solve, with the
        # gradients of the right-hand side and of every stored entry
        {"name": "adjoint_varcoef2d_512", "op": "adjoint", "system": "varcoef2d", "size": 512},
        # a program's own iteration over the VEC operations, odd length
        {"name": "vec_1000003", "op": "vec", "n": 1000003, "dtype": "f64"},
        # setup-time algebra: A A, A + B / 2, lower part and transpose
        {"name": "setup_poisson3d_64", "op": "setup", "system": "poisson3d", "size": 64},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["pcg", "pcg", "ir", "spmv", "spmv", "jacobi", "bicgstab", "gmres", "fgmres",
                     "adjoint", "vec", "setup"])
    case = {"op": op}
    if op == "vec":
        return {"op": op, "n": _log_int(rng, 100, 8000000), "dtype": rng.choice(["f64", "f32"])}
    if op == "adjoint":
        return {"op": op, "system": "varcoef2d", "size": _log_int(rng, 16, 512)}
    if op in ("gmres", "fgmres"):
        return {"op": op, "system": rng.choice(["convdiff2d", "varcoef2d"]),
                "size": _log_int(rng, 10, 1024 if op == "gmres" else 700),
                "iters": rng.randint(31, 240)}
    if op == "setup":
        kind = rng.choice(["poisson2d", "poisson3d", "varcoef2d"])
        return {"op": op, "system": kind,
                "size": _log_int(rng, 8, 64) if kind == "poisson3d" else _log_int(rng, 20, 512)}
    kinds = ["poisson2d", "poisson3d", "varcoef2d", "powerlaw"]
    if op == "bicgstab":
        kinds = ["poisson3d", "convdiff2d"]
    case["system"] = rng.choice(kinds)
    hi = {"poisson2d": 512, "poisson3d": 128, "varcoef2d": 512, "convdiff2d": 128,
          "powerlaw": 1048576 if op == "spmv" else 262144}[case["system"]]
    if op == "bicgstab":
        hi = min(hi, 112)
    case["size"] = _log_int(rng, {"powerlaw": 256, "poisson3d": 8}.get(case["system"], 10), hi)
    if op == "spmv":
        case["dtype"] = rng.choice(["f64", "f32"])
    return case


# ---- what a program holds before the call -------------------------------------------
@functools.lru_cache(maxsize=1)
def _ctx():
    return fx.Context(0)


def _device(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda").to(dtype)


def _vec(ctx, t):
    """The library's view of a torch vector (the tensor keeps the memory)."""
    return fx.Vec.wrap(ctx, t.data_ptr(), t.shape[0], fx.F32 if t.dtype == torch.float32 else fx.F64)


def _csr(ctx, A):
    return fx.Csr(ctx, A[0].shape[0] - 1, A[0].shape[0] - 1, *A)


def _params(**kw):
    return fx.params(**{"maxIter": 20000, "absTol": 0.0, **kw})


_SOLVERS = {  # solver, weight of its Jacobi preconditioner, parameters
    "pcg": (fx.CG, 1.0, {"relTol": 1e-8}),
    "bicgstab": (fx.BICGSTAB, 1.0, {"relTol": 1e-13}),
    "gmres": (fx.GMRES, 1.0, {"relTol": 1e-30, "restart": RESTART}),
    "fgmres": (fx.FGMRES, 1.0, {"relTol": 1e-30, "restart": RESTART}),
    "jacobi": (fx.JACOBI, 2.0 / 3.0, {"relTol": 1e-30, "maxIter": SWEEPS}),
}


def prepare(case, seed):
    op, ctx = case["op"], _ctx()
    dt = torch.float32 if case.get("dtype") == "f32" else torch.float64
    if op == "vec":
        t = {k: _device(_uniform(seed, s, case["n"]), dt) for s, k in enumerate("xyvw")}
        torch.cuda.synchronize()
        return {"op": op, "t": t, **{k: _vec(ctx, v) for k, v in t.items()}}
    A = _system(case, seed)
    n = A[0].shape[0] - 1
    if op == "adjoint":
        pattern = SparsePattern(ctx, _Host(A), SolveOptions())
        return {"op": op, "pattern": pattern,
                "values": _device(A[2]).requires_grad_(),
                "b": _device(_apply(A, _uniform(seed, 0, n))).requires_grad_(),
                "g": _device(_apply_t(A, _uniform(seed, 1, n)))}
    if op == "setup":
        rng = np.random.default_rng([seed, 2])
        A = (A[0], A[1], rng.uniform(0.5, 1.5, A[1].shape[0]))
        B = (A[0], A[1], rng.uniform(0.5, 1.5, A[1].shape[0]))
        t = _device(_uniform(seed, 0, n))
        torch.cuda.synchronize()
        return {"op": op, "ctx": ctx, "A": _csr(ctx, A), "B": _csr(ctx, B), "t": t,
                "v": _vec(ctx, t)}
    M = _csr(ctx, A)
    if op == "spmv":
        if dt == torch.float32:
            M.make_f32()
        t = {"x": _device(_uniform(seed, 0, n), dt), "b": _device(_uniform(seed, 1, n), dt),
             "y": torch.zeros(n, dtype=dt, device="cuda"),
             "r": torch.zeros(n, dtype=dt, device="cuda")}
        torch.cuda.synchronize()
        return {"op": op, "A": M, "t": t, **{k: _vec(ctx, v) for k, v in t.items()}}
    t = {"b": _device(_apply(A, _uniform(seed, 0, n))),
         "x": torch.zeros(n, dtype=torch.float64, device="cuda")}
    torch.cuda.synchronize()
    state = {"op": op, "A": M, "t": t, **{k: _vec(ctx, v) for k, v in t.items()}}
    if op == "ir":
        state["solver"] = fx.IR(ctx, M, 1.0, _params(maxIter=50, relTol=1e-12),
                                _params(relTol=1e-4))
        return state
    kind, weight, prm = _SOLVERS[op]
    if "iters" in case:
        prm = {**prm, "maxIter": case["iters"]}
    state["pc"] = fx.Precond(ctx, "jacobi", M, weight, 1)
    state["prm"] = _params(**prm)
    state["solver"] = fx.Solver(ctx, kind)
    state["solver"].Setup(M, state["pc"], state["prm"])
    return state


class _Host:
    """A host matrix as SparsePattern takes it."""

    def __init__(self, A):
        self.row_ptr, self.col_ind, self.values = A
        self.nrow = self.mcol = A[0].shape[0] - 1
        self.diag_ptr = None


def run(state):
    op = state["op"]
    if op == "spmv":
        state["A"].Apply(state["x"], state["y"])
        state["A"].Residual(state["b"], state["x"], state["r"])
        return state["t"]["y"], state["t"]["r"]
    if op == "vec":
        # one step of a program's own iteration: a new vector, its scaling,
        # a dot product, an update with its norm, and the step's size
        x, y, v, w = state["x"], state["y"], state["v"], state["w"]
        w.WAXPBY(0.5, x, -0.25, y)
        w.PointwiseMult(v)
        dot = w.Dot(x)
        w.AXPY(0.125, y)
        norm = w.AXPY_Norm2(-0.0625, x)
        w.XPAY(0.75, v)
        return state["t"]["w"], dot, norm, w.Norm2(), w.NormInf()
    if op == "adjoint":
        values, b = state["values"], state["b"]
        x = sparse_solve(values, b, state["pattern"])
        grads = torch.autograd.grad(x, (values, b), state["g"])
        return (x.detach(), *grads)
    if op == "setup":
        ctx, A, B = state["ctx"], state["A"], state["B"]
        out = []
        for C in (fx.Csr.mult(A, A), fx.Csr.add(1.0, A, 0.5, B), A.lower_tri(), A.transpose()):
            y = torch.empty_like(state["t"])
            values = torch.empty(C.nnz, dtype=torch.float64, device="cuda")
            C.Apply(state["v"], _vec(ctx, y))
            fx.Vec.wrap(ctx, C.values_ptr, C.nnz).copy_to(_vec(ctx, values))
            out += [y, values]
        ctx.sync()
        return out
    state["x"].set(0.0)
    if op in ("gmres", "fgmres"):
        # as Krylov() does: the restart length (and FGMRES's Z) as set up
        state["solver"].Setup(state["A"], state["pc"], state["prm"])
        state["solver"].Clean()
    state["solver"].Solve(state["b"], state["x"])
    return state["t"]["x"]


# ---- what a call cannot do without, and its result in 64 bits --------------------------
def _iterations(case):
    """About how many iterations the case's solve takes."""
    m, kind = case["size"], case["system"]
    if "iters" in case:
        return case["iters"]
    if case["op"] == "jacobi":
        return SWEEPS
    tight = {"pcg": 1.0, "ir": 1.5, "bicgstab": 0.8, "adjoint": 2.6}[case["op"]]
    per = {"poisson2d": 2.2, "poisson3d": 2.5, "varcoef2d": 2.0, "convdiff2d": 1.7}
    return max(10, int(tight * (15 if kind == "powerlaw" else per[kind] * m)))


def work(case):
    op = case["op"]
    s = 4 if case.get("dtype") == "f32" else 8
    if op == "vec":
        return {"bytes": 4 * s * case["n"], "flops": 14 * case["n"]}
    n, nnz = _order(case)
    matrix = (s + 4) * nnz + 4 * n
    if op == "spmv":
        return {"bytes": matrix + 4 * s * n, "flops": 4 * nnz}
    if op == "setup":
        # A and B read once; four results written, and their products with v
        wide = case["system"] == "poisson3d"
        stored = (25 if wide else 13) * n + nnz + (nnz + n) // 2 + nnz
        return {"bytes": 2 * matrix + 12 * stored + 5 * 8 * n,
                "flops": 2 * (49 if wide else 25) * n + 2 * stored}
    vectors = {"gmres": 60, "fgmres": 60, "bicgstab": 24, "jacobi": 5}.get(op, 12)
    flops = _iterations(case) * ((4 if op == "bicgstab" else 2) * nnz + vectors * n)
    return {"bytes": matrix + 2 * 8 * n + (matrix if op == "adjoint" else 0), "flops": flops}


def exact(case, seed):
    op = case["op"]
    f32 = case.get("dtype") == "f32"

    def given(stream, n):
        a = _uniform(seed, stream, n)
        return a.astype(np.float32).astype(np.float64) if f32 else a

    if op == "vec":
        x, y, v = (given(i, case["n"]) for i in range(3))
        w = (0.5 * x - 0.25 * y) * v
        dot = float(w @ x)
        w = w + 0.125 * y - 0.0625 * x
        norm = float(np.linalg.norm(w))
        w = 0.75 * w + v
        return w, dot, norm, float(np.linalg.norm(w)), float(np.max(np.abs(w)))
    A = _system(case, seed)
    n = A[0].shape[0] - 1
    if op == "spmv":
        va = A[2].astype(np.float32).astype(np.float64) if f32 else A[2]
        y = _apply((A[0], A[1], va), given(0, n))
        return y, given(1, n) - y
    if op == "adjoint":
        x, lam = _uniform(seed, 0, n), _uniform(seed, 1, n)
        rows = np.repeat(np.arange(n), np.diff(A[0].astype(np.int64)))
        return x, -lam[rows] * x[A[1]], lam
    if op == "setup":
        rng = np.random.default_rng([seed, 2])
        A = (A[0], A[1], rng.uniform(0.5, 1.5, A[1].shape[0]))
        B = (A[0], A[1], rng.uniform(0.5, 1.5, A[1].shape[0]))
        v = _uniform(seed, 0, n)
        rows = np.repeat(np.arange(n), np.diff(A[0].astype(np.int64)))
        low = (A[0], A[1], np.where(A[1] <= rows, A[2], 0.0))
        return [_apply(A, _apply(A, v)), None, _apply(A, v) + 0.5 * _apply(B, v), None,
                _apply(low, v), None, _apply_t(A, v), None]
    if op == "jacobi":
        b, x = _apply(A, _uniform(seed, 0, n)), np.zeros(n)
        rows = np.repeat(np.arange(n), np.diff(A[0].astype(np.int64)))
        scale = (2.0 / 3.0) / A[2][A[1] == rows]
        if n > 300000:
            return None  # 50 sweeps take too long here
        for _ in range(SWEEPS):
            x = x + scale * (b - _apply(A, x))
        return x
    if op in ("gmres", "fgmres"):
        return None  # a budget of iterations, not a solution
    return _uniform(seed, 0, n)  # b = A x in 64 bits, so x solves it
