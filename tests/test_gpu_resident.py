"""Solver loops that stay on the chip against the same loops kernel by kernel
(FASPXX_FX_NORESIDENT=1): the per-element arithmetic and the decisions are the
same, only the order of the sums differs.

Tolerances: a sum of n products in another order moves by at most about
log2(n) eps relative to the sum of magnitudes, so early residuals agree to
1e-10.  How far that carries a solution depends on the system (on the
unpreconditioned 181^2 variable-coefficient one the oracle's own CG solution
moves by 7e-9 .. 6e-8, and its count by one, when b moves by an ulp in an
eighth of its entries), so the solve kernel by kernel is repeated with such
right-hand sides and the solutions are held to four times that spread, and to
1e-10 where the spread is smaller still."""
import numpy as np
import pytest

from faspxx_amd import fx
from faspxx_amd import problems as P
from perturb import ulp_perturbed
from test_gpu_rowvalues import box2d

pytestmark = pytest.mark.gpu


def spd_box(m, k):
    """9 entries per row, symmetric, positive definite."""
    A = box2d(m, k)
    rows = np.repeat(np.arange(A.nrow), np.diff(A.row_ptr.astype(np.int64)))
    A.values[:] = np.where(A.col_ind == rows, 9.0, -1.0)
    return A


def solve(ctx, monkeypatch, resident, kind, A, prm, pc="jacobi", weight=1.0, x0=None, b=None,
          transposed=False):
    if not resident:
        monkeypatch.setenv("FASPXX_FX_NORESIDENT", "1")
    M = fx.Csr.from_problem(ctx, A)
    if transposed:  # built on the device: 16-bit deltas, no patterns
        M = M.transpose()
        assert M.layout == "d16"
    p = fx.Precond(ctx, "jacobi", M, weight, 1) if pc == "jacobi" else fx.Precond(ctx, "identity")
    s = fx.Solver(ctx, kind)
    s.Setup(M, p, fx.params(**prm))
    xs = np.random.default_rng(A.nrow).uniform(-1, 1, A.nrow)
    vb = fx.Vec.from_numpy(ctx, A.matvec(xs) if b is None else b)
    out = []
    for _ in range(2):  # the second solve starts from the first one's workspace
        x = fx.Vec.from_numpy(ctx, np.zeros(A.nrow) if x0 is None else x0)
        out.append((s.Solve(vb, x), x.numpy(), s.history()))
    monkeypatch.delenv("FASPXX_FX_NORESIDENT", raising=False)
    assert s.last_path == "fused"
    assert np.array_equal(out[0][1], out[1][1])  # run to run the same bits
    return out[1]


def check(ctx, monkeypatch, kind, A, prm, b=None, tol=1e-10, **kw):
    """Resident against kernel by kernel."""
    if b is None:
        b = A.matvec(np.random.default_rng(A.nrow).uniform(-1, 1, A.nrow))
    r1, x1, h1 = solve(ctx, monkeypatch, True, kind, A, prm, b=b, **kw)
    r0, x0, h0 = solve(ctx, monkeypatch, False, kind, A, prm, b=b, **kw)
    near = [solve(ctx, monkeypatch, False, kind, A, prm, b=ulp_perturbed(b, s), **kw)
            for s in range(2)]
    scale = np.linalg.norm(x0)
    spread = max(np.linalg.norm(x - x0) for _, x, _ in near)
    counts = [r.numIter for r, _, _ in near] + [r0.numIter]
    assert r1.retcode == r0.retcode
    assert min(counts) - 1 <= r1.numIter <= max(counts) + 1
    if max(counts) == min(counts):
        assert r1.numIter == r0.numIter and len(h1) == len(h0)
    k = min(len(h0), len(h1), 30)
    assert np.allclose(h1[:k], h0[:k], rtol=tol, atol=0)
    assert np.linalg.norm(x1 - x0) <= max(tol * scale, 4 * spread)
    assert np.isclose(r1.norm2, r0.norm2, rtol=0.2, atol=1e-300)


# one workgroup of one and two rows per thread, its limits, several
# workgroups, their limits (a ragged last one), two, four and eight rows per
# thread, and the first size that does not fit
SYSTEMS = {
    "p2d_1": lambda: P.poisson2d(1), "p2d_32": lambda: P.poisson2d(32),
    "p2d_33": lambda: P.poisson2d(33), "p2d_45": lambda: P.poisson2d(45),
    "p2d_46": lambda: P.poisson2d(46), "p3d_33": lambda: P.poisson3d(33),
    "fv_181": lambda: P.varcoef_fv(181)[0], "fv_512": lambda: P.varcoef_fv(512)[0],
    "fv_513": lambda: P.varcoef_fv(513)[0], "p3d_65": lambda: P.poisson3d(65),
    "p3d_81": lambda: P.poisson3d(81), "fv_725": lambda: P.varcoef_fv(725)[0],
    "p3d_102": lambda: P.poisson3d(102), "box_31": lambda: spd_box(31, 29),
    "box_130": lambda: spd_box(130, 131), "box_520": lambda: spd_box(520, 531),
}
PRM = dict(maxIter=60, relTol=1e-30, absTol=0.0)


@pytest.mark.parametrize("name", list(SYSTEMS))
@pytest.mark.parametrize("pc", ["jacobi", "identity"])
def test_cg_resident(ctx, monkeypatch, name, pc):
    A = SYSTEMS[name]()
    prm = dict(maxIter=3000, relTol=1e-8, absTol=0.0) if A.nrow < 40000 else PRM
    check(ctx, monkeypatch, fx.CG, A, prm, pc=pc)


@pytest.mark.parametrize("m", [20, 90, 520, 730])
def test_cg_resident_column_deltas(ctx, monkeypatch, m):
    A = P.varcoef_fv(m)[0]
    check(ctx, monkeypatch, fx.CG, A, PRM, transposed=True)


@pytest.mark.parametrize("prm", [
    dict(maxIter=0), dict(maxIter=1), dict(maxIter=7, relTol=1e-12), dict(maxIter=25, minIter=5),
    dict(maxIter=200, relTol=1e-6, savIter=5), dict(maxIter=2000, relTol=1e-19, restart=2),
    dict(maxIter=40, minIter=40)])
@pytest.mark.parametrize("m", [16, 70])
def test_cg_resident_stops(ctx, monkeypatch, prm, m):
    """Every way out of the loop: limits, minIter, the safe-guard's copies,
    the false-convergence check."""
    A = P.poisson2d(m)
    prm = dict(dict(relTol=1e-8, absTol=0.0), **prm)
    if prm["relTol"] == 1e-19:  # stops on rounding: the same way out, about as far
        new = solve(ctx, monkeypatch, True, fx.CG, A, prm)
        old = solve(ctx, monkeypatch, False, fx.CG, A, prm)
        assert new[0].retcode == old[0].retcode
        assert abs(new[0].numIter - old[0].numIter) <= 0.1 * old[0].numIter + 2
        assert np.linalg.norm(new[1] - old[1]) <= 1e-10 * np.linalg.norm(old[1])
    else:
        check(ctx, monkeypatch, fx.CG, A, prm)


@pytest.mark.parametrize("m", [20, 70])
def test_cg_resident_breakdown_and_zero(ctx, monkeypatch, m):
    """A right-hand side of zeros ((q, p) vanishes at once) and an exact start."""
    A = P.poisson2d(m)
    xs = np.random.default_rng(1).uniform(-1, 1, A.nrow)
    for b, x0 in ((np.zeros(A.nrow), None), (A.matvec(xs), xs)):
        prm = dict(maxIter=50, relTol=1e-30, absTol=0.0)
        new = solve(ctx, monkeypatch, True, fx.CG, A, prm, b=b, x0=x0)
        old = solve(ctx, monkeypatch, False, fx.CG, A, prm, b=b, x0=x0)
        assert new[0].retcode == old[0].retcode
        assert np.linalg.norm(new[1] - old[1]) <= 1e-12 * max(1.0, np.linalg.norm(old[1]))


@pytest.mark.parametrize("dim,m", [(2, 1), (2, 32), (2, 33), (2, 45), (2, 46), (2, 200), (2, 513),
                                   (3, 65), (3, 82), (3, 103)])
def test_ir_resident(ctx, monkeypatch, dim, m):
    """The refinement with its inner loop resident and kernel by kernel: both
    reach the outer tolerance, so the solutions differ by at most twice the
    condition number times it."""
    A = P.poisson2d(m) if dim == 2 else P.poisson3d(m)
    b = A.matvec(np.random.default_rng(m).uniform(-1, 1, A.nrow))
    out = []
    for off in (False, True):
        if off:
            monkeypatch.setenv("FASPXX_FX_NORESIDENT", "1")
        ir = fx.IR(ctx, fx.Csr.from_problem(ctx, A), 1.0,
                   fx.params(maxIter=50, relTol=1e-12, absTol=0.0),
                   fx.params(maxIter=20000, relTol=1e-4, absTol=0.0))
        monkeypatch.delenv("FASPXX_FX_NORESIDENT", raising=False)
        vb, runs = fx.Vec.from_numpy(ctx, b), []
        for _ in range(2):  # the second solve queues its outer steps ahead
            x = fx.Vec(ctx, A.nrow)
            res, inner = ir.Solve(vb, x)
            assert res.retcode == 0
            assert np.linalg.norm(b - A.matvec(x.numpy())) < 1.01e-12 * np.linalg.norm(b)
            runs.append((x.numpy(), res.numIter, inner))
        assert np.array_equal(runs[0][0], runs[1][0]) and runs[0][1:] == runs[1][1:]
        out.append(runs[1])
    cond = 1.0 / np.tan(np.pi / (2.0 * (m + 1))) ** 2
    (x1, o1, i1), (x0, o0, i0) = out
    assert abs(o1 - o0) <= 1 and abs(i1 - i0) <= 0.15 * i0 + 2
    assert np.linalg.norm(x1 - x0) <= 2e-12 * cond * np.linalg.norm(x0) + 1e-12
