"""BiCGStab's resident loop against the kernel-by-kernel one
(FASPXX_FX_NORESIDENT=1).  The two differ by the order of the sums, so the
bound on x is the larger of a relative one and four times what the
kernel-by-kernel loop itself moves when b moves by an ulp; few iterations,
since the recurrence enlarges any difference."""
import numpy as np
import pytest

from faspxx_amd import fx, problems as P
from test_gpu_resident import SYSTEMS as ALL, check, solve

pytestmark = pytest.mark.gpu

# one workgroup of one and two rows per thread, its limits, several
# workgroups, two and four rows per thread, and the first size that does not fit
SYSTEMS = {k: ALL[k] for k in ("p2d_32", "p2d_33", "p2d_45", "p2d_46", "p3d_33", "fv_181",
                               "fv_512", "fv_513", "p3d_65", "p3d_81", "fv_725", "p3d_102",
                               "box_31", "box_130", "box_520")}
SYSTEMS["convdiff_40"] = lambda: P.convdiff2d(40)
SYSTEMS["convdiff_301"] = lambda: P.convdiff2d(301)
SYSTEMS["convdiff_777"] = lambda: P.convdiff2d(777)


@pytest.mark.parametrize("name", list(SYSTEMS))
@pytest.mark.parametrize("pc", ["jacobi", "identity"])
def test_bicgstab_resident(ctx, monkeypatch, name, pc):
    check(ctx, monkeypatch, fx.BICGSTAB, SYSTEMS[name](),
          dict(maxIter=12, relTol=1e-12, absTol=0.0), tol=1e-8, pc=pc)


@pytest.mark.parametrize("m", [20, 90, 520])
def test_bicgstab_resident_column_deltas(ctx, monkeypatch, m):
    check(ctx, monkeypatch, fx.BICGSTAB, P.varcoef_fv(m)[0],
          dict(maxIter=12, relTol=1e-12, absTol=0.0), tol=1e-8, transposed=True)


@pytest.mark.parametrize("prm", [
    dict(maxIter=0), dict(maxIter=1), dict(maxIter=7, relTol=1e-12), dict(maxIter=14, minIter=5),
    dict(maxIter=100, relTol=1e-3, savIter=5), dict(maxIter=200, relTol=1e-2, restart=2),
    dict(maxIter=10, minIter=10)])
@pytest.mark.parametrize("m", [16, 70])
def test_bicgstab_resident_stops(ctx, monkeypatch, m, prm):
    prm = {"absTol": 0.0, "relTol": 1e-30, **prm}
    check(ctx, monkeypatch, fx.BICGSTAB, P.poisson2d(m), prm, tol=1e-8)


@pytest.mark.parametrize("m", [16, 70])
def test_bicgstab_resident_converges(ctx, monkeypatch, m):
    """To a tolerance: the true residual, whatever the count."""
    A = P.convdiff2d(m)
    xs = np.random.default_rng(m).uniform(-1, 1, A.nrow)
    b = A.matvec(xs)
    for resident in (True, False):
        r, x, h = solve(ctx, monkeypatch, resident, fx.BICGSTAB, A,
                        dict(maxIter=2000, relTol=1e-10, absTol=0.0), b=b)
        assert r.retcode == 0 and len(h) == r.numIter
        assert np.linalg.norm(b - A.matvec(x)) <= 1e-9 * np.linalg.norm(b) * 10


@pytest.mark.parametrize("m", [16, 70])
def test_bicgstab_resident_zero_rhs_and_exact_start(ctx, monkeypatch, m):
    A = P.poisson2d(m)
    prm = dict(maxIter=50, relTol=1e-8, absTol=1e-14)
    b = np.zeros(A.nrow)
    got = [solve(ctx, monkeypatch, res, fx.BICGSTAB, A, prm, b=b)[:2] for res in (True, False)]
    assert got[0][0].retcode == got[1][0].retcode and got[0][0].numIter == got[1][0].numIter
    assert np.array_equal(got[0][1], got[1][1])


def test_bicgstab_resident_one_unknown(ctx, monkeypatch):
    """The first half step solves it, and omega is 0 / 0 (the recurrence has
    no guard there): not a number on either path."""
    out = []
    for resident in (True, False):
        if not resident:
            monkeypatch.setenv("FASPXX_FX_NORESIDENT", "1")
        M = fx.Csr.from_problem(ctx, P.poisson2d(1))
        s = fx.Solver(ctx, fx.BICGSTAB)
        s.Setup(M, fx.Precond(ctx, "jacobi", M, 1.0, 1), fx.params(maxIter=3, relTol=1e-12))
        x = fx.Vec(ctx, 1)
        r = s.Solve(fx.Vec.from_numpy(ctx, np.array([0.1])), x)
        out.append((r.retcode, r.numIter, np.isnan(x.numpy()[0])))
    assert out[0] == out[1] and out[0][2]
