"""Resident loops report that they ran, and a solve whose launch is refused or
whose wait gives up goes on kernel by kernel: one that starts over gives the
bits of FASPXX_FX_NORESIDENT=1, whose whole work it then does."""
import numpy as np
import pytest

from faspxx_amd import fx
from faspxx_amd import problems as P

pytestmark = pytest.mark.gpu


class Case:
    """A solver kept over several solves of one system, from the same x."""

    def __init__(self, ctx, kind, A, **prm):
        self.ctx, self.A = ctx, A
        rng = np.random.default_rng(A.nrow)
        self.b, self.x0 = A.matvec(rng.uniform(-1, 1, A.nrow)), rng.uniform(-1, 1, A.nrow)
        M = fx.Csr.from_problem(ctx, A)
        if kind == "ir":
            inner = fx.params(maxIter=20000, relTol=prm.pop("inner", 1e-4), absTol=0.0)
            self.s = fx.IR(ctx, M, 1.0, fx.params(maxIter=50, absTol=0.0, **prm), inner)
        else:
            pc = fx.Precond(ctx, "jacobi", M, 1.0, 1)
            self.s = fx.Solver(ctx, kind)
            self.s.Setup(M, pc, fx.params(absTol=0.0, **prm))
            self.keep = pc

    def solve(self):
        x = fx.Vec.from_numpy(self.ctx, self.x0)
        r = self.s.Solve(fx.Vec.from_numpy(self.ctx, self.b), x)
        return (r[0] if isinstance(r, tuple) else r), x.numpy(), self.s.last_resident


CASES = [(fx.CG, dict(maxIter=3000, relTol=1e-8)), (fx.BICGSTAB, dict(maxIter=40, relTol=1e-30)),
         ("ir", dict(relTol=1e-12))]


@pytest.mark.parametrize("kind,prm", CASES)
@pytest.mark.parametrize("m", [32, 70])
def test_resident_is_reported(ctx, monkeypatch, kind, prm, m):
    assert Case(ctx, kind, P.poisson2d(m), **prm).solve()[2]
    monkeypatch.setenv("FASPXX_FX_NORESIDENT", "1")
    assert not Case(ctx, kind, P.poisson2d(m), **prm).solve()[2]


@pytest.mark.parametrize("kind,prm", CASES)
@pytest.mark.parametrize("m,env", [(32, "LAUNCHES"), (70, "LAUNCHES"), (70, "FAIL"),
                                   (200, "FAIL")])
def test_starts_over(ctx, monkeypatch, kind, prm, m, env):
    """A launch refused at once, and one whose workgroups leave as after a wait
    that gave up: kernel by kernel from the caller's x, and again so on the
    next solve."""
    monkeypatch.setenv("FASPXX_FX_NORESIDENT", "1")
    r0, x0, _ = Case(ctx, kind, P.poisson2d(m), **prm).solve()
    monkeypatch.delenv("FASPXX_FX_NORESIDENT")
    monkeypatch.setenv("FASPXX_FX_RESIDENT_" + env, "1" if env == "FAIL" else "0")
    c = Case(ctx, kind, P.poisson2d(m), **prm)
    for _ in range(2):
        r, x, resident = c.solve()
        assert not resident
        assert (r.retcode, r.numIter) == (r0.retcode, r0.numIter)
        assert np.array_equal(x, x0)


def test_later_launch_refused_cg(ctx, monkeypatch):
    """The first 2048 iterations resident, the rest kernel by kernel."""
    monkeypatch.setenv("FASPXX_FX_RESIDENT_LAUNCHES", "1")
    c = Case(ctx, fx.CG, P.varcoef_fv(1000)[0], maxIter=20000, relTol=1e-11)
    r, x, resident = c.solve()
    assert r.retcode == 0 and r.numIter > 2048 and not resident
    r0 = c.b - c.A.matvec(c.x0)
    assert np.linalg.norm(c.b - c.A.matvec(x)) <= 1.001e-11 * np.linalg.norm(r0)


def test_later_launch_refused_ir(ctx, monkeypatch):
    """An inner loop of more than 2048 iterations starts over."""
    A, prm = P.varcoef_fv(1000)[0], dict(relTol=1e-12, inner=1e-8)
    monkeypatch.setenv("FASPXX_FX_NORESIDENT", "1")
    r0, x0, _ = Case(ctx, "ir", A, **prm).solve()
    monkeypatch.delenv("FASPXX_FX_NORESIDENT")
    monkeypatch.setenv("FASPXX_FX_RESIDENT_LAUNCHES", "1")
    r, x, resident = Case(ctx, "ir", A, **prm).solve()
    assert not resident and (r.retcode, r.numIter) == (r0.retcode, r0.numIter)
    assert np.array_equal(x, x0)


def test_one_workgroup_solves_overlap():
    """Solves of one workgroup on two contexts run side by side: both take less
    than one after the other would."""
    import threading
    import time

    A = P.poisson2d(44)
    cs = [Case(fx.Context(0), fx.CG, A, maxIter=800, minIter=800) for _ in range(2)]
    for c in cs:
        c.b, c.x0 = 1e80 * c.b, np.zeros(A.nrow)  # (p, q) of 800 iterations stays above 1e-40
        r, _, resident = c.solve()
        assert resident and r.numIter == 800

    def seconds(which):
        gate = threading.Barrier(len(which) + 1)

        def work(c):
            gate.wait()
            for _ in range(4):
                c.solve()
        ts = [threading.Thread(target=work, args=(c,)) for c in which]
        for t in ts:
            t.start()
        gate.wait()
        t0 = time.perf_counter()
        for t in ts:
            t.join()
        return time.perf_counter() - t0

    alone, both = min(seconds(cs[:1]) for _ in range(3)), min(seconds(cs) for _ in range(3))
    assert both < 1.6 * alone
    for c in cs:
        c.ctx.close()
