"""BiCGStab's iteration count on the 1024 x 1024 upwind system is set by
rounding: right-hand sides an ulp apart spread it over some 280 iterations, so
a band of a few counts cannot tell one order of summation from another.  What
two correct loops share is the distribution: the means over right-hand sides
an ulp apart agree within three standard errors of their difference."""
import numpy as np
import pytest

from faspxx_amd import fx
from perturb import ulp_perturbed

pytestmark = pytest.mark.gpu


def test_counts_of_both_loops(ctx, monkeypatch, problems):
    pr, n = problems(3, None), 24
    counts = []
    for resident in (True, False):
        if not resident:
            monkeypatch.setenv("FASPXX_FX_NORESIDENT", "1")
        M = fx.Csr.from_problem(ctx, pr.A)
        pc = fx.Precond(ctx, "jacobi", M, 1.0, 1)
        s = fx.Solver(ctx, fx.BICGSTAB)
        s.Setup(M, pc, fx.params(maxIter=5000, relTol=1e-8, absTol=0.0))
        got = []
        for k in range(n):
            x = fx.Vec(ctx, pr.A.nrow)
            r = s.Solve(fx.Vec.from_numpy(ctx, ulp_perturbed(pr.b, k)), x)
            assert r.retcode == 0 and s.last_resident == resident
            got.append(r.numIter)
        print("resident" if resident else "kernel by kernel", sorted(got))
        counts.append(np.array(got, float))
    a, b = counts
    error = np.sqrt((a.var(ddof=1) + b.var(ddof=1)) / n)
    assert abs(a.mean() - b.mean()) <= 3 * error
