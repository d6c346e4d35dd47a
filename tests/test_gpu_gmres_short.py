"""GMRES and FGMRES with the shortest cycles, on both sides of the length from
which a column is orthogonalised in three kernels (4), against the
per-operation solver.  The tolerance is that of test_gpu_gmres_orth.py."""
import numpy as np
import pytest

from faspxx_amd import fx
from test_gpu_gmres_orth import rect, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [fx.GMRES, fx.FGMRES])
@pytest.mark.parametrize("restart", [3, 4])
@pytest.mark.parametrize("m,k", [(61, 67), (300, 301)])
def test_short_cycles(ctx, monkeypatch, kind, restart, m, k):
    prm = dict(maxIter=3 * restart + 1, relTol=1e-30, absTol=0.0, restart=restart,
               maxRestart=restart, minRestart=restart)
    A = rect(m, k)
    (r1, x1, _), (r0, x0, _) = (run(ctx, monkeypatch, kind, A, prm, o) for o in (False, True))
    assert r1.numIter == r0.numIter
    assert np.linalg.norm(x1 - x0) <= 1e-11 * np.linalg.norm(x0)
