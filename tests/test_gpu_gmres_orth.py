"""The fused GMRES / FGMRES orthogonalisation (one workgroup; dot products,
triangular solve and update; a kernel per step for long cycles) against the
per-operation solver, whose modified Gram-Schmidt runs step by step.

Tolerance: after a fixed number of iterations on these systems the oracle's
GMRES and FGMRES iterates move by at most 3e-14 relative when b moves by an
ulp, and a sum in another order is a change of that size per step, so 1e-11
leaves three orders of magnitude."""
import numpy as np
import pytest

from faspxx_amd import fx
from faspxx_amd import problems as P

pytestmark = pytest.mark.gpu


def rect(m, k):
    """Upwind-like 5-point system on an m x k grid (any parity of rows)."""
    i = np.arange(m * k, dtype=np.int64)
    ix, iy = i % m, i // m
    cols = np.stack([i - m, i - 1, i, i + 1, i + m], axis=1)
    mask = np.stack([iy > 0, ix > 0, np.ones(m * k, bool), ix < m - 1, iy < k - 1], axis=1)
    vals = np.tile([-1.4, -1.9, 5.3, -0.9, -1.0], (m * k, 1))
    return P._from_dense_stencil(m * k, cols, vals, mask)


def run(ctx, monkeypatch, kind, A, prm, ops):
    if ops:
        monkeypatch.setenv("FASPXX_FX_NO_FAST", "1")
    M = fx.Csr.from_problem(ctx, A)
    s = fx.Solver(ctx, kind)
    s.Setup(M, fx.Precond(ctx, "jacobi", M, 1.0, 1), fx.params(**prm))
    x = fx.Vec(ctx, A.nrow)
    b = np.random.default_rng(A.nrow).uniform(-1, 1, A.nrow)
    res = s.Solve(fx.Vec.from_numpy(ctx, b), x)
    monkeypatch.delenv("FASPXX_FX_NO_FAST", raising=False)
    assert s.last_path == ("ops" if ops else "fused")
    return res, x.numpy(), s.history()


# one row and two, the last size of one workgroup and the first beyond it (even and
# odd rows), a pack per thread in one and several workgroups, its last size and
# the first with four, the last with four and the first with passes
@pytest.mark.parametrize("m,k", [(1, 1), (2, 1), (31, 33), (32, 64), (683, 3), (41, 50), (77, 107),
                                 (512, 512), (263, 997), (1024, 1024), (1025, 1023)])
@pytest.mark.parametrize("kind", [fx.GMRES, fx.FGMRES])
def test_orthogonalisation_sizes(ctx, monkeypatch, kind, m, k):
    A = rect(m, k)
    prm = dict(maxIter=min(33, A.nrow), relTol=1e-30, absTol=0.0)
    (r1, x1, h1), (r0, x0, h0) = (run(ctx, monkeypatch, kind, A, prm, o) for o in (False, True))
    assert r1.numIter == r0.numIter and r1.retcode == r0.retcode
    assert np.linalg.norm(x1 - x0) <= 1e-11 * np.linalg.norm(x0)
    keep = h0[:len(h1)] > 1e-9 * h0[0]  # a solved system's last estimates are rounding
    assert np.allclose(h1[:len(h0)][keep], h0[:len(h1)][keep], rtol=1e-9, atol=0)


# (lengths under 3 wrap around in the reference's adaption, restart - 3 unsigned)
@pytest.mark.parametrize("restart", [3, 5, 62, 63, 64, 70])
@pytest.mark.parametrize("m,k", [(40, 50), (61, 67)])
def test_orthogonalisation_cycle_lengths(ctx, monkeypatch, restart, m, k):
    A = rect(m, k)
    prm = dict(maxIter=2 * restart + 3, relTol=1e-12, absTol=0.0, restart=restart,
               maxRestart=restart, minRestart=restart)
    (r1, x1, _), (r0, x0, _) = (run(ctx, monkeypatch, fx.GMRES, A, prm, o) for o in (False, True))
    assert abs(r1.numIter - r0.numIter) <= 1
    assert np.linalg.norm(x1 - x0) <= 1e-11 * np.linalg.norm(x0)
