"""Which solves run resident: those that are faster so.  Long rows gather past
the L2 entry by entry and stay kernel by kernel; where they run resident the
result is the kernel-by-kernel one."""
import itertools

import numpy as np
import pytest

from faspxx_amd import fx
from faspxx_amd import problems as P
from test_gpu_resident import check

pytestmark = pytest.mark.gpu


def stencil(m, offsets, seed=0):
    """Symmetric positive definite on len(offsets[0]) dimensions of m points:
    the offsets and their negatives, weights that differ from row to row."""
    dim = len(offsets[0])
    n, i = m ** dim, np.arange(m ** dim, dtype=np.int64)
    at = [(i // m ** d) % m for d in range(dim)]
    both = [tuple(-a for a in o) for o in offsets] + [(0,) * dim] + list(offsets)
    both.sort(key=lambda o: sum(a * m ** d for d, a in enumerate(o)))
    cols, vals, mask = [], [], []
    for o in both:
        c = i + sum(a * m ** d for d, a in enumerate(o))
        w = 0.5 + ((i + c + seed) * 2654435761 % 1000003) / 2000006.0
        cols.append(c)
        vals.append(-w if any(o) else np.full(n, 1.0 + len(both)))
        mask.append(np.all([(a + d >= 0) & (a + d < m) for a, d in zip(at, o)], axis=0))
    return P._from_dense_stencil(n, np.stack(cols, 1), np.stack(vals, 1), np.stack(mask, 1))


def box(m, dim):
    """3^dim entries per row."""
    half = [o for o in itertools.product((-1, 0, 1), repeat=dim) if o > (0,) * dim]
    return stencil(m, half)


PLANE = [(1, 0), (0, 1), (1, 1), (1, -1), (2, 0), (0, 2), (2, 1), (1, 2), (2, -1), (1, -2)]


def star(m, entries):
    return stencil(m, PLANE[:entries // 2])


def resident(ctx, kind, A):
    M = fx.Csr.from_problem(ctx, A)
    b, x = fx.Vec.from_numpy(ctx, np.ones(A.nrow)), fx.Vec(ctx, A.nrow)
    if kind == "ir":
        s = fx.IR(ctx, M, 1.0, fx.params(maxIter=2, relTol=1e-12), fx.params(maxIter=3))
        s.Solve(b, x)
        return s.last_resident
    pc = fx.Precond(ctx, "jacobi", M, 1.0, 1)
    s = fx.Solver(ctx, kind)
    s.Setup(M, pc, fx.params(maxIter=3, relTol=1e-30))
    s.Solve(b, x)
    return s.last_resident


@pytest.mark.parametrize("name,make,cg,bi,ir", [
    # one workgroup of one row per thread: up to 17 entries; of two: up to 11
    ("17 entries, 30^2", lambda: star(30, 17), True, True, True),
    ("19 entries, 30^2", lambda: star(30, 19), False, False, False),
    ("27 entries, 9^3", lambda: box(9, 3), False, False, False),
    ("11 entries, 45^2", lambda: star(45, 11), True, True, True),
    ("13 entries, 45^2", lambda: star(45, 13), False, False, False),
    # several workgroups: up to 11 entries, two rows per thread 11 near, 9 far
    ("11 entries, 70^2", lambda: star(70, 11), True, True, True),
    ("13 entries, 70^2", lambda: star(70, 13), False, False, False),
    ("27 entries, 20^3", lambda: box(20, 3), False, False, False),
    ("11 entries, 520^2", lambda: star(520, 11), True, True, True),
    ("9 entries far, 66^3", lambda: stencil(66, [(1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 0)]),
     True, True, True),
    ("11 entries far, 66^3", lambda: stencil(66, [(1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 0),
                                                  (1, 0, 1)]), False, False, False),
    # four rows per thread
    ("5 entries, 800^2", lambda: star(800, 5), True, True, True),
    ("9 entries near, 800^2", lambda: star(800, 9), True, True, True),
    ("7 entries far, 82^3", lambda: stencil(82, [(1, 0, 0), (0, 1, 0), (0, 0, 1)]),
     True, True, False),
    # eight: CG where rows of five entries reach no further than their workgroup
    ("5 entries, 1100^2", lambda: star(1100, 5), False, False, False),
    ("5 entries, 1160^2", lambda: star(1160, 5), True, False, False),
    ("9 entries, 1160^2", lambda: star(1160, 9), False, False, False),
    ("7 entries far, 110^3", lambda: stencil(110, [(1, 0, 0), (0, 1, 0), (0, 0, 1)]),
     False, False, False),
    ("row values, 101^3", lambda: P.poisson3d(101), True, True, True),
    ("row values, 102^3", lambda: P.poisson3d(102), True, False, False),
    ("row values, 128^3", lambda: P.poisson3d(128), True, False, False),
    ("5 entries, 1449^2", lambda: star(1449, 5), False, False, False),  # does not fit
])
def test_resident_routes(ctx, name, make, cg, bi, ir):
    A = make()
    assert [resident(ctx, k, A) for k in (fx.CG, fx.BICGSTAB, "ir")] == [cg, bi, ir]


@pytest.mark.parametrize("pc", ["jacobi", "identity"])
@pytest.mark.parametrize("m", [1160, 1448])
def test_cg_eight_rows_per_thread(ctx, monkeypatch, m, pc):
    """Values re-read from memory, a ragged and the largest last workgroup."""
    check(ctx, monkeypatch, fx.CG, P.varcoef_fv(m)[0],
          dict(maxIter=60, relTol=1e-30, absTol=0.0), pc=pc)


@pytest.mark.parametrize("m,entries", [(30, 17), (45, 11), (70, 11), (520, 11), (800, 9)])
def test_longest_resident_rows(ctx, monkeypatch, m, entries):
    A = star(m, entries)
    check(ctx, monkeypatch, fx.CG, A, dict(maxIter=40, relTol=1e-30, absTol=0.0))
    check(ctx, monkeypatch, fx.BICGSTAB, A, dict(maxIter=8, relTol=1e-30, absTol=0.0), tol=1e-8)
