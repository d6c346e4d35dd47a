"""The device kernels of the sparse algebra at the edges of their work split:
products whose rows have as many candidates as a row's table holds, one more,
and rows of R that repeat a column; row blocks of matrices built on the
device, with row counts around a tile and rows around a block's capacity."""
import numpy as np
import pytest

from faspxx_amd import fx
from oracle import Matrix
from test_gpu_spalg import check, dev

pytestmark = pytest.mark.gpu


def matrix(oracle, lens, mcol, seed, repeat=False):
    """Rows of the given lengths, columns in no order; `repeat` allows a
    column several times in a row."""
    rng = np.random.default_rng(seed)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    ci = np.concatenate([rng.choice(mcol, int(k), replace=repeat) for k in lens] or [[]])
    ci = ci.astype(np.uint32)
    n = len(lens)
    dp = np.zeros(n, np.uint32)
    for i in range(n):
        hit = np.flatnonzero(ci[rp[i]:rp[i + 1]] == i)
        dp[i] = rp[i] + hit[0] if len(hit) else 0
    return Matrix(n, mcol, rp, ci, rng.uniform(-1, 1, len(ci)), dp)


# rows of L times rows of R: candidates per row of L R
@pytest.mark.parametrize("repeat", [False, True])
@pytest.mark.parametrize("k,r", [(1, 1), (7, 9), (8, 8), (5, 13), (4, 17), (1, 64), (64, 1),
                                 (8, 64), (27, 19), (1, 512), (512, 1), (513, 1), (3, 171),
                                 (5, 128)])
def test_mult_candidates(ctx, oracle, k, r, repeat):
    rng = np.random.default_rng(k * 1000 + r)
    n = 1031
    # half of the rows as long as given, the others shorter, some empty
    ll = np.where(rng.random(513) < 0.5, k, rng.integers(0, k + 1, 513))
    rl = np.where(rng.random(n) < 0.5, r, rng.integers(0, r + 1, n))
    L = matrix(oracle, ll, n, 1, repeat)
    for mcol in (600, 40000):
        R = matrix(oracle, rl, mcol, 2, repeat)
        check(fx.Csr.mult(dev(ctx, L), dev(ctx, R)), oracle.mat_mult(L, R))
    S = Matrix(L.nrow, L.mcol, L.rp, L.ci, None, L.dp)
    check(fx.Csr.mult(dev(ctx, S), dev(ctx, R)), oracle.mat_mult(S, R), values=False)


def test_mult_without_entries(ctx, oracle):
    L = matrix(oracle, [2, 2, 2], 4, 3)
    L.ci[:] = [0, 1, 1, 0, 0, 1]
    R = matrix(oracle, [0, 0, 3, 1], 4, 4)
    C = fx.Csr.mult(dev(ctx, L), dev(ctx, R))
    assert C.nnz == 0


@pytest.mark.parametrize("k", [32768, 65537])
def test_mult_refuses_too_many_candidates(ctx, k):
    """One row of L that selects one row of 65536 entries k times: 2^31
    candidates, and more than a 32-bit count holds."""
    m = 65536
    L = fx.Csr(ctx, 1, 1, np.array([0, k]), np.zeros(k, np.uint32), np.ones(k))
    R = fx.Csr(ctx, 1, m, np.array([0, m]), np.arange(m), np.ones(m))
    with pytest.raises(fx.FxError) as e:
        fx.Csr.mult(L, R)
    assert e.value.code == -20  # ERROR_ALLOC_MEM


LENGTHS = {
    "short": lambda n, rng: rng.integers(0, 9, n),
    "empty but one": lambda n, rng: np.where(np.arange(n) == n // 2, 5, 0),
    "seven": lambda n, rng: np.full(n, 7),
    "eight": lambda n, rng: np.full(n, 8),
    "about a block": lambda n, rng: np.where(rng.random(n) < 0.02, rng.integers(1785, 1800, n),
                                             rng.integers(0, 4, n)),
    "long last": lambda n, rng: np.where(np.arange(n) >= n - 3, 1793, 3),
}


@pytest.mark.parametrize("n", [1, 255, 257, 2047, 2048, 2049, 4096, 10007])
@pytest.mark.parametrize("name", list(LENGTHS))
def test_device_row_blocks(ctx, oracle, n, name):
    """A^T of a matrix whose columns have the given lengths, and what is
    built from it: entries and products with a vector."""
    rng = np.random.default_rng(n)
    mcol = 2500
    At = matrix(oracle, LENGTHS[name](n, rng), mcol, n + 1)
    if At.nnz == 0:
        pytest.skip("no entries")
    order = np.argsort(At.ci, kind="stable")  # A: At's entries by column
    rows = np.repeat(np.arange(n), np.diff(At.rp.astype(np.int64)))
    A = fx.Csr(ctx, mcol, n, np.concatenate([[0], np.cumsum(np.bincount(At.ci, minlength=mcol))]),
               rows[order].astype(np.uint32), At.va[order])
    T = A.transpose()
    rp, ci, va, _ = T.download()
    assert np.array_equal(rp, At.rp)
    sums = np.zeros((2, n))
    x = rng.uniform(-1, 1, mcol)
    for i in range(n):
        s, e = At.rp[i], At.rp[i + 1]
        o = np.argsort(At.ci[s:e], kind="stable")
        assert np.array_equal(ci[s:e], At.ci[s:e][o]) and np.array_equal(va[s:e], At.va[s:e][o])
        sums[0, i] = At.va[s:e] @ x[At.ci[s:e]]
        sums[1, i] = np.abs(At.va[s:e] * x[At.ci[s:e]]).sum()
    y = fx.Vec(ctx, n)
    T.Apply(fx.Vec.from_numpy(ctx, x), y)
    # two summation orders of up to 1800 products: 1800 * 2^-53 each
    assert np.all(np.abs(y.numpy() - sums[0]) <= 2 * 1800 * 2.0**-53 * sums[1])
    two = fx.Csr.add(1.0, T, 1.0, T)
    y2 = fx.Vec(ctx, n)
    two.Apply(fx.Vec.from_numpy(ctx, x), y2)
    assert np.all(np.abs(y2.numpy() - 2 * sums[0]) <= 4 * 1800 * 2.0**-53 * sums[1])
