"""Row blocks of a matrix built on the device where the launches that form them
change: one tile of 2048 rows, up to 32, more."""
import numpy as np
import pytest

from faspxx_amd import fx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2048, 2049, 4097, 32 * 2048, 32 * 2048 + 1, 33 * 2048 + 5])
@pytest.mark.parametrize("long", [0.0, 0.01])
def test_product_with_a_transpose(ctx, n, long):
    """A^T of 3000 rows by n: every row of A^T is a row of the table's blocks,
    some longer than a block."""
    rng = np.random.default_rng(n)
    m = 3000
    lens = np.where(rng.random(n) < long, rng.integers(1780, 1800, n), rng.integers(0, 9, n))
    lens[-1] = max(lens[-1], 1)
    rows = np.repeat(np.arange(n), lens)  # of A^T
    cols = rng.integers(0, m, rows.shape[0])
    key = np.unique(rows * m + cols)
    rows, cols = key // m, key % m
    va = rng.uniform(-1, 1, key.shape[0])
    order = np.lexsort((rows, cols))
    rp = np.concatenate([[0], np.cumsum(np.bincount(cols, minlength=m))])
    A = fx.Csr(ctx, m, n, rp, rows[order].astype(np.uint32), va[order])
    T = A.transpose()
    trp, tci, tva, _ = T.download()
    assert np.array_equal(trp, np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))]))
    assert np.array_equal(tci, cols) and np.array_equal(tva, va)
    x = rng.uniform(-1, 1, m)
    y = fx.Vec(ctx, n)
    y.set(7.0)
    T.Apply(fx.Vec.from_numpy(ctx, x), y)
    want = np.bincount(rows, va * x[cols], n)
    size = np.bincount(rows, np.abs(va * x[cols]), n)
    # two summation orders of up to 1800 products: 1800 * 2^-53 each
    assert np.all(np.abs(y.numpy() - want) <= 2 * 1800 * 2.0**-53 * size)
