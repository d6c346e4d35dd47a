"""Reductions at the edges of their work split: one workgroup (up to 1024
elements), the groups of 32 workgroups that are counted, more partials than
one summing pass takes (1024 workgroups), and more than four elements a
thread (2^21); each form twice, so that a count left over would show."""
import ctypes as C
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 255, 256, 1024, 1025, 32 * 1024, 32 * 1024 + 1, 64 * 1024 + 3,
         1024 * 1024, 1024 * 1024 + 1, (1 << 21) - 1, (1 << 21) + 5, (1 << 22) + 1027]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", SIZES)
def test_reductions(ctx, n, dtype):
    from faspxx_amd import fx
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n).astype(dtype)
    y = rng.standard_normal(n).astype(dtype)
    x[n // 3], y[n - 1] = 7.5, -8.25
    X, Y = fx.Vec.from_numpy(ctx, x), fx.Vec.from_numpy(ctx, y)
    x8, y8 = x.astype(np.float64), y.astype(np.float64)
    # double sums by one fma per element, at most n / 2^19 + 2048 of them in one
    # chain: their error is below chain * 2^-53 * sum |x y|
    u = (n / 2**19 + 2100) * 2.0**-53
    dot, dabs = math.fsum(x8 * y8), math.fsum(np.abs(x8 * y8))
    nrm = math.sqrt(math.fsum(x8 * x8))
    dev = fx.Vec(ctx, 2, fx.F64)
    ptr = fx.load().fx_vec_data(dev.h)
    for _ in range(2):
        d = X.Dot(Y)
        assert abs(d - dot) <= u * dabs + 2.0**-52 * dabs
        n2 = X.Norm2()
        assert abs(n2 - nrm) <= (u + 2.0**-52) * nrm
        assert Y.NormInf() == np.abs(y8).max()
        assert X.Max() == x8.max() and X.Min() == x8.min()
        fx._chk(fx.load().fx_dot_dev(ctx.h, X.h, Y.h, C.c_void_p(ptr)))
        fx._chk(fx.load().fx_norm2_dev(ctx.h, X.h, C.c_void_p(ptr + 8)))
        assert list(dev.numpy()) == [d, n2]
    # the updates reduce what they store, bit for bit like the plain forms
    z = fx.Vec.from_numpy(ctx, y)
    assert z.AXPY_Norm2(0.5, X) == z.Norm2()
    np.testing.assert_array_equal(z.numpy(), y + dtype(0.5) * x)
    assert z.AXPY_Dot(-0.25, X, Y) == z.Dot(Y)
    assert z.AXPY_Dot(-0.25, X, z) == z.Dot(z)
    assert z.XPAY_Norm2(0.75, X) == z.Norm2()


def test_reductions_of_special_values(ctx):
    from faspxx_amd import fx
    n = 40000
    for bad, where in ((np.nan, 0), (np.inf, n - 1), (-np.inf, 20000)):
        x = np.ones(n)
        x[where] = bad
        X = fx.Vec.from_numpy(ctx, x)
        assert not math.isfinite(X.Dot(X)) and not math.isfinite(X.Norm2())
        if not math.isnan(bad):
            assert X.NormInf() == math.inf
    e = fx.Vec(ctx, 0, fx.F64)
    assert e.Dot(e) == 0.0 and e.Norm2() == 0.0 and e.NormInf() == 0.0
