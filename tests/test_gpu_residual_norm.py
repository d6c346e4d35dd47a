"""Residual's max-norm on both sides of the size from which its partials are
combined by a second launch (f64 131072 rows, f32 196608): b - A x where some
|x_i| >= 1e-20, wherever it is, and b itself where there is none."""
import numpy as np
import pytest

from test_gpu_rowvalues import diag

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1025, 32 * 1024 + 1, 128 * 1024, 128 * 1024 + 1, 192 * 1024,
                               192 * 1024 + 1, 500003])
def test_residual_shortcut(ctx, n):
    from faspxx_amd import fx
    M = fx.Csr.from_problem(ctx, diag(n))
    M.make_f32()
    for dt, npdt in ((fx.F64, np.float64), (fx.F32, np.float32)):
        b = np.random.default_rng(n).uniform(1, 2, n).astype(npdt)
        vb, r = fx.Vec.from_numpy(ctx, b, dt), fx.Vec(ctx, n, dt)
        a = npdt(3.0 / 7.0)
        for at in (None, 0, n // 2, n - 1):
            x = np.full(n, 1e-21, npdt)
            if at is not None:
                x[at] = -1e-3
            M.Residual(vb, fx.Vec.from_numpy(ctx, x, dt), r)
            want = b.copy()
            if at is not None:  # fma(-a, x, b) in double, rounded once to the type
                exact = b.astype(np.longdouble) - np.longdouble(a) * x.astype(np.longdouble)
                want = exact.astype(npdt)
            got = r.numpy()
            assert np.all(np.abs(got - want) <= np.finfo(npdt).eps * np.abs(want))
            assert np.array_equal(got, b) == (at is None)


def test_reductions_on_a_callers_stream_behind_a_busy_null_stream():
    """A context made on a non-blocking stream while the null stream is busy:
    its first reductions find their counts cleared."""
    import torch
    from faspxx_amd import fx
    st = torch.cuda.Stream()
    a = torch.randn(4096, 4096, device="cuda")
    with torch.cuda.stream(st):
        t = torch.arange(100000, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        for _ in range(5):
            with torch.cuda.stream(torch.cuda.default_stream()):
                for _ in range(4):
                    a @ a
            c = fx.Context(0, stream=st.cuda_stream)
            x = fx.Vec.wrap(c, t.data_ptr(), t.numel())
            assert [x.NormInf() for _ in range(3)] == [99999.0] * 3
            x.close()
            c.close()
        torch.cuda.synchronize()
