"""Row values: a row-pattern matrix whose rows of one pattern hold the same
values is read from a dictionary, with the bits of the entry-by-entry form
(FASPXX_FX_NOROWVAL=1), and is read entry by entry again once its values
change."""
import numpy as np
import pytest

from faspxx_amd import problems as P

pytestmark = pytest.mark.gpu


def box2d(m, k):
    """9-point box stencil on an m x k grid: rows of up to 9 entries."""
    i = np.arange(m * k, dtype=np.int64)
    ix, iy = i % m, i // m
    offs = [(dx, dy) for dy in (-1, 0, 1) for dx in (-1, 0, 1)]
    cols = np.stack([i + dx + m * dy for dx, dy in offs], axis=1)
    mask = np.stack([(ix + dx >= 0) & (ix + dx < m) & (iy + dy >= 0) & (iy + dy < k)
                     for dx, dy in offs], axis=1)
    vals = np.tile([0.1, -0.7, 0.3, -1.1, 8.0 / 3.0, -0.9, 0.2, -0.6, 0.4], (m * k, 1))
    return P._from_dense_stencil(m * k, cols, vals, mask)


def diag(n):
    i = np.arange(n, dtype=np.int64)[:, None]
    return P._from_dense_stencil(n, i, np.full((n, 1), 3.0 / 7.0), np.ones((n, 1), bool))


# the kernels use row values above 256 * 1024 rows: the last sizes without
# them, the first with them, ragged last workgroups, rows of one entry, of up
# to 8 (padded dictionary) and of up to 9
SYSTEMS = {
    "diag_262144": lambda: diag(262144), "diag_262145": lambda: diag(262145),
    "poisson2d_513": lambda: P.poisson2d(513), "poisson3d_65": lambda: P.poisson3d(65),
    "convdiff_530": lambda: P.convdiff2d(530), "box_517x511": lambda: box2d(517, 511),
    "box_3x87500": lambda: box2d(3, 87500), "poisson2d_33": lambda: P.poisson2d(33),
}


def make(ctx, A, monkeypatch, off):
    from faspxx_amd import fx
    if off:
        monkeypatch.setenv("FASPXX_FX_NOROWVAL", "1")
    M = fx.Csr.from_problem(ctx, A)
    monkeypatch.delenv("FASPXX_FX_NOROWVAL", raising=False)
    M.make_f32()
    return M


def products(ctx, M, n):
    """Apply and Residual in both precisions."""
    from faspxx_amd import fx
    out = []
    for dt, npdt in ((fx.F64, np.float64), (fx.F32, np.float32)):
        x = np.random.default_rng(n).uniform(-1, 1, n).astype(npdt)
        vx, vb = fx.Vec.from_numpy(ctx, x, dt), fx.Vec.from_numpy(ctx, x[::-1].copy(), dt)
        y, r = fx.Vec(ctx, n, dt), fx.Vec(ctx, n, dt)
        M.Apply(vx, y)
        M.Residual(vb, vx, r)
        out += [y.numpy(), r.numpy()]
    return out


@pytest.mark.parametrize("name", list(SYSTEMS))
def test_row_values_same_bits(ctx, monkeypatch, name):
    import torch
    A = SYSTEMS[name]()
    n = A.nrow
    M, M0 = make(ctx, A, monkeypatch, False), make(ctx, A, monkeypatch, True)
    assert M.layout == M0.layout == "pattern"

    def same():
        for a, b in zip(products(ctx, M, n), products(ctx, M0, n)):
            assert np.array_equal(a, b)

    same()
    for m in (M, M0):
        m.shift_diag(0.25)
    same()
    M, M0 = make(ctx, A, monkeypatch, False), make(ctx, A, monkeypatch, True)
    v = torch.tensor(np.random.default_rng(5).uniform(1, 2, A.nnz), device="cuda")
    torch.cuda.synchronize()
    for m in (M, M0):
        m.set_values_dev(v.data_ptr())
    ctx.sync()
    same()


def test_row_values_written_through_the_pointer(ctx, monkeypatch):
    from faspxx_amd import fx
    A = P.poisson2d(515)
    M, M0 = make(ctx, A, monkeypatch, False), make(ctx, A, monkeypatch, True)
    v = np.random.default_rng(6).uniform(1, 2, A.nnz)
    for m in (M, M0):
        fx.Vec.wrap(ctx, m.values_ptr, A.nnz).upload(v)
    a, b = products(ctx, M, A.nrow), products(ctx, M0, A.nrow)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


def test_captured_apply_follows_new_values():
    """A product captured in a graph while the matrix has row values reads
    the new values once they are set, on every replay."""
    import torch
    from faspxx_amd import fx
    A = P.poisson3d(65)
    n = A.nrow
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        c = fx.Context(0, stream=st.cuda_stream)
        M = fx.Csr.from_problem(c, A)
        x = torch.tensor(np.random.default_rng(1).uniform(-1, 1, n), device="cuda")
        y = torch.zeros_like(x)
        v = torch.tensor(np.random.default_rng(2).uniform(1, 2, A.nnz), device="cuda")
        vx, vy = fx.Vec.wrap(c, x.data_ptr(), n), fx.Vec.wrap(c, y.data_ptr(), n)
        M.Apply(vx, vy)
        st.synchronize()
        want0 = y.cpu().numpy()
        g = torch.cuda.CUDAGraph()
        g.capture_begin(capture_error_mode="thread_local")
        M.Apply(vx, vy)
        g.capture_end()
        for k in range(4):
            if k == 2:
                M.set_values_dev(v.data_ptr())
                B = P.CSR(n, n, A.row_ptr, A.col_ind, v.cpu().numpy(), A.diag_ptr)
                fx.Csr.from_problem(c, B).Apply(vx, vy)
                st.synchronize()
                want0 = y.cpu().numpy()
            y.zero_()
            g.replay()
            st.synchronize()
            assert np.array_equal(y.cpu().numpy(), want0)
        del g
        c.close()


def test_solver_follows_new_values(ctx):
    """A set-up solver whose matrix loses its row values between two solves."""
    import torch
    from faspxx_amd import fx
    A = P.poisson3d(66)
    M = fx.Csr.from_problem(ctx, A)
    pc = fx.Precond(ctx, "identity")
    s = fx.Solver(ctx, fx.CG)
    s.Setup(M, pc, fx.params(maxIter=2000, relTol=1e-10, absTol=0.0))
    xs = np.random.default_rng(3).uniform(-1, 1, A.nrow)
    x = fx.Vec(ctx, A.nrow)
    assert s.Solve(fx.Vec.from_numpy(ctx, A.matvec(xs)), x).retcode == 0
    scale = np.random.default_rng(4).uniform(1, 2, A.nrow)
    rows = np.repeat(np.arange(A.nrow), np.diff(A.row_ptr.astype(np.int64)))
    v = A.values * np.sqrt(scale[rows] * scale[A.col_ind])  # still SPD
    t = torch.tensor(v, device="cuda")
    torch.cuda.synchronize()
    M.set_values_dev(t.data_ptr())
    B = P.CSR(A.nrow, A.mcol, A.row_ptr, A.col_ind, v, A.diag_ptr)
    x.set(0.0)
    res = s.Solve(fx.Vec.from_numpy(ctx, B.matvec(xs)), x)
    assert res.retcode == 0 and s.last_path == "fused"
    assert np.linalg.norm(x.numpy() - xs) / np.linalg.norm(xs) < 1e-7
