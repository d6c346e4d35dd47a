"""Row values on both sides of the sizes from which the SpMV kernels take them
(f64 409600 rows, f32 720896): the bits of the entry-by-entry form, before and
after the values change, and in a product captured before they do."""
import numpy as np
import pytest

from faspxx_amd import problems as P
from test_gpu_rowvalues import box2d, diag, make, products

pytestmark = pytest.mark.gpu

# the last sizes that stream and the first that do not, ragged last workgroups,
# rows of one entry, of up to 8 and of up to 9
SYSTEMS = {
    "diag_409600": lambda: diag(409600), "diag_409601": lambda: diag(409601),
    "diag_720896": lambda: diag(720896), "diag_720897": lambda: diag(720897),
    "poisson2d_641": lambda: P.poisson2d(641), "poisson3d_90": lambda: P.poisson3d(90),
    "box_641x640": lambda: box2d(641, 640), "box_3x240301": lambda: box2d(3, 240301),
}


@pytest.mark.parametrize("name", list(SYSTEMS))
def test_same_bits(ctx, monkeypatch, name):
    A = SYSTEMS[name]()
    M, M0 = make(ctx, A, monkeypatch, False), make(ctx, A, monkeypatch, True)
    for _ in range(2):
        for a, b in zip(products(ctx, M, A.nrow), products(ctx, M0, A.nrow)):
            assert np.array_equal(a, b)
        M.shift_diag(0.25)
        M0.shift_diag(0.25)


@pytest.mark.parametrize("name", ["poisson3d_90", "box_641x640"])
def test_captured_product_follows_new_values(name):
    import torch
    from faspxx_amd import fx
    A = SYSTEMS[name]()
    n = A.nrow
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        c = fx.Context(0, stream=st.cuda_stream)
        M = fx.Csr.from_problem(c, A)
        x = torch.tensor(np.random.default_rng(1).uniform(-1, 1, n), device="cuda")
        y = torch.zeros_like(x)
        v = torch.tensor(np.random.default_rng(2).uniform(1, 2, A.nnz), device="cuda")
        vx, vy = fx.Vec.wrap(c, x.data_ptr(), n), fx.Vec.wrap(c, y.data_ptr(), n)
        g = torch.cuda.CUDAGraph()
        g.capture_begin(capture_error_mode="thread_local")
        M.Apply(vx, vy)
        g.capture_end()
        for k in range(4):
            if k == 2:
                M.set_values_dev(v.data_ptr())
            B = P.CSR(n, n, A.row_ptr, A.col_ind, A.values if k < 2 else v.cpu().numpy(),
                      A.diag_ptr)
            fx.Csr.from_problem(c, B).Apply(vx, vy)
            st.synchronize()
            want = y.cpu().numpy()
            y.zero_()
            g.replay()
            st.synchronize()
            assert np.array_equal(y.cpu().numpy(), want)
        del g
        c.close()


def test_pointer_asked_for_during_a_capture():
    """The values' pointer handed out while the context's stream is captured:
    a product captured before it reads what is then written through it, though
    the second graph never runs."""
    import torch
    from faspxx_amd import fx
    A = SYSTEMS["poisson3d_90"]()
    n = A.nrow
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        c = fx.Context(0, stream=st.cuda_stream)
        M = fx.Csr.from_problem(c, A)
        x = torch.tensor(np.random.default_rng(1).uniform(-1, 1, n), device="cuda")
        y, z = torch.zeros_like(x), torch.zeros_like(x)
        v = np.random.default_rng(2).uniform(1, 2, A.nnz)
        vx, vy = fx.Vec.wrap(c, x.data_ptr(), n), fx.Vec.wrap(c, y.data_ptr(), n)
        fx.Csr.from_problem(c, P.CSR(n, n, A.row_ptr, A.col_ind, v, A.diag_ptr)).Apply(vx, vy)
        st.synchronize()
        want = y.cpu().numpy()
        g0, g1 = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
        g0.capture_begin(capture_error_mode="thread_local")
        M.Apply(vx, vy)
        g0.capture_end()
        g1.capture_begin(capture_error_mode="thread_local")
        z.fill_(1.0)
        ptr = M.values_ptr
        g1.capture_end()
        fx.Vec.wrap(c, ptr, A.nnz).upload(v)
        for _ in range(3):
            y.zero_()
            g0.replay()
            st.synchronize()
            assert np.array_equal(y.cpu().numpy(), want)
        del g0, g1
        c.close()
