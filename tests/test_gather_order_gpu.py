"""GPU parity of the gather-order image (flashx_amd/csrc/hotcols.cpp,
image_dev.hip): the
default-mode SpMM of a matrix whose X is large runs on a copy of the matrix
with its most used columns relabelled into a dense front block of X that is
restaged every call.  FMX_HOT_MIN_BYTES=0 makes small matrices take that
path too.  Bars as for the plain path: integers bit-exact; FP32 within one
rounding of the exact (FP64) sums; FP64 within 1e-12; rows without
non-zeros exactly 0; streamed equal to resident; the sequential mode
unchanged (it never uses the relabelled image)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def dev(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def rel(y, ref):
    y = np.asarray(y, np.float64)
    ref = np.asarray(ref, np.float64)
    z = ref == 0
    assert np.all(y[z] == 0)
    return float((np.abs(y - ref)[~z] / np.abs(ref[~z])).max())


@pytest.fixture
def forced(monkeypatch):
    monkeypatch.setenv("FMX_HOT_MIN_BYTES", "0")


@pytest.fixture(scope="module")
def rmat16(orc):
    return orc.rmat_edges(16, 16 << 16, seed=2024)


@pytest.mark.parametrize("lh,lw,cap", [(6, 15, None), (15, 15, None), (8, 12, "300"), (4, 10, None)])
def test_gather_order_matches_oracle(fmx, orc, rmat16, forced, monkeypatch, lh, lw, cap):
    if cap:
        monkeypatch.setenv("FMX_ITEM_CAP", cap)
    src, dst = rmat16
    img = orc.build_2d(src, dst, n=1 << 16, log2h=lh, log2w=lw)
    spm = fmx.SparseMatrix.upload(img.data, img.offs)
    rng = np.random.default_rng(lh + 10 * lw)
    for k in (1, 4, 8, 16):
        Xi = rng.integers(-9, 10, (img.n, k)).astype(np.int32)
        assert np.array_equal(spm.multiply(dev(Xi)).cpu().numpy(), orc.spmm(img, Xi)), k
        Xf = rng.random((img.n, k)).astype(np.float32)
        assert rel(spm.multiply(dev(Xf)).cpu().numpy(), orc.spmm(img, Xf.astype(np.float64))) <= 2.0 ** -24
        Xd = rng.random((img.n, 3))  # 24-byte rows: the runtime-width path
        assert rel(spm.multiply(dev(Xd)).cpu().numpy(), orc.spmm(img, Xd)) <= 1e-12
        # the sequential mode keeps the reference's column order
        import torch
        Y = torch.empty((img.n, k), dtype=torch.float32, device="cuda")
        spm.multiply_async(dev(Xf), Y, seq=True)
        assert np.array_equal(Y.cpu().numpy(), orc.spmm(img, Xf))


def test_gather_order_weighted_streamed_layouts(fmx, orc, rmat16, forced):
    """Weighted values follow their entries; a streamed matrix streams its own
    gather-order image and gives the resident bits; column-major operands and
    row scales go through the same path."""
    import torch
    src, dst = rmat16
    vals = (np.random.default_rng(4).random(src.size) + 0.5).astype(np.float32)
    img = orc.build_2d_w(src, dst, vals, n=1 << 16, log2h=7, log2w=15)
    res = fmx.SparseMatrix.upload(img.data, img.offs)
    st = fmx.SparseMatrix.upload_streamed(img.data, img.offs, chunk_bytes=1 << 16)
    # the resident image is relabelled on the device, the streamed one from
    # its host copy: the same hot columns
    assert res.info.hot_columns == st.info.hot_columns > 0
    X = np.random.default_rng(5).random((img.n, 8)).astype(np.float32)
    Yr = res.multiply(dev(X)).cpu().numpy()
    assert rel(Yr, orc.spmm(img, X.astype(np.float64))) <= 2.0 ** -24 + 1e-15
    assert np.array_equal(st.multiply(dev(X)).cpu().numpy(), Yr)
    Xt = dev(X)
    Yc = torch.empty((8, img.n), dtype=torch.float32, device="cuda").t()
    res.multiply_async(Xt.t().contiguous().t(), Yc)
    assert np.array_equal(Yc.cpu().numpy(), Yr)
    post = torch.rand(img.n, dtype=torch.float64, device="cuda") + 0.5
    Ys = torch.empty_like(Xt)
    res.multiply_scaled_async(Xt, Ys, post=post)
    want = orc.spmm(img, X.astype(np.float64)) * post.cpu().numpy()[:, None]
    assert rel(Ys.cpu().numpy(), want) <= 2.0 ** -24 + 1e-15


@pytest.mark.parametrize("n,k,col", [(65536, 8, True), (65536, 16, False), (50001, 3, True)])
def test_gather_order_restages_x_rows_only(fmx, orc, rmat16, forced, n, k, col):
    """A column-major or pre-scaled X is restaged with as many rows as X has;
    the image's extra (hot) columns have no rows of their own in X or in the
    scales, which end with their allocations here."""
    import torch
    src, dst = (v[(rmat16[0] < n) & (rmat16[1] < n)] for v in rmat16)
    img = orc.build_2d(src, dst, n=n, log2h=6, log2w=15)
    spm = fmx.SparseMatrix.upload(img.data, img.offs)
    assert spm.info.hot_columns > 0
    rng = np.random.default_rng(n + k)
    X = rng.random((n, k)).astype(np.float32)
    pre, post = rng.random(n) + 0.5, rng.random(n) + 0.5
    Xt = dev(X.T).t() if col else dev(X)
    Y = torch.empty((n, k), dtype=torch.float32, device="cuda")
    spm.multiply_scaled_async(Xt, Y, pre=dev(pre), post=dev(post))
    staged = (X.astype(np.float64) * pre[:, None]).astype(np.float32).astype(np.float64)
    want = orc.spmm(img, staged) * post[:, None]
    assert rel(Y.cpu().numpy(), want) <= 2.0 ** -24 + 1e-15


@pytest.mark.parametrize("graph,n,weighted,k,hot", [
    ("even", 1 << 21, False, 16, False), ("even", 1 << 20, True, 16, False), ("even", 1 << 19, False, 4, False),
    ("even", 1 << 20, False, 4, False), ("even", 1 << 20, False, 1, True), ("ring", 1 << 20, False, 10, False),
    ("rmat", 1 << 21, False, 16, True), ("rmat", 1 << 20, True, 16, True), ("rmat", 1 << 18, True, 16, False),
    ("rmat", 1 << 21, True, 4, True)])
def test_gather_order_where_columns_are_skewed(fmx, monkeypatch, graph, n, weighted, k, hot):
    """Which image a multiply runs on, told by the hot block that the first
    call of a context allocates: the gather order where a small share of the
    columns is hot, the plain image where columns are picked evenly or there
    are too few for the width; and the products are right on either."""
    import torch
    monkeypatch.delenv("FMX_HOT_MIN_BYTES", raising=False)
    ctx = fmx.Context()
    g = torch.Generator(device="cuda")
    g.manual_seed(n + k)
    if graph == "ring":
        src = torch.arange(n, device="cuda", dtype=torch.int32).repeat(4)
        dst = torch.cat([(src[:n] + j) % n for j in (1, 2, 3, 4)])
    elif graph == "even":
        src, dst = (torch.randint(0, n, (4 * n,), device="cuda", generator=g, dtype=torch.int32) for _ in range(2))
    else:
        src, dst = fmx.rmat_edges((n - 1).bit_length(), 4 * n, 7)
    if weighted:
        vals = torch.ones(src.numel(), device="cuda")
        spm = fmx.SparseMatrix.build_weighted(src, dst, vals, n=n, log2_h=15, ctx=ctx)
    else:
        spm = fmx.SparseMatrix.build(src, dst, n=n, log2_h=15, ctx=ctx)
    block = spm.info.hot_columns * k * 4
    assert block > 3 << 20
    X = torch.randint(-9, 10, (n, k), device="cuda", generator=g).float()
    Y = torch.empty_like(X)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    spm.multiply_async(X, Y)
    torch.cuda.synchronize()
    taken = free - torch.cuda.mem_get_info()[0]
    assert taken >= block if hot else taken < block, (taken, block)
    monkeypatch.setenv("FMX_HOT_MIN_BYTES", "0" if not hot else str(1 << 60))
    Z = torch.empty_like(X)
    spm.multiply_async(X, Z)
    assert torch.equal(Y, Z)


@pytest.mark.parametrize("dt", ["int64", "float64"])
def test_one_column_below_its_alignment(fmx, orc, rmat16, forced, dt):
    """One column of 8-byte elements that starts between two of them: the
    one-column form takes it as it takes an aligned one."""
    import torch
    src, dst = rmat16
    img = orc.build_2d(src, dst, n=1 << 16, log2h=6, log2w=15)
    spm = fmx.SparseMatrix.upload(img.data, img.offs)
    X = np.random.default_rng(4).integers(-9, 10, (img.n, 1)).astype(dt)
    raw = torch.zeros(8 * img.n + 4, dtype=torch.uint8, device="cuda")
    raw[4:].copy_(torch.from_numpy(X.view(np.uint8).reshape(-1)))
    Y = torch.empty((img.n, 1), dtype=getattr(torch, dt), device="cuda")
    ctx = spm.ctx
    ctx.check(fmx.lib().fmx_spmm(ctx.handle, spm.handle, fmx.dtype_code(Y.dtype), 1, raw.data_ptr() + 4, 1,
                                 Y.data_ptr(), 1, ctx.stream_ptr()), "fmx_spmm")
    assert np.array_equal(Y.cpu().numpy(), orc.spmm(img, X))


def test_gather_order_from_more_columns_of_8_byte_elements(fmx, monkeypatch):
    """FP64 rows of two and more elements take the gather order from 1,050,000
    columns, one element from 500,000 (told as above)."""
    import torch
    monkeypatch.delenv("FMX_HOT_MIN_BYTES", raising=False)
    for n, k, hot in ((1 << 20, 4, False), (1 << 21, 4, True), (1 << 21, 1, True), (1 << 20, 7, False)):
        ctx = fmx.Context()
        src, dst = fmx.rmat_edges((n - 1).bit_length(), 4 * n, 7)
        spm = fmx.SparseMatrix.build(src, dst, n=n, log2_h=15, ctx=ctx)
        block = spm.info.hot_columns * k * 8
        X = torch.ones((n, k), device="cuda", dtype=torch.float64)
        Y = torch.empty_like(X)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        spm.multiply_async(X, Y)
        torch.cuda.synchronize()
        taken = free - torch.cuda.mem_get_info()[0]
        assert taken >= block > 2 << 20 if hot else taken < block, (n, k, taken, block)
