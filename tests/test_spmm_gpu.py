"""GPU parity of fmx_spmm (HIP, through the C ABI) against the oracle.

Bars: integer operands bit-exact; FP64 within 1e-12 relative, FP32 within
1e-5 relative of the oracle's reference-order product (the tolerances the
path is specified with); rows without non-zeros exactly 0.
"""
import gc
import os

import numpy as np
import pytest

import tiny_kat

pytestmark = pytest.mark.gpu

TOL = {np.float32: 1e-5, np.float64: 1e-12}


def to_dev(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def rel_err(y, ref):
    y = np.asarray(y, np.float64)
    ref = np.asarray(ref, np.float64)
    zero = ref == 0
    assert np.all(y[zero] == 0), "rows without non-zeros must be exactly 0"
    d = np.abs(y - ref)[~zero] / np.abs(ref[~zero])
    return float(d.max()) if d.size else 0.0


def check(fmx, orc, img, X, spm=None):
    spm = spm or fmx.SparseMatrix.upload(img.data, img.offs)
    Y = spm.multiply(to_dev(X)).cpu().numpy()
    ref = orc.spmm(img, X)
    if np.issubdtype(X.dtype, np.integer):
        assert np.array_equal(Y, ref)
    else:
        e = rel_err(Y, ref)
        assert e <= TOL[X.dtype.type], e
    return Y, ref


@pytest.fixture(scope="module")
def rmat16(orc):
    # config 1: R-MAT scale 16, edge factor 16, dedup, self edges removed
    src, dst = orc.rmat_edges(16, 16 << 16, seed=2024)
    return src, dst


def test_tiny_kat(fmx, orc):
    img = orc.Image(np.frombuffer(tiny_kat.IMAGE, np.uint8), tiny_kat.OFFS, tiny_kat.N)
    spm = fmx.SparseMatrix.upload(img.data, img.offs)
    assert spm.get_nnz() == 7 and spm.get_num_rows() == 6
    for dt in (np.int32, np.int64, np.float32, np.float64):
        Y = spm.multiply(to_dev(np.array(tiny_kat.X, dt))).cpu().numpy()
        assert np.array_equal(Y, np.array(tiny_kat.Y, dt)), dt
    # download round trip
    data, offs = spm.download()
    assert bytes(data) == tiny_kat.IMAGE and list(offs) == tiny_kat.OFFS


@pytest.mark.parametrize("lh,lw", [(15, 15), (10, 10), (8, 15), (4, 12)])
def test_config1_int32_exact_fp64(fmx, orc, rmat16, lh, lw):
    src, dst = rmat16
    img = orc.build_2d(src, dst, n=1 << 16, log2h=lh, log2w=lw)
    rng = np.random.default_rng(7)
    spm = fmx.SparseMatrix.upload(img.data, img.offs)
    Xi = rng.integers(0, 8, (img.n, 8)).astype(np.int32)
    check(fmx, orc, img, Xi, spm)
    Xd = rng.random((img.n, 8))
    check(fmx, orc, img, Xd, spm)


def test_seq_kat(fmx, orc, rmat16):
    # rand_mat_gen.cpp:178-199: A*[0..n-1] = sum of column ids per row
    src, dst = rmat16
    img = orc.build_2d(src, dst, n=1 << 16, log2h=12, log2w=15)
    spm = fmx.SparseMatrix.upload(img.data, img.offs)
    import torch
    Y = spm.multiply(torch.arange(img.n, dtype=torch.int64, device="cuda")).cpu().numpy()
    r, c = orc.nonzeros(img)
    want = np.bincount(r.astype(np.int64), weights=c.astype(np.float64), minlength=img.n)
    assert np.array_equal(Y, want.astype(np.int64))


def test_exact_fp_pattern(fmx, orc, rmat16):
    # test-2d_multiply.cpp:35-41: X[i][j] = (i%100)*(j+1) -> exact in FP
    src, dst = rmat16
    img = orc.build_2d(src, dst, n=1 << 16, log2h=8, log2w=15)
    spm = fmx.SparseMatrix.upload(img.data, img.offs)
    i = np.arange(img.n)[:, None]
    for k in (4, 16):
        Xi = (i % 100) * (np.arange(k)[None, :] + 1)
        for dt in (np.float32, np.float64):
            Y = spm.multiply(to_dev(Xi.astype(dt))).cpu().numpy()
            assert np.array_equal(Y, orc.spmm(img, Xi.astype(dt)))


@pytest.mark.parametrize("k", [1, 2, 3, 4, 7, 8, 16, 32, 64])
def test_widths(fmx, orc, rmat16, k):
    src, dst = rmat16
    img = orc.build_2d(src, dst, n=1 << 16, log2h=8, log2w=15)
    spm = fmx.SparseMatrix.upload(img.data, img.offs)
    rng = np.random.default_rng(k)
    check(fmx, orc, img, rng.random((img.n, k)).astype(np.float32), spm)
    check(fmx, orc, img, rng.random((img.n, k)), spm)
    check(fmx, orc, img, rng.integers(-9, 9, (img.n, k)).astype(np.int64), spm)
    check(fmx, orc, img, rng.integers(-9, 9, (img.n, k)).astype(np.int32), spm)


def test_strided_operands(fmx, orc, rmat16):
    import torch
    src, dst = rmat16
    img = orc.build_2d(src, dst, n=1 << 16, log2h=8, log2w=15)
    spm = fmx.SparseMatrix.upload(img.data, img.offs)
    rng = np.random.default_rng(5)
    Xfull = rng.random((img.n, 24)).astype(np.float32)
    Xd = torch.from_numpy(Xfull).cuda()[:, 3:19]  # ldx = 24, misaligned start
    Yfull = torch.full((img.n, 40), -1.0, device="cuda")
    Y = Yfull[:, 8:24]
    spm.multiply_async(Xd, Y)
    torch.cuda.synchronize()
    ref = orc.spmm(img, np.ascontiguousarray(Xfull[:, 3:19]))
    assert rel_err(Y.cpu().numpy(), ref) <= 1e-5
    assert torch.all(Yfull[:, :8] == -1) and torch.all(Yfull[:, 24:] == -1)


def test_split_bands_and_determinism(fmx, orc, rmat16):
    src, dst = rmat16
    img = orc.build_2d(src, dst, n=1 << 16, log2h=10, log2w=15)
    rng = np.random.default_rng(9)
    X = rng.random((img.n, 16)).astype(np.float32)
    Xi = rng.integers(0, 8, (img.n, 16)).astype(np.int32)
    os.environ["FMX_ITEM_CAP"] = "300"  # force every band to be split
    try:
        spm = fmx.SparseMatrix.upload(img.data, img.offs)
        Y1, _ = check(fmx, orc, img, X, spm)
        check(fmx, orc, img, Xi, spm)
        # widths drained in 256-word chunks
        check(fmx, orc, img, rng.random((img.n, 32)).astype(np.float32), spm)
        check(fmx, orc, img, rng.random((img.n, 16)), spm)
        check(fmx, orc, img, rng.integers(-9, 9, (img.n, 16)).astype(np.int64), spm)
    finally:
        del os.environ["FMX_ITEM_CAP"]
    spm2 = fmx.SparseMatrix.upload(img.data, img.offs)
    Ya = spm2.multiply(to_dev(X)).cpu().numpy()
    Yb = spm2.multiply(to_dev(X)).cpu().numpy()
    assert np.array_equal(Ya, Yb)  # deterministic call to call
    assert rel_err(Y1, Ya) <= 1e-5


def test_empty_rows_and_ragged(fmx, orc):
    # n not a multiple of H, isolated vertices, empty block rows
    rng = np.random.default_rng(3)
    n = 5000
    src = rng.integers(0, 1200, 20000).astype(np.uint32)
    dst = rng.integers(0, n - 7, 20000).astype(np.uint32)
    img = orc.build_2d(src, dst, n=n, log2h=7, log2w=9)
    spm = fmx.SparseMatrix.upload(img.data, img.offs)
    X = rng.random((n, 5))
    Y, ref = check(fmx, orc, img, X, spm)
    assert np.all(Y[1200:] == 0)


def test_errors(fmx, orc):
    import torch
    img = orc.Image(np.frombuffer(tiny_kat.IMAGE, np.uint8), tiny_kat.OFFS, tiny_kat.N)
    spm = fmx.SparseMatrix.upload(img.data, img.offs)
    with pytest.raises(fmx.FmxError) as e:
        spm.multiply(torch.zeros((5, 2), device="cuda"))
    assert e.value.status == fmx.EDIM
    assert not spm.multiply_into(torch.zeros((6, 2), device="cuda"),
                                 torch.zeros((6, 2), device="cuda", dtype=torch.float64))
    with pytest.raises(fmx.FmxError) as e:
        spm.multiply(torch.zeros((6, 2), device="cuda", dtype=torch.int16))
    assert e.value.status == fmx.ETYPE
    bad = bytearray(tiny_kat.IMAGE)
    bad[4096 + 16 + 2] = 0x05
    with pytest.raises(fmx.FmxError) as e:
        fmx.SparseMatrix.upload(bytes(bad), tiny_kat.OFFS)
    assert e.value.status == fmx.EFORMAT
    with pytest.raises(fmx.FmxError) as e:
        fmx.SparseMatrix.upload(tiny_kat.IMAGE, tiny_kat.OFFS[:-1])
    assert e.value.status == fmx.EFORMAT
    with pytest.raises(fmx.FmxError) as e:
        fmx.SparseMatrix.upload(tiny_kat.BAD_EMPTY_IMAGE, tiny_kat.BAD_EMPTY_OFFS)
    assert e.value.status == fmx.EFORMAT


def test_rmat_generator_matches_oracle(fmx, orc):
    for scale, m, seed, perm in ((16, 1 << 20, 2024, True), (9, 5000, 1, False), (21, 333, 5, True)):
        s, d = fmx.rmat_edges(scale, m, seed, permute=perm)
        so, do = orc.rmat_edges(scale, m, seed, permute=perm)
        assert np.array_equal(s.cpu().numpy().view(np.uint32), so)
        assert np.array_equal(d.cpu().numpy().view(np.uint32), do)


def test_row_32767_header(fmx, orc):
    from test_oracle import last_row_edges
    src, dst = last_row_edges()
    img = orc.build_2d(src, dst, n=40001, log2h=15, log2w=15)
    X = np.arange(40001 * 2, dtype=np.int64).reshape(-1, 2)
    check(fmx, orc, img, X)
    spm = fmx.SparseMatrix.build(to_dev(src.view(np.int32)), to_dev(dst.view(np.int32)), n=40001,
                                 log2_h=15, log2_w=15, flags=fmx.BUILD_DEDUP)
    data, offs = spm.download()
    assert np.array_equal(data, img.data) and np.array_equal(offs, img.offs)


def test_fp32_within_bound_of_either_tile_order(fmx, orc, rmat16):
    """With hilbert_order the reference visits each task's tiles along a
    Hilbert curve (sparse_matrix.cpp:120-186) and its FP32 row sums change
    rounding; the FP64-accumulated GPU result is within 1e-5 of the
    reference's sums in both orders."""
    src, dst = rmat16
    img = orc.build_2d(src, dst, n=1 << 16, log2h=8, log2w=8)
    spm = fmx.SparseMatrix.upload(img.data, img.offs)
    X = np.random.default_rng(21).random((img.n, 16)).astype(np.float32)
    Y = spm.multiply(to_dev(X)).cpu().numpy()
    for hil in (False, True):
        ref = orc.spmm_exec(img, X, 16, hil)
        assert rel_err(Y, ref) <= 1e-5, hil


@pytest.mark.parametrize("lh", [6, 7])
def test_config2_rmat22_spmm_parity(fmx, orc, lh):
    """The scale-22 workload itself: R-MAT scale 22, edge factor 16, dedup,
    in the autotuned 64 x 32768 tiles and in 128 x 32768 tiles, times
    4,194,304 x 16 operands; the FP32 operand is the benchmark's own
    (torch.rand on the device, seed 22).
    - int32: bit-exact.
    - FP32, sequential mode (FMX_SPMM_SEQ): bit-identical to the oracle's
      reference-order FP32 sums.
    - FP32, default mode (FP64 sums rounded once): within 2^-24 relative of
      the exact sums (the FP64 sums of FP32 terms, exact here: multiples of
      2^-24 below 2^29), and elementwise within |ref - exact| + 2^-24 |exact|
      of the reference's FP32 sums, whose own error reaches about 1.3e-5 on
      this operand's hub rows.
    - FP64: within 1e-12 (default) and bit-identical (sequential).
    Rows without non-zeros are exactly 0 in every mode."""
    import torch
    n = 1 << 22
    s, d = fmx.rmat_edges(22, 16 << 22, 22)
    spm = fmx.SparseMatrix.build(s, d, n=n, log2_h=lh, log2_w=15, flags=fmx.BUILD_DEDUP)
    del s, d
    data, offs = spm.download()
    img = orc.Image(data, offs, n)
    rng = np.random.default_rng(22 + lh)
    Xi = rng.integers(0, 8, (n, 16)).astype(np.int32)
    assert np.array_equal(spm.multiply(to_dev(Xi)).cpu().numpy(), orc.spmm(img, Xi, threads=8))
    del Xi
    g = torch.Generator(device="cuda")
    g.manual_seed(22)
    Xt = torch.rand((n, 16), dtype=torch.float32, device="cuda", generator=g)
    Xf = Xt.cpu().numpy()
    ref = orc.spmm(img, Xf, threads=8)
    exact = orc.spmm(img, Xf.astype(np.float64), threads=8)
    Y = spm.multiply(Xt).cpu().numpy()
    assert rel_err(Y, exact) <= 2.0 ** -24
    nz = exact != 0
    bound = np.abs(ref.astype(np.float64) - exact) + 2.0 ** -24 * np.abs(exact)
    assert np.all(np.abs(Y.astype(np.float64) - ref)[nz] <= bound[nz])
    Ys = torch.empty_like(Xt)
    spm.multiply_async(Xt, Ys, seq=True)
    assert np.array_equal(Ys.cpu().numpy(), ref)
    del Xt, Xf, Y, Ys, ref, exact, bound, nz
    Xd = rng.random((n, 16))
    refd = orc.spmm(img, Xd, threads=8)
    Xdt = to_dev(Xd)
    assert rel_err(spm.multiply(Xdt).cpu().numpy(), refd) <= 1e-12
    Yd = torch.empty_like(Xdt)
    spm.multiply_async(Xdt, Yd, seq=True)
    assert np.array_equal(Yd.cpu().numpy(), refd)


@pytest.mark.parametrize("k,pad", [(2, 1), (3, 0), (5, 2), (6, 0), (7, 0), (9, 1), (10, 0), (16, 3), (20, 0), (33, 0),
                                   (63, 0), (65, 0), (129, 0), (257, 0)])
def test_runtime_widths(fmx, orc, k, pad):
    """Widths without a compiled form, and aligned widths with odd strides: the
    runtime-width form (one 16-byte load per lane, the last lane's starting
    early) and, past 64 lanes, the flat one; binary and weighted.  Small whole
    numbers, so every type must be exact; X ends with its last row."""
    import torch
    s, d = orc.rmat_edges(11, 16 << 11, seed=k)
    n = (1 << 11) - 7
    ok = (s < n) & (d < n)
    s, d = s[ok], d[ok]
    rng = np.random.default_rng(k)
    img = orc.build_2d(s, d, n=n, log2h=6, log2w=10)
    a = fmx.SparseMatrix.upload(img.data, img.offs)
    for dt in (np.int32, np.int64, np.float32, np.float64):
        vals = rng.integers(1, 5, s.size).astype(dt)
        wimg = orc.build_2d_w(s, d, vals, n=n, log2h=6, log2w=10)
        w = fmx.SparseMatrix.upload(wimg.data, wimg.offs)
        X = rng.integers(-9, 10, (n, k)).astype(dt)
        buf = torch.zeros(n * (k + pad) - pad, dtype=torch.from_numpy(X).dtype, device="cuda")
        Xt = buf.as_strided((n, k), (k + pad, 1))
        Xt.copy_(torch.from_numpy(X))
        for spm, im in ((a, img), (w, wimg)):
            Y = torch.full((n, k + pad), 77, dtype=Xt.dtype, device="cuda")
            spm.multiply_async(Xt, Y[:, :k])
            assert np.array_equal(Y[:, :k].cpu().numpy(), orc.spmm(im, X)), dt
            assert bool((Y[:, k:] == 77).all())


@pytest.mark.parametrize("k,pad,tall", [(1, 0, True), (2, 1, True), (4, 0, True), (1, 2, False), (4, 4, False),
                                        (5, 1, False), (8, 1, False), (16, 16, False)])
def test_wide_queue_forms(fmx, orc, monkeypatch, k, pad, tall):
    """Bands of 256 rows and more, and the gather order with X's rows further
    apart than the hot block's: the forms whose queue entry holds a 32-bit
    column and a 16-bit row.  Binary and weighted; small whole numbers, so
    every type must be exact."""
    import torch
    if tall:
        monkeypatch.setenv("FMX_WORK_ROWS", "0")
        monkeypatch.setenv("FMX_HOT_MIN_BYTES", str(1 << 40))
    else:
        monkeypatch.setenv("FMX_HOT_MIN_BYTES", "0")
    s, d = orc.rmat_edges(12, 16 << 12, seed=k)
    n = (1 << 12) - 5
    ok = (s < n) & (d < n)
    s, d = s[ok], d[ok]
    rng = np.random.default_rng(k)
    lh = 12 if tall else 6
    img = orc.build_2d(s, d, n=n, log2h=lh, log2w=10)
    a = fmx.SparseMatrix.upload(img.data, img.offs)
    for dt in (np.int32, np.int64, np.float32, np.float64):
        vals = rng.integers(1, 5, s.size).astype(dt)
        wimg = orc.build_2d_w(s, d, vals, n=n, log2h=lh, log2w=10)
        w = fmx.SparseMatrix.upload(wimg.data, wimg.offs)
        X = rng.integers(-9, 10, (n, k)).astype(dt)
        buf = torch.zeros(n * (k + pad) - pad, dtype=torch.from_numpy(X).dtype, device="cuda")
        Xt = buf.as_strided((n, k), (k + pad, 1))
        Xt.copy_(torch.from_numpy(X))
        for spm, im in ((a, img), (w, wimg)):
            Y = torch.full((n, k), 77, dtype=Xt.dtype, device="cuda")
            spm.multiply_async(Xt, Y)
            assert np.array_equal(Y.cpu().numpy(), orc.spmm(im, X)), dt


@pytest.mark.parametrize("hot", ["0", str(1 << 40)])
def test_streams_and_graphs_keep_their_own_scratch(fmx, orc, rmat16, monkeypatch, hot):
    """Calls on six streams at once, and a captured call replayed between
    larger eager ones: the partial bands and the hot block of one never serve
    another.  Integers, so every product must be exact."""
    import torch
    monkeypatch.setenv("FMX_HOT_MIN_BYTES", hot)
    src, dst = rmat16
    img = orc.build_2d(src, dst, n=1 << 16, log2h=15, log2w=15)
    spm = fmx.SparseMatrix.upload(img.data, img.offs)
    rng = np.random.default_rng(3)
    streams = [torch.cuda.Stream() for _ in range(6)]
    X = [rng.integers(-9, 10, (img.n, 4)).astype(np.int32) for _ in streams]
    ref = [orc.spmm(img, x) for x in X]
    Xt = [to_dev(x) for x in X]
    Y = [[torch.empty_like(x) for _ in range(4)] for x in Xt]
    torch.cuda.synchronize()
    for n in (2, 6):  # 2: one buffer each, 6: more streams than buffers
        for r in range(4):
            for i in range(n):
                with torch.cuda.stream(streams[i]):
                    spm.multiply_async(Xt[i], Y[i][r])
        torch.cuda.synchronize()
        for i in range(n):
            for y in Y[i]:
                assert np.array_equal(y.cpu().numpy(), ref[i]), (n, i)
                y.zero_()
        torch.cuda.synchronize()
    Xg, Yg = Xt[0].clone(), torch.empty_like(Xt[0])
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        spm.multiply_async(Xg, Yg)
    wide = rng.integers(-9, 10, (img.n, 16)).astype(np.int32)
    Xw, refw = to_dev(wide), orc.spmm(img, wide)
    Yw = torch.empty_like(Xw)
    torch.cuda.synchronize()
    for i in range(4):
        Xg.copy_(Xt[i])
        torch.cuda.synchronize()
        Yg.zero_()
        torch.cuda.synchronize()
        g.replay()
        with torch.cuda.stream(streams[i]):
            spm.multiply_async(Xw, Yw)
        torch.cuda.synchronize()
        assert np.array_equal(Yg.cpu().numpy(), ref[i]), i
        assert np.array_equal(Yw.cpu().numpy(), refw), i


@pytest.mark.parametrize("n", [1, 127, 128, 129, 1000])
@pytest.mark.parametrize("k", [1, 2, 4, 7, 31, 32, 33, 64, 67])
def test_restaged_operands(fmx, orc, n, k):
    """Column-major and scaled operands at the edges of the restaging tiles
    (128 rows, 32 columns, 16-byte pieces, unaligned bases and strides): a ring
    moves each row of X to its neighbour, and powers of two scale exactly."""
    import torch
    i = np.arange(n, dtype=np.uint32)
    img = orc.build_2d(i, (i + 1) % n, n=n, log2h=6, log2w=10, flags=orc.DEDUP | 2)
    spm = fmx.SparseMatrix.upload(img.data, img.offs)
    assert spm.get_nnz() == n
    rng = np.random.default_rng(n + k)
    pre = 2.0 ** rng.integers(-3, 4, n)
    pd = torch.from_numpy(pre).cuda()
    for dt in (np.int32, np.int64, np.float32, np.float64):
        X = rng.integers(-99, 100, (n, k)).astype(dt)
        td = torch.from_numpy(X).dtype
        ref = np.roll(X, -1, axis=0)
        col = torch.zeros((k, n + 3), dtype=td, device="cuda")[:, 1 : n + 1].t()
        wide = torch.zeros((n, k + 5), dtype=td, device="cuda")[:, 1 : k + 1]
        row = torch.zeros((n, k), dtype=td, device="cuda")
        for x in (col, wide, row):
            x.copy_(torch.from_numpy(X))
            Y = torch.empty((n, k), dtype=td, device="cuda")
            spm.multiply_async(x, Y)
            assert np.array_equal(Y.cpu().numpy(), ref), (dt, x.stride())
            if np.issubdtype(dt, np.floating):
                spm.multiply_scaled_async(x, Y, pre=pd)
                assert np.array_equal(Y.cpu().numpy(), np.roll(X * pre[:, None], -1, axis=0).astype(dt)), (dt, x.stride())


def _two_matrices(fmx, n, k, ctx=None):
    """Two matrices in gather order with split bands, integer operands, and
    the exact products."""
    import torch
    out = []
    for seed in (5, 6):
        src, dst = fmx.rmat_edges((n - 1).bit_length(), 16 * n, seed)
        spm = fmx.SparseMatrix.build(src, dst, n=n, log2_h=6, log2_w=15, ctx=ctx)
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        X = torch.randint(-9, 10, (n, k), device="cuda", generator=g, dtype=torch.int32)
        out.append((spm, X, spm.multiply(X)))
    return out


def test_each_capture_gets_scratch_of_its_own(fmx, monkeypatch):
    """Captured multiplies (nothing is replayed here): each capture allocates
    the scratch it holds -- here the hot block, at least 3 MB -- whether an
    earlier eager call left some or not, and an eager call keeps its own."""
    import torch
    monkeypatch.setenv("FMX_HOT_MIN_BYTES", "0")
    pair = _two_matrices(fmx, 1 << 18, 16)
    least = min(spm.info.hot_columns for spm, _, _ in pair) * 16 * 4
    assert least > 3 << 20
    Y = [torch.empty_like(X) for _, X, _ in pair]
    warm = torch.cuda.Stream()
    graphs = []
    with torch.cuda.stream(warm):
        for (spm, X, _), y in zip(pair, Y):
            spm.multiply_async(X, y)
    torch.cuda.synchronize()
    for i in (0, 1, 0):
        gc.collect()
        torch.cuda.empty_cache()  # as a capture's start does
        free = torch.cuda.mem_get_info()[0]
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=warm):
            pair[i][0].multiply_async(pair[i][1], Y[i])
        graphs.append(g)
        torch.cuda.synchronize()
        assert free - torch.cuda.mem_get_info()[0] >= least, len(graphs)


@pytest.mark.parametrize("hot", ["0", str(1 << 40)])
def test_captured_multiplies_replay_side_by_side(fmx, monkeypatch, hot):
    """Graphs of two matrices and a second one of the first, captured after one
    eager call each and replayed at once on three streams; and both matrices
    in one graph, on two branches.  Integers, so every product must be exact."""
    import torch
    monkeypatch.setenv("FMX_HOT_MIN_BYTES", hot)
    pair = _two_matrices(fmx, 1 << 16, 4)
    pair.append((pair[0][0], pair[0][1].flip(0).contiguous(), None))
    pair[2] = (pair[2][0], pair[2][1], pair[2][0].multiply(pair[2][1]))
    Y = [torch.empty_like(X) for _, X, _ in pair]
    torch.cuda.synchronize()
    graphs = []
    for (spm, X, _), y in zip(pair, Y):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for _ in range(3):
                spm.multiply_async(X, y)
        graphs.append(g)
    streams = [torch.cuda.Stream() for _ in graphs]
    for _ in range(5):
        for y in Y:
            y.zero_()
        torch.cuda.synchronize()
        for _ in range(10):
            for g, s in zip(graphs, streams):
                with torch.cuda.stream(s):
                    g.replay()
        pair[1][0].multiply(pair[1][1])  # an eager call beside them
        torch.cuda.synchronize()
        for i, (y, (_, _, want)) in enumerate(zip(Y, pair)):
            assert torch.equal(y, want), i
    both, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(both):
        main = torch.cuda.current_stream()
        side.wait_stream(main)
        for _ in range(4):
            pair[0][0].multiply_async(pair[0][1], Y[0])
            with torch.cuda.stream(side):
                pair[1][0].multiply_async(pair[1][1], Y[1])
        main.wait_stream(side)
    for _ in range(5):
        Y[0].zero_(), Y[1].zero_()
        torch.cuda.synchronize()
        both.replay()
        torch.cuda.synchronize()
        assert torch.equal(Y[0], pair[0][2]) and torch.equal(Y[1], pair[1][2])


@pytest.mark.parametrize("hot", ["0", str(1 << 40)])
def test_many_streams_in_turn_do_not_wait_for_the_device(fmx, monkeypatch, hot):
    """Eight streams in turn, more than there are scratch buffers: a call
    queues its work and returns while another stream is busy (some 200 ms of
    matrix products), and every product is exact."""
    import torch
    monkeypatch.setenv("FMX_HOT_MIN_BYTES", hot)
    pair = _two_matrices(fmx, 1 << 15, 4)
    streams = [torch.cuda.Stream() for _ in range(8)]
    Y = [torch.empty_like(pair[0][1]) for _ in streams]
    busy, done = torch.cuda.Stream(), torch.cuda.Event()
    M = torch.rand((4096, 4096), device="cuda")
    torch.mm(M, M)

    def turns():
        for i, s in enumerate(streams):
            spm, X, _ = pair[i % 2]
            with torch.cuda.stream(s):
                spm.multiply_async(X, Y[i])

    for _ in range(3):
        turns()
    torch.cuda.synchronize()
    for y in Y:
        y.zero_()
    torch.cuda.synchronize()
    with torch.cuda.stream(busy):
        for _ in range(200):
            torch.mm(M, M)
        done.record()
    turns()
    waited = done.query()
    torch.cuda.synchronize()
    for i, y in enumerate(Y):
        assert torch.equal(y, pair[i % 2][2]), i
    assert not waited


def test_threads_own_streams_have_their_own_scratch(fmx, monkeypatch):
    """hipStreamPerThread is one handle and another stream in each host thread:
    a second thread's first call (nothing runs meanwhile) allocates scratch of
    its own, and calls queued from both threads in turn keep theirs apart."""
    import threading

    import torch
    monkeypatch.setenv("FMX_HOT_MIN_BYTES", "0")
    ctx = fmx.Context()  # (without scratch of earlier calls' streams)
    pair = _two_matrices(fmx, 1 << 18, 16, ctx)
    least = min(spm.info.hot_columns for spm, _, _ in pair) * 16 * 4
    Y = [torch.empty_like(X) for _, X, _ in pair]
    torch.cuda.synchronize()
    free, turn, errors = [], [threading.Semaphore(1), threading.Semaphore(0)], []

    def worker(i):
        spm, X, _ = pair[i]
        for r in range(6):
            turn[i].acquire()
            try:
                if r == 0:
                    before = torch.cuda.mem_get_info()[0]
                for _ in range(1 if r == 0 else 3):
                    st = fmx.lib().fmx_spmm(ctx.handle, spm.handle, fmx.dtype_code(X.dtype), 16, X.data_ptr(), 16,
                                            Y[i].data_ptr(), 16, 2)  # hipStreamPerThread
                    if st:
                        errors.append(st)
                if r == 0:
                    torch.cuda.synchronize()
                    free.append(before - torch.cuda.mem_get_info()[0])
            finally:
                turn[1 - i].release()

    threads = [threading.Thread(target=worker, args=(i,)) for i in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors
    assert all(f >= least for f in free), free
    for y, (_, _, want) in zip(Y, pair):
        assert torch.equal(y, want)


@pytest.mark.parametrize("lh", [5, 6, 15])
@pytest.mark.parametrize("dt", ["int64", "float64"])
def test_few_entries_a_chunk_cost_8_byte_types_no_more(fmx, lh, dt):
    """One column on a sparse graph, whose chunks of 512 words hold far fewer
    entries than a batch has places: 8-byte elements, which are added one by
    one, take at most 1.6 times as long as 4-byte ones (twice the bytes of X
    and Y beside the same image; adding the empty places too took 2 to 3.4
    times as long)."""
    import torch
    n = 1 << 20
    g = torch.Generator(device="cuda")
    g.manual_seed(9)
    src, dst = (torch.randint(0, n, (4 * n,), device="cuda", generator=g, dtype=torch.int32) for _ in range(2))
    spm = fmx.SparseMatrix.build(src, dst, n=n, log2_h=lh)

    def us(dtype):
        X = torch.randint(-9, 10, (n, 1), device="cuda", generator=g).to(dtype)
        Y = torch.empty_like(X)
        best = 1e9
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                spm.multiply_async(X, Y)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) * 50)
        return best

    narrow, wide = us(torch.float32), us(getattr(torch, dt))
    assert wide <= 1.6 * narrow, (wide, narrow)
