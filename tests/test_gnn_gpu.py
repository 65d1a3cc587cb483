"""GPU kernels of the learned warm start against the FP64 oracle
(orc_gnn_loss_grad, itself pinned by finite differences in
test_gnn_oracle.py): forward output, loss and every parameter gradient, in
the FP32 mode against FP64 and the BF16-MFMA mode against the checker with
the same operands rounded to BF16."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def dev(x, dt=None):
    import torch
    t = torch.from_numpy(np.ascontiguousarray(x))
    if dt is not None:
        t = t.to(dt)
    return t.cuda()


def setup_graph(fmx, orc, scale=10, seed=3):
    import torch
    s, d = fmx.rmat_edges(scale, 8 << scale, seed)
    flags = fmx.BUILD_DEDUP | fmx.BUILD_SYMMETRIZE
    spm = fmx.SparseMatrix.build(s, d, n=1 << scale, log2_h=7, log2_w=12, flags=flags)
    img = orc.build_2d(s.cpu().numpy().view(np.uint32), d.cpu().numpy().view(np.uint32), n=1 << scale,
                       log2h=7, log2w=12, flags=orc.DEDUP | orc.SYMMETRIZE)
    r, c = orc.nonzeros(img)
    order = np.lexsort((c, r))
    r, c = r[order].astype(np.int64), c[order].astype(np.int64)
    n = img.n
    rowptr = np.zeros(n + 1, np.int64)
    np.add.at(rowptr, r + 1, 1)
    rowptr = np.cumsum(rowptr)
    return spm, img, rowptr, c


# mode 1: FP32 products against the FP64 checker.  mode 0: BF16 matrix-core
# products against the checker with the same operands rounded to BF16 (what
# remains is FP32 accumulation and the odd operand that rounds the other way).
@pytest.mark.parametrize("mode,tol", [(1, 2e-4), (0, 1e-2)])
def test_forward_backward_vs_oracle(fmx, orc, mode, tol):
    import torch
    spm, img, rowptr, col = setup_graph(fmx, orc)
    n = img.n
    X0 = torch.empty((n, 16), dtype=torch.float32, device="cuda")
    dinv = torch.empty(n, dtype=torch.float64, device="cuda")
    L = fmx.lib()
    L.fmx_gnn_features(fmx.default_context().handle, spm.handle, 7, X0.data_ptr(), dinv.data_ptr(), None)
    torch.cuda.synchronize()
    deg = np.diff(rowptr)
    assert np.allclose(X0[:, 0].cpu().numpy(), np.log1p(deg), rtol=1e-6)
    assert np.allclose(dinv.cpu().numpy(), np.where(deg > 0, 1 / np.sqrt(np.maximum(deg, 1)), 0))
    rng = np.random.default_rng(0)
    npar = L.fmx_gnn_param_count()
    assert npar == orc.gnn_param_count()
    P = (rng.standard_normal(npar) * 0.15).astype(np.float32)
    U, _ = np.linalg.qr(rng.standard_normal((n, 16)))
    acts = torch.empty(L.fmx_gnn_acts_floats(n), dtype=torch.float32, device="cuda")
    work = torch.empty(L.fmx_gnn_work_floats(n), dtype=torch.float32, device="cuda")
    Y = torch.empty((n, 16), dtype=torch.float32, device="cuda")
    Pd = dev(P)
    ctx = fmx.default_context()
    ctx.check(L.fmx_gnn_forward(ctx.handle, spm.handle, dinv.data_ptr(), Pd.data_ptr(), X0.data_ptr(),
                                acts.data_ptr(), Y.data_ptr(), work.data_ptr(), mode, None), "forward")
    Ud = dev(U.astype(np.float32))
    dY = torch.empty_like(Y)
    import ctypes
    loss = ctypes.c_double()
    ctx.check(L.fmx_subspace_loss(ctx.handle, n, 16, Y.data_ptr(), Ud.data_ptr(), ctypes.byref(loss),
                                  dY.data_ptr(), None), "loss")
    G = torch.zeros(npar, dtype=torch.float32, device="cuda")
    ctx.check(L.fmx_gnn_backward(ctx.handle, spm.handle, dinv.data_ptr(), Pd.data_ptr(), X0.data_ptr(),
                                 acts.data_ptr(), dY.data_ptr(), G.data_ptr(), work.data_ptr(), mode,
                                 None), "backward")
    torch.cuda.synchronize()
    ref_loss, ref_g, ref_Y = orc.gnn_loss_grad(rowptr, col, dinv.cpu().numpy(),
                                               X0.cpu().numpy().astype(np.float64),
                                               U.astype(np.float32).astype(np.float64),
                                               P.astype(np.float64), bf16=(mode == 0))
    Yg = Y.cpu().numpy()
    assert np.abs(Yg - ref_Y).max() <= tol * np.abs(ref_Y).max()
    assert abs(loss.value - ref_loss) <= tol * max(1.0, abs(ref_loss))
    g = G.cpu().numpy()
    # per parameter block, relative to the block's largest gradient
    offs = [0]
    for l in range(3):
        din = 16 if l == 0 else 64
        offs += [offs[-1] + din * 64, offs[-1] + 2 * din * 64, offs[-1] + 2 * din * 64 + 64]
    offs.append(npar)
    for a, b in zip(offs[:-1], offs[1:]):
        scale = np.abs(ref_g[a:b]).max()
        assert np.abs(g[a:b] - ref_g[a:b]).max() <= tol * scale + 1e-12, (a, b)


def test_adam_step(fmx):
    import torch
    import ctypes
    L = fmx.lib()
    ctx = fmx.default_context()
    rng = np.random.default_rng(1)
    p = rng.standard_normal(1000).astype(np.float32)
    g = rng.standard_normal(1000).astype(np.float32)
    m = np.zeros(1000, np.float32)
    v = np.zeros(1000, np.float32)
    pd, gd, md, vd = dev(p), dev(g), dev(m), dev(v)
    for step in (1, 2):
        ctx.check(L.fmx_adam(ctx.handle, 1000, pd.data_ptr(), gd.data_ptr(), md.data_ptr(), vd.data_ptr(),
                             1e-2, 0.9, 0.999, 1e-8, step, None), "adam")
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - 1e-2 * (m / (1 - 0.9 ** step)) / (np.sqrt(v / (1 - 0.999 ** step)) + 1e-8)
    torch.cuda.synchronize()
    assert np.allclose(pd.cpu().numpy(), p, rtol=1e-5, atol=1e-6)


def test_dcsbm_generator_matches_oracle(fmx, orc):
    for n, seed in ((1 << 12, 5), (1 << 16, 11)):
        s, d = fmx.dcsbm_edges(n, seed)
        bstart, wtab = fmx.dcsbm_params(n)
        so, do = orc.dcsbm_edges(n, bstart, wtab, 20, n * 8, seed)
        assert np.array_equal(s.cpu().numpy().view(np.uint32), so)
        assert np.array_equal(d.cpu().numpy().view(np.uint32), do)


@pytest.mark.parametrize("n", [1, 17, 200, 1031, 33000])
def test_mfma_products_ragged_rows(fmx, n):
    """The BF16 products and gradients at row counts around their tiles (16
    rows a wave, 32 a gradient step, 128 a block step), against the same
    network in FP64 with the operands of every product rounded to BF16.
    dY is given, so nothing depends on the loss.  What remains is FP32
    accumulation and the odd operand that rounds the other way: 1e-2 of each
    block's largest value, as above."""
    import torch
    g = torch.Generator().manual_seed(n)
    e = torch.randint(0, n, (2, 5 * n), generator=g).int()
    spm = fmx.SparseMatrix.build(e[0].contiguous().cuda(), e[1].contiguous().cuda(), n=n, log2_h=7, log2_w=12,
                                 flags=fmx.BUILD_DEDUP | fmx.BUILD_SYMMETRIZE)
    r, c = torch.cat([e[0], e[1]]).long(), torch.cat([e[1], e[0]]).long()
    key = torch.unique((r * n + c)[r != c])
    r, c = key // n, key % n
    deg = torch.bincount(r, minlength=n).double()
    dinv = torch.where(deg > 0, deg.clamp(min=1).rsqrt(), torch.zeros_like(deg))
    f32 = lambda x: x.float().double()
    bf = lambda x: x.float().bfloat16().double()
    spread = lambda x: torch.zeros_like(x).index_add_(0, r, x[c])
    agg = lambda x: f32(f32(spread(f32(x * dinv[:, None]))) * dinv[:, None])
    L, ctx = fmx.lib(), fmx.default_context()
    P = (torch.randn(L.fmx_gnn_param_count(), generator=g) * 0.15)
    X0, dY = torch.randn((n, 16), generator=g), torch.randn((n, 16), generator=g)
    at, W = 0, []
    for d in (16, 64, 64):
        W.append((P[at:at + 64 * d].view(d, 64).double(), P[at + 64 * d:at + 128 * d].view(d, 64).double(),
                  P[at + 128 * d:at + 128 * d + 64].double()))
        at += 128 * d + 64
    Wo = P[at:].view(64, 16).double()
    Hs, Ag = [X0.double()], []
    for Ws, Wn, b in W:
        Ag.append(agg(Hs[-1]))
        Hs.append(f32(torch.relu(bf(Hs[-1]) @ bf(Ws) + bf(Ag[-1]) @ bf(Wn) + b)))
    want_Y = bf(Hs[3]) @ bf(Wo)
    grads = [bf(Hs[3]).t() @ bf(dY)]
    dZ = f32(bf(dY) @ bf(Wo).t()) * (Hs[3] > 0)
    for l in (2, 1, 0):
        Ws, Wn, _ = W[l]
        grads[:0] = [bf(Hs[l]).t() @ bf(dZ), bf(Ag[l]).t() @ bf(dZ), dZ.sum(0)]
        if l:
            dZ = f32(bf(dZ) @ bf(Ws).t() + agg(f32(bf(dZ) @ bf(Wn).t()))) * (Hs[l] > 0)
    acts = torch.empty(L.fmx_gnn_acts_floats(n), device="cuda")
    work = torch.empty(L.fmx_gnn_work_floats(n), device="cuda")
    Y, G = torch.empty((n, 16), device="cuda"), torch.full((P.numel(),), 7.0, device="cuda")
    X0d, dYd, Pd, dv = X0.cuda(), dY.cuda(), P.cuda(), dinv.cuda()
    ctx.check(L.fmx_gnn_forward(ctx.handle, spm.handle, dv.data_ptr(), Pd.data_ptr(), X0d.data_ptr(),
                                acts.data_ptr(), Y.data_ptr(), work.data_ptr(), 0, None), "forward")
    ctx.check(L.fmx_gnn_backward(ctx.handle, spm.handle, dv.data_ptr(), Pd.data_ptr(), X0d.data_ptr(),
                                 acts.data_ptr(), dYd.data_ptr(), G.data_ptr(), work.data_ptr(), 0, None), "backward")
    torch.cuda.synchronize()
    assert (Y.cpu().double() - want_Y).abs().max() <= 1e-2 * want_Y.abs().max()
    got = G.cpu().double()
    at = 0
    for w in grads:
        part = got[at:at + w.numel()].view(w.shape)
        assert (part - w).abs().max() <= 1e-2 * w.abs().max() + 1e-12, (at, w.shape)
        at += w.numel()
    assert at == got.numel()
