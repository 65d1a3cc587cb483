"""The work that a user of this framework has it do, as cases that can be timed.

Every case goes through the public entry points of flashx_amd.fmx and
flashx_amd.learned (and, where those have no wrapper, the C functions that
learned.py calls).  Graphs are R-MAT (a, b, c, d) = (.57, .19, .19, .05) or a
degree-corrected block model, relabelled at random; all inputs come from the
seed alone.

listed() names the cases, draw() gives more of the same ranges, prepare()
makes what a program has in hand before the call, run() is one pass, work()
what a pass cannot do without, and exact() the same result in 64 bits from
plain torch.
"""
import ctypes
import math

import torch

import flashx_amd.fmx as F
from flashx_amd import learned

DEV = "cuda:0"
DTYPES = {"i32": torch.int32, "i64": torch.int64, "f32": torch.float32, "f64": torch.float64}
SIZE = {"i32": 4, "i64": 8, "f32": 4, "f64": 8}
NEV = 16  # columns of the warm-start network's output


def listed():
    return [
        # The benchmark: R-MAT scale 22, edge factor 16, X of 16 FP32 columns,
        # the tile shape that the autotuner picks for it.
        _spmm("spmm_f32_k16_4m", n=1 << 22, degree=16, k=16, dtype="f32", tile=5),
        # An ordinary small product: scale 16 in the default tiles, FP64.
        _spmm("spmm_f64_k8_65k", n=1 << 16, degree=16, k=8, dtype="f64", tile=15),
        # The smallest calls: one integer column on a graph of 4,096 vertices
        # (degrees, neighbour counts), where latency is all.
        _spmm("spmv_i32_4k", n=1 << 12, degree=16, k=1, dtype="i32", tile=15),
        # Weighted edges (ratings, similarities): FP32 values, 16 columns.
        _spmm("spmm_weighted_f32_k16_1m", n=1 << 20, degree=16, k=16, dtype="f32", tile=15, weighted=True),
        # A ragged graph and a width that is no power of two, operands
        # column-major as the reference's eigensolver keeps them.
        _spmm("spmm_f32_k10_col_700k", n=700001, degree=12, k=10, dtype="f32", tile=15, col=True),
        # The eigensolver's operator D^-1/2 A D^-1/2 on one Krylov block.
        _spmm("spmm_scaled_f32_k16_260k", n=1 << 18, degree=16, k=16, dtype="f32", tile=6, scaled=True, sym=True),
        # A block of a scale-22 Krylov basis against a new block: V^T W ...
        {"name": "gram_f32_96x16_4m", "kind": "gram", "n": 1 << 22, "ka": 96, "kb": 16, "dtype": "f32"},
        # ... and W - V C.
        {"name": "gemm_f32_96x16_4m", "kind": "gemm", "n": 1 << 22, "ka": 96, "kc": 16, "dtype": "f32", "beta": 1.0},
        # PageRank of a directed graph: ten sweeps through its transpose.
        {"name": "pagerank_1m", "kind": "pagerank", "n": 1 << 20, "degree": 16, "iters": 10},
        # Non-negative factors of rank 20 of a directed graph.
        {"name": "nmf_k20_260k", "kind": "nmf", "n": 260000, "degree": 16, "k": 20, "iters": 4},
        # From an edge list to the tiled matrix, and one product with it.
        {"name": "build_1m", "kind": "build", "n": 1 << 20, "degree": 16, "sym": False, "tile": 5},
        # One training step of the warm-start network: the prediction, the
        # subspace loss and the parameters' gradients.
        {"name": "gnn_step_131k", "kind": "gnn", "n": 1 << 17, "degree": 16, "train": True},
    ]


def _spmm(name, n, degree, k, dtype, tile, weighted=False, scaled=False, sym=False, col=False, seq=False):
    c = {"kind": "spmm", "n": n, "degree": degree, "k": k, "dtype": dtype, "tile": tile, "weighted": weighted,
         "scaled": scaled, "sym": sym, "col": col, "seq": seq}
    return dict(c, name=name) if name else c


def draw(rng):
    """One more case: sizes log-uniform over the listed ones' range, half of
    them not powers of two, and no dearer than the largest listed."""

    def size(lo, hi):
        e = rng.uniform(math.log2(lo), math.log2(hi))
        return int(round(2.0 ** e)) | 1 if rng.random() < 0.5 else 1 << int(round(e))

    kind = rng.choice(["spmm"] * 6 + ["gram", "gemm", "pagerank", "nmf", "build", "gnn"])
    if kind == "spmm":
        dtype = rng.choice(["f32", "f32", "f64", "i32", "i64"])
        real = dtype[0] == "f"
        k = rng.choice([1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 16, 20, 24, 32, 40, 64])
        degree = rng.choice([4, 8, 16, 24])
        n = size(1 << 11, 1 << 21)
        while n * degree * k * SIZE[dtype] > (1 << 30):
            n //= 2
        form = rng.random()
        scaled, col = real and 0.2 <= form < 0.4, 0.4 <= form < 0.55
        while (scaled or col) and n * k * SIZE[dtype] > (32 << 20):  # operands of at most 32 MB
            n //= 2
        return _spmm(None, n, degree, k, dtype, rng.choice([5, 6, 7, 15]), weighted=form < 0.2, scaled=scaled,
                     sym=rng.random() < 0.3, col=col, seq=real and 0.55 <= form < 0.65)
    if kind == "gram":
        dtype = rng.choice(["f32", "f64"])
        ka = rng.choice([4, 8, 10, 16, 24, 32, 48, 64, 80, 96, 112, 128])
        kb = rng.choice([ka, 8, 10, 16, 32])
        return {"kind": kind, "n": size(1 << 13, 1 << (22 if dtype == "f32" and ka + kb <= 112 else 20)), "ka": ka,
                "kb": kb, "dtype": dtype}
    if kind == "gemm":
        dtype = rng.choice(["f32", "f64"])
        ka = rng.choice([4, 8, 10, 16, 24, 32, 48, 64, 80, 96, 128])
        kc = rng.choice([4, 8, 10, 16, 20, 32, 48, 64])
        return {"kind": kind, "n": size(1 << 13, 1 << (22 if dtype == "f32" and ka + 2 * kc <= 128 else 20)),
                "ka": ka, "kc": kc, "dtype": dtype, "beta": rng.choice([0.0, 1.0])}
    if kind == "pagerank":
        return {"kind": kind, "n": size(1 << 14, 1 << 20), "degree": rng.choice([4, 8, 16]),
                "iters": rng.randint(4, 10)}
    if kind == "nmf":
        return {"kind": kind, "n": size(1 << 13, 1 << 18), "degree": rng.choice([8, 16]),
                "k": rng.choice([4, 8, 10, 16, 20]), "iters": rng.randint(1, 4)}
    if kind == "build":
        sym = rng.random() < 0.4
        return {"kind": kind, "n": size(1 << 13, 1 << (19 if sym else 20)), "degree": rng.choice([8, 16]),
                "sym": sym, "tile": rng.choice([5, 7, 15])}
    train = rng.random() < 0.6
    return {"kind": "gnn", "n": size(1 << 13, 1 << (17 if train else 18)), "degree": rng.choice([8, 16]),
            "train": train}


# ---- inputs ------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _rmat(n, degree, g):
    """n * degree R-MAT edges over n vertices, relabelled at random."""
    m, levels = n * degree, max(1, (n - 1).bit_length())
    src = torch.zeros(m, dtype=torch.int64, device=DEV)
    dst = torch.zeros(m, dtype=torch.int64, device=DEV)
    for _ in range(levels):
        u = torch.rand(m, device=DEV, generator=g)
        src.mul_(2).add_(u >= 0.76)
        dst.mul_(2).add_(((u >= 0.57) & (u < 0.76)) | (u >= 0.95))
    label = torch.randperm(n, device=DEV, generator=g)
    return [label[(v * n) >> levels].to(torch.int32) for v in (src, dst)]


def _blocks(n, degree, g):
    """n * degree / 2 edges of a degree-corrected block model: 32 contiguous
    blocks, 20 : 1 in favour of the own block, power-law degrees."""
    m = n * degree // 2
    theta = (1.0 - torch.rand(n, device=DEV, generator=g, dtype=torch.float64)).pow(-1.0 / 1.5)
    weight = theta.clamp(max=math.sqrt(n)).mul(1024.0).to(torch.int64)
    upto = weight.cumsum(0)
    bound = torch.tensor([n * b // 32 for b in range(33)], device=DEV)
    mass = torch.cat([torch.zeros(1, dtype=torch.int64, device=DEV), upto])
    total = int(upto[-1])

    def pick(lo, width):
        at = lo + (torch.rand(m, device=DEV, generator=g, dtype=torch.float64) * width).to(torch.int64)
        return torch.searchsorted(upto, at, right=True).clamp(max=n - 1)

    src = pick(0, total)
    block = torch.searchsorted(bound, src, right=True) - 1
    lo, hi = mass[bound[block]], mass[bound[block + 1]]
    own = torch.rand(m, device=DEV, generator=g) < 20.0 / 21.0
    dst = pick(torch.where(own, lo, torch.zeros_like(lo)), torch.where(own, hi - lo, torch.full_like(lo, total)))
    return src.to(torch.int32), dst.to(torch.int32), bound


def _dense(rows, k, dtype, g, col=False):
    """A dense operand: U[0, 1), or small whole numbers."""
    shape = (k, rows) if col else (rows, k)
    if dtype[0] == "i":
        X = torch.randint(0, 8, shape, device=DEV, generator=g, dtype=DTYPES[dtype])
    else:
        X = torch.rand(shape, device=DEV, generator=g, dtype=DTYPES[dtype])
    return X.t() if col else X


def _spmm_inputs(c, seed):
    g = _gen(seed)
    src, dst = _rmat(c["n"], c["degree"], g)
    vals = None
    if c["weighted"]:
        if c["dtype"][0] == "i":
            vals = torch.randint(1, 6, (src.numel(),), device=DEV, generator=g, dtype=DTYPES[c["dtype"]])
        else:
            vals = torch.rand(src.numel(), device=DEV, generator=g, dtype=DTYPES[c["dtype"]])
    scale = None
    if c["scaled"]:  # D^-1/2 of the given degrees, 0 for a vertex without edges
        both = torch.cat([src, dst])
        deg = torch.bincount(both, minlength=c["n"]).double()
        scale = torch.where(deg > 0, deg.clamp(min=1).rsqrt(), torch.zeros_like(deg))
    return src, dst, vals, scale, _dense(c["n"], c["k"], c["dtype"], g, c["col"])


def _tall(c, seed):
    g = _gen(seed)
    dt = DTYPES[c["dtype"]]
    A = torch.randn((c["n"], c["ka"]), device=DEV, generator=g, dtype=dt)
    if c["kind"] == "gram":
        return A, torch.randn((c["n"], c["kb"]), device=DEV, generator=g, dtype=dt)
    C = torch.randn((c["ka"], c["kc"]), device=DEV, generator=g, dtype=torch.float64) / math.sqrt(c["ka"])
    return A, C, torch.randn((c["n"], c["kc"]), device=DEV, generator=g, dtype=dt)


class _Graph:
    """What WarmStartNet asks of a graph: the matrix, features, D^-1/2 and the
    wanted subspace (here the first 16 blocks' indicator vectors)."""

    def __init__(self, c, seed, with_matrix=True):
        n = self.n = c["n"]
        g = _gen(seed)
        self.src, self.dst, bound = _blocks(n, c["degree"], g)
        pairs = _pairs(self.src, self.dst, n, True)[0]
        deg = torch.bincount(pairs // n, minlength=n).double()
        self.dinv = torch.where(deg > 0, deg.clamp(min=1).rsqrt(), torch.zeros_like(deg))
        self.X0 = torch.zeros((n, 16), device=DEV)
        self.X0[:, 0] = torch.log1p(deg).float()
        self.X0[:, 1:9] = torch.rand((n, 8), device=DEV, generator=g) * 2 - 1
        block = torch.searchsorted(bound, torch.arange(n, device=DEV), right=True) - 1
        size = (bound[1:] - bound[:-1]).double()
        self.U = torch.zeros((n, NEV), device=DEV)
        for j in range(NEV):
            self.U[:, j] = (block == j).float() * float(size[j].rsqrt())
        self.params = learned.init_params(seed % 1000)
        if with_matrix:
            self.spm = F.SparseMatrix.build(self.src, self.dst, n=n, log2_h=learned.LOG2_H, log2_w=learned.LOG2_W,
                                            flags=F.BUILD_DEDUP | F.BUILD_SYMMETRIZE)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "spmm":
        src, dst, vals, scale, X = _spmm_inputs(c, seed)
        flags = F.BUILD_DEDUP | (F.BUILD_SYMMETRIZE if c["sym"] else 0)
        if vals is None:
            A = F.SparseMatrix.build(src, dst, n=c["n"], log2_h=c["tile"], flags=flags)
        else:
            A = F.SparseMatrix.build_weighted(src, dst, vals, n=c["n"], log2_h=c["tile"], flags=flags)
        Y = torch.empty((c["k"], c["n"]), dtype=X.dtype, device=DEV).t() if c["col"] else torch.empty_like(X)
        return {"case": c, "A": A, "X": X, "Y": Y, "scale": scale}
    if kind in ("gram", "gemm"):
        return {"case": c, "ops": _tall(c, seed)}
    if kind in ("pagerank", "nmf"):
        src, dst = _rmat(c["n"], c["degree"], _gen(seed))
        return {"case": c, "A": F.SparseMatrix.build(src, dst, n=c["n"]),
                "At": F.SparseMatrix.build(dst, src, n=c["n"]), "seed": seed}
    if kind == "build":
        g = _gen(seed)
        src, dst = _rmat(c["n"], c["degree"], g)
        return {"case": c, "src": src, "dst": dst, "X": _dense(c["n"], 4, "i32", g)}
    graph = _Graph(c, seed)
    return {"case": c, "graph": graph, "net": learned.WarmStartNet(params=graph.params)}


# ---- one pass ----------------------------------------------------------------

def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "spmm":
        A, X, Y = state["A"], state["X"], state["Y"]
        if c["scaled"]:
            return A.multiply_scaled_async(X, Y, pre=state["scale"], post=state["scale"])
        return A.multiply_async(X, Y, seq=c["seq"])
    if kind == "gram":
        return F.gram(*state["ops"])
    if kind == "gemm":
        A, C, Y = state["ops"]
        if c["beta"] == 0.0:
            return F.gemm_tall(A, C)
        return F.gemm_tall(A, C, alpha=-1.0, beta=c["beta"], Y=Y)
    if kind == "pagerank":
        return F.pagerank(state["A"], state["At"], max_iters=c["iters"])[0]
    if kind == "nmf":
        W, tH, dist = F.nmf(state["A"], c["k"], max_iters=c["iters"], At=state["At"], seed=state["seed"])
        return {"W": W, "tH": tH, "dist": dist}
    if kind == "build":
        flags = F.BUILD_DEDUP | (F.BUILD_SYMMETRIZE if c["sym"] else 0)
        A = F.SparseMatrix.build(state["src"], state["dst"], n=c["n"], log2_h=c["tile"], flags=flags)
        return {"Y": A.multiply(state["X"]), "nnz": A.get_nnz(), "bytes": A.info.image_bytes}
    g, net = state["graph"], state["net"]
    Y = net.forward(g)
    if not c["train"]:
        return Y
    acts, work, _, dY = net._buffers(g.n)
    ctx, L = g.spm.ctx, F.lib()
    loss = ctypes.c_double()
    ctx.check(L.fmx_subspace_loss(ctx.handle, g.n, NEV, Y.data_ptr(), g.U.data_ptr(), ctypes.byref(loss),
                                  dY.data_ptr(), None), "fmx_subspace_loss")
    ctx.check(L.fmx_gnn_backward(ctx.handle, g.spm.handle, g.dinv.data_ptr(), net.P.data_ptr(), g.X0.data_ptr(),
                                 acts.data_ptr(), dY.data_ptr(), net.G.data_ptr(), work.data_ptr(), net.mode, None),
              "fmx_gnn_backward")
    return {"Y": Y, "loss": loss.value, "grads": net.G}


# ---- what a pass cannot do without -------------------------------------------

def work(case):
    """Bytes and operations of one pass, each input read once and each result
    written once.  A non-zero is 4 bytes (its column and its row inside a
    tile), plus its value if it has one."""
    c, kind, n = case, case["kind"], case["n"]
    edges = n * c.get("degree", 0)
    if kind == "spmm":
        s = SIZE[c["dtype"]]
        nnz = edges * (2 if c["sym"] else 1)
        return {"bytes": nnz * (4 + (s if c["weighted"] else 0)) + 2 * n * c["k"] * s + (16 * n if c["scaled"] else 0),
                "flops": 2.0 * nnz * c["k"]}
    if kind == "gram":
        return {"bytes": n * (c["ka"] + c["kb"]) * SIZE[c["dtype"]] + 8 * c["ka"] * c["kb"],
                "flops": 2.0 * n * c["ka"] * c["kb"]}
    if kind == "gemm":
        cols = c["ka"] + c["kc"] * (2 if c["beta"] else 1)
        return {"bytes": n * cols * SIZE[c["dtype"]], "flops": 2.0 * n * c["ka"] * c["kc"]}
    if kind == "pagerank":  # the degrees' product, then a sweep reads the transpose, the ranks and the degrees
        return {"bytes": edges * 4 + 4 * n + c["iters"] * (edges * 4 + 12 * n), "flops": 2.0 * edges * (c["iters"] + 1)}
    if kind == "nmf":  # both products and both updates: each factor is read twice and written once
        k = c["k"]
        return {"bytes": c["iters"] * (edges * 8 + 6 * n * k * 4),
                "flops": c["iters"] * (4.0 * edges * k + 8.0 * n * k * k)}
    if kind == "build":  # the edge list, the image once written and once read, the product's operands
        nnz = edges * (2 if c["sym"] else 1)
        return {"bytes": 8 * edges + 8 * nnz + 32 * n, "flops": 2.0 * nnz * 4}
    # per layer: the matrix, H read, N H and the next H written; twice that back
    fwd = 3 * edges * 4 + n * 4 * (16 + 16 + 64 + 2 * (64 + 64 + 64) + 64 + 16)
    flops = 2.0 * (edges * (16 + 64 + 64) + n * (32 * 64 + 2 * 128 * 64 + 64 * 16))
    return {"bytes": fwd * (3 if c["train"] else 1), "flops": flops * (3 if c["train"] else 1)}


# ---- the same in 64 bits -----------------------------------------------------

def _pairs(src, dst, n, sym, vals=None):
    """The distinct non-zeros row * n + column in order, without the
    diagonal, and each one's value (the first edge's among equals)."""
    a, b = src.long(), dst.long()
    keys = torch.stack([a * n + b, b * n + a], 1).flatten() if sym else a * n + b
    keep = torch.stack([a != b, a != b], 1).flatten() if sym else a != b
    keys = keys[keep]
    if vals is None:
        return torch.unique(keys), None
    v = (torch.stack([vals, vals], 1).flatten() if sym else vals)[keep]
    keys, order = torch.sort(keys, stable=True)
    first = torch.ones_like(keys, dtype=torch.bool)
    first[1:] = keys[1:] != keys[:-1]
    return keys[first], v[order][first]


def _times(keys, n, X, vals=None):
    """A X for the non-zeros keys, in X's type, some millions at a time."""
    Y = torch.zeros((n, X.shape[1]), dtype=X.dtype, device=DEV)
    step = max(1 << 16, (1 << 26) // X.shape[1])
    for i in range(0, keys.numel(), step):
        part = keys[i:i + step]
        rows = X[part % n]
        if vals is not None:
            rows = rows * vals[i:i + step, None].to(X.dtype)
        Y.index_add_(0, part // n, rows)
    return Y


class _Agg(torch.autograd.Function):
    """N H for the symmetric N = D^-1/2 A D^-1/2."""

    @staticmethod
    def forward(ctx, H, graph):
        ctx.graph = graph
        return _Agg.times(H, graph)

    @staticmethod
    def backward(ctx, dOut):
        return _Agg.times(dOut, ctx.graph), None

    @staticmethod
    def times(H, graph):
        keys, n, dinv = graph
        return _times(keys, n, H * dinv[:, None]) * dinv[:, None]


def exact(case, seed):
    c, kind = case, case["kind"]
    n = c["n"]
    if kind == "spmm":
        if c["dtype"][0] == "i":
            return None  # whole numbers
        src, dst, vals, scale, X = _spmm_inputs(c, seed)
        keys, v = _pairs(src, dst, n, c["sym"], vals)
        X = X.double()
        if scale is not None:
            return _times(keys, n, X * scale[:, None], v) * scale[:, None]
        return _times(keys, n, X, v)
    if kind in ("gram", "gemm"):
        step, ops = 1 << 18, _tall(c, seed)
        if kind == "gram":
            A, B = ops
            return sum(A[i:i + step].double().t().contiguous() @ B[i:i + step].double() for i in range(0, n, step))
        A, C, Y = ops
        if c["beta"] == 0.0:
            return torch.cat([A[i:i + step].double() @ C for i in range(0, n, step)])
        return torch.cat([c["beta"] * Y[i:i + step].double() - A[i:i + step].double() @ C for i in range(0, n, step)])
    if kind == "pagerank":
        src, dst = _rmat(n, c["degree"], _gen(seed))
        keys = _pairs(src, dst, n, False)[0]
        back = (keys % n) * n + keys // n
        deg = torch.bincount(keys // n, minlength=n).double().clamp(min=1)
        pr = torch.full((n,), 1.0 / n, dtype=torch.float64, device=DEV)
        for _ in range(c["iters"]):
            new = 0.85 * _times(back, n, (pr / deg)[:, None])[:, 0] + 0.15 / n
            done = bool(((new - pr).abs() < 0.001 / n).all())
            pr = new
            if done:
                break
        return pr
    if kind == "nmf":
        g = _gen(seed)
        src, dst = _rmat(n, c["degree"], g)
        keys = _pairs(src, dst, n, False)[0]
        back = (keys % n) * n + keys // n
        g = _gen(seed)
        W = torch.rand((n, c["k"]), device=DEV, generator=g).double()
        tH = torch.rand((n, c["k"]), device=DEV, generator=g).double()
        eps, dist = 1e-8, []
        for it in range(c["iters"]):
            tH = (tH * _times(back, n, W)).clamp(min=eps) / (tH @ (W.t().contiguous() @ W) + eps)
            W = (W * _times(keys, n, tH)).clamp(min=eps) / (W @ (tH.t().contiguous() @ tH) + eps)
            if it % 5 == 0:
                G = W.t().contiguous() @ W
                dist.append(float(keys.numel() - 2 * (_times(back, n, W) * tH).sum() + ((tH @ G) * tH).sum()))
        return {"W": W, "tH": tH, "dist": dist}
    if kind == "build":
        return None  # whole numbers
    g = _Graph(c, seed, with_matrix=False)
    graph = (_pairs(g.src, g.dst, n, True)[0], n, g.dinv)
    P = torch.from_numpy(g.params).to(DEV).double().requires_grad_(c["train"])
    at, H = 0, g.X0.double()

    def take(rows, cols):
        nonlocal at
        at += rows * cols
        return P[at - rows * cols:at].view(rows, cols)

    for d in (16, 64, 64):
        Ws, Wn, b = take(d, 64), take(d, 64), take(1, 64)
        H = torch.relu(H @ Ws + _Agg.apply(H, graph) @ Wn + b)
    Y = H @ take(64, NEV)
    if not c["train"]:
        return Y
    U = g.U.double()
    G, C = Y.t().contiguous() @ Y, U.t().contiguous() @ Y
    loss = NEV - torch.trace(torch.linalg.solve(G, C.t().contiguous() @ C))
    grads, = torch.autograd.grad(loss, P)
    return {"Y": Y.detach(), "loss": float(loss), "grads": grads}
