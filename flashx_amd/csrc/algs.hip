// algs.hip -- callers of the SpMM path: PageRank (k = 1) and NMF (k columns).
//
// fmx_pagerank restates matrix/libmatrix-algs/PageRank.cpp:49-137 on the
// device, FP32 as the reference computes it:
//   out_deg = max(A * 1, 1)                       (get_out_degree, :49-60, :83)
//   pr = 1/n                                      (mat_init_operate, :31-43)
//   repeat: in = pr / out_deg; pr1 = in * out_deg (:101-105; pr_init, pr_step)
//           out = A^T * in                        (:110, the SpMM kernel, k = 1)
//           pr2 = d * out + (1 - d) / n           (:118-119)
//           converged = #{|pr1 - pr2| < 0.001/n}  (:97, :120-124); pr = pr2
//   until every vertex has converged or max_iters.
// The element-wise steps use explicitly rounded operations, so that no
// multiply-add is contracted and each step rounds as the reference's does;
// only the SpMV sum differs (FP64 accumulation, rounded once).
#include <algorithm>
#include <vector>

#include "dense.h"
#include "fmx_internal.h"

namespace fmx {
namespace {

constexpr int kT = 256;

uint32_t grid_for_n(fmx_ctx *ctx, uint64_t n)
{
    uint64_t b = (n + kT - 1) / kT;
    uint64_t cap = (uint64_t)ctx->num_cus * 8;
    return (uint32_t)(b < 1 ? 1 : (b > cap ? cap : b));
}

__global__ void __launch_bounds__(kT) pr_fill(float *x, uint64_t n, float v)
{
    for (uint64_t i = blockIdx.x * (uint64_t)kT + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kT) x[i] = v;
}

__global__ void __launch_bounds__(kT) pr_init(float *deg, float *pr, float *in, uint64_t n, float p0)
{
    for (uint64_t i = blockIdx.x * (uint64_t)kT + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kT) {
        const float d = deg[i] > 1.0f ? deg[i] : 1.0f;
        deg[i] = d;
        pr[i] = p0;
        in[i] = __fdiv_rn(p0, d);
    }
}

// One iteration's element-wise steps behind its SpMV, and the next SpMV's
// operand: pr1 is recomputed from this iteration's operand instead of being
// stored, so a vertex costs three loads and two stores.  Each block writes
// its count of converged vertices to counts (host memory that the device
// sees), which the host adds up: one atomic counter for all waves made this
// the longest kernel of an iteration (2^20 vertices: 93 us, the atomics
// queueing on one word; 7 us like this).
__global__ void __launch_bounds__(kT) pr_step(const float *out, const float *deg, float *pr, float *in, uint64_t n,
                                              float damping, float add, float eps, uint32_t *counts)
{
    __shared__ uint32_t wave[kT / 64];
    uint32_t c = 0;
    for (uint64_t i = blockIdx.x * (uint64_t)kT + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kT) {
        const float d = deg[i];
        const float p1 = __fmul_rn(in[i], d);
        const float p2 = __fadd_rn(__fmul_rn(out[i], damping), add);
        c += fabsf(p1 - p2) < eps ? 1u : 0u;
        pr[i] = p2;
        in[i] = __fdiv_rn(p2, d);
    }
    for (int d = 32; d; d >>= 1) c += __shfl_xor(c, d, 64);
    if ((threadIdx.x & 63) == 0) wave[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (int w = 0; w < kT / 64; w++) t += wave[w];
        counts[blockIdx.x] = t;
    }
}

// X = max(X * N, eps) / (X G + eps), X rows x k, G k x k: the denominators'
// FP64 sums are rounded to FP32, and every FP32 step is rounded
// (fm.pmax2(X * N, eps) / (den + eps), NMF.cpp:180-192,206-217).  The
// denominators never reach memory: X and N are read and X written once, which
// bounds it (260,000 x 20: 63 MB).  A block stages rows of X, and G, in LDS,
// zero-padded to four columns; a thread keeps four rows by four columns, rows
// `rg` apart so that neighbouring lanes read different banks.  FP64 FMAs and
// the FP64 matrix cores run at one rate, and the former need no padding to 16.
// 260,000 x 20: 19 us, where the product (22) and an element-wise update
// reading its result (13) took 35; an iteration over 262,144 vertices, 8 edges
// each: 122 / 97 us at 4 columns, 249 / 220 at 20, 949 / 683 at 64.
constexpr int kUpdRows = 4, kUpdCols = 4;

struct UpdShape {
    int k, k4, cg, rg, ks;  // columns, padded to 4; column groups, row groups; LDS row stride of X (words)
    __host__ __device__ explicit UpdShape(int k_) : k(k_)
    {
        k4 = (k + 3) & ~3;
        cg = k4 / kUpdCols;
        rg = kT / cg;
        ks = k4 % 8 ? k4 : k4 + 4;
    }
    __host__ __device__ int rows() const { return kUpdRows * rg; }
    size_t lds() const { return (size_t)k4 * k4 * 8 + (size_t)rows() * ks * 4; }
};

template <bool VEC>
__global__ void __launch_bounds__(kT) nmf_update(float *X, const float *N, const double *G, uint64_t n, int k_,
                                                 float eps)
{
    extern __shared__ double lds_g[];
    const UpdShape f(k_);
    float *lds_x = (float *)(lds_g + f.k4 * f.k4);
    for (int e = threadIdx.x; e < f.k4 * f.k4; e += kT) {
        const int i = e / f.k4, j = e % f.k4;
        lds_g[e] = i < f.k && j < f.k ? G[i * f.k + j] : 0.0;
    }
    const int r = threadIdx.x / f.cg, c0 = threadIdx.x % f.cg * kUpdCols;
    for (uint64_t t0 = blockIdx.x * (uint64_t)f.rows(); t0 < n; t0 += gridDim.x * (uint64_t)f.rows()) {
        const int rows = (int)min((uint64_t)f.rows(), n - t0);
        __syncthreads();  // the last tile's rows are read
        if constexpr (VEC) {
            for (int e = threadIdx.x; e < rows * f.cg; e += kT)
                *(float4 *)(lds_x + e / f.cg * f.ks + e % f.cg * 4) = *(const float4 *)(X + t0 * f.k + e * 4);
        } else {
            for (int e = threadIdx.x; e < rows * f.k4; e += kT) {
                const int i = e / f.k4, j = e % f.k4;
                lds_x[i * f.ks + j] = j < f.k ? X[(t0 + i) * f.k + j] : 0.0f;
            }
        }
        __syncthreads();
        if (r >= f.rg || r >= rows) continue;  // every thread reaches the next tile's barrier
        float num[kUpdRows][kUpdCols];
#pragma unroll
        for (int q = 0; q < kUpdRows; q++) {
            const int row = r + q * f.rg;
            const float *p = N + (t0 + row) * f.k + c0;
            if constexpr (VEC) {
                const float4 v = row < rows ? *(const float4 *)p : float4{0, 0, 0, 0};
                num[q][0] = v.x;
                num[q][1] = v.y;
                num[q][2] = v.z;
                num[q][3] = v.w;
            } else {
#pragma unroll
                for (int j = 0; j < kUpdCols; j++) num[q][j] = row < rows && c0 + j < f.k ? p[j] : 0.0f;
            }
        }
        double acc[kUpdRows][kUpdCols] = {};
        const float *xr[kUpdRows];  // (rows past the end read the first row)
#pragma unroll
        for (int q = 0; q < kUpdRows; q++) xr[q] = lds_x + (r + q * f.rg < rows ? r + q * f.rg : r) * f.ks;
        for (int i = 0; i < f.k4; i += 4) {
            float x[kUpdRows][4];
#pragma unroll
            for (int q = 0; q < kUpdRows; q++) {
                const float4 v = *(const float4 *)(xr[q] + i);
                x[q][0] = v.x;
                x[q][1] = v.y;
                x[q][2] = v.z;
                x[q][3] = v.w;
            }
#pragma unroll
            for (int h = 0; h < 4; h++) {
                const double *g = lds_g + (i + h) * f.k4 + c0;
#pragma unroll
                for (int j = 0; j < kUpdCols; j++)
#pragma unroll
                    for (int q = 0; q < kUpdRows; q++) acc[q][j] = fma((double)x[q][h], g[j], acc[q][j]);
            }
        }
#pragma unroll
        for (int q = 0; q < kUpdRows; q++) {
            const int row = r + q * f.rg;
            if (row >= rows) continue;
            float y[kUpdCols];
#pragma unroll
            for (int j = 0; j < kUpdCols; j++)
                y[j] = __fdiv_rn(fmaxf(__fmul_rn(xr[q][c0 + j], num[q][j]), eps), __fadd_rn((float)acc[q][j], eps));
            float *p = X + (t0 + row) * f.k + c0;
            if constexpr (VEC) {
                *(float4 *)p = float4{y[0], y[1], y[2], y[3]};
            } else {
#pragma unroll
                for (int j = 0; j < kUpdCols; j++)
                    if (c0 + j < f.k) p[j] = y[j];
            }
        }
    }
}

}  // namespace
}  // namespace fmx

using namespace fmx;

extern "C" {

fmx_status fmx_pagerank(fmx_ctx *ctx, const fmx_spm *A, const fmx_spm *At, int max_iters, float damping,
                        float *pr, int *iters, void *stream)
{
    if (!ctx || !A || !pr) return fail(ctx, FMX_EINVAL, "null argument");
    if (!At) At = A;
    if (A->nrows != A->ncols || At->nrows != A->nrows || At->ncols != A->ncols)
        return fail(ctx, FMX_EDIM, "PageRank needs a square matrix and its transpose");
    if (A->esz || At->esz) return fail(ctx, FMX_EUNSUPPORTED, "PageRank runs on binary matrices");
    if (max_iters < 0) return fail(ctx, FMX_EINVAL, "max_iters must be >= 0");
    FMX_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = (hipStream_t)stream;
    const uint64_t n = A->nrows;
    if (iters) *iters = 0;
    if (n == 0) return FMX_OK;
    // per-block counts of converged vertices, in the context's pinned memory
    const uint32_t gs = (uint32_t)std::min<uint64_t>({(n + kT - 1) / kT, (uint64_t)ctx->num_cus * 2, 1024});
    uint32_t *counts = (uint32_t *)((char *)ctx->pinned + kPinnedCounts);
    float *buf = nullptr;
    hipEvent_t ev = nullptr;
    FMX_HIP(ctx, dev_malloc(ctx, (void **)&buf, 3 * n * sizeof(float)));
    if (hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) {
        (void)hipFree(buf);
        return fail(ctx, FMX_EHIP, "PageRank event");
    }
    float *deg = buf, *in = buf + n, *out = buf + 2 * n;
    const uint32_t g = grid_for_n(ctx, n);
    fmx_status st = FMX_OK;
    // out_deg = max(A * 1, 1); the ones vector lives in `in` for this step
    hipLaunchKernelGGL(pr_fill, dim3(g), dim3(kT), 0, s, in, n, 1.0f);
    st = fmx_spmm(ctx, A, FMX_F32, 1, in, 1, deg, 1, s);
    if (!st) {
        hipLaunchKernelGGL(pr_init, dim3(g), dim3(kT), 0, s, deg, pr, in, n, (float)(1.0 / (double)n));
        const float eps = (float)(0.001 / (double)n);
        const float add = (float)((1.0 - (double)damping) / (double)n);
        // The next SpMV is launched before the host waits for this step's
        // counts, which would leave the GPU idle for 22 us an iteration; it
        // touches only `out`, which nothing reads if this was the last step.
        // That one SpMV is then for nothing, so it is only done where it
        // takes less than ten such gaps (0.2 ms: about 2^25 non-zeros).
        const bool ahead = !At->streamed() && At->nnz <= (1ull << 25);
        int it = 0;
        if (max_iters) st = fmx_spmm(ctx, At, FMX_F32, 1, in, 1, out, 1, s);
        while (!st && it < max_iters) {
            hipLaunchKernelGGL(pr_step, dim3(gs), dim3(kT), 0, s, out, deg, pr, in, n, damping, add, eps,
                               counts);
            if (hipGetLastError() != hipSuccess) {
                st = fail(ctx, FMX_EHIP, "PageRank step");
                break;
            }
            if (++it == max_iters) break;  // the counts no longer matter
            bool ok = hipEventRecord(ev, s) == hipSuccess;
            if (ok && ahead) st = fmx_spmm(ctx, At, FMX_F32, 1, in, 1, out, 1, s);
            if (st) break;
            if (!ok || hipEventSynchronize(ev) != hipSuccess) {
                st = fail(ctx, FMX_EHIP, "PageRank convergence count");
                break;
            }
            uint64_t c = 0;
            for (uint32_t b = 0; b < gs; b++) c += ((volatile uint32_t *)counts)[b];
            if (c >= n) break;
            if (!ahead) st = fmx_spmm(ctx, At, FMX_F32, 1, in, 1, out, 1, s);
        }
        if (iters) *iters = it;
    }
    if (hipStreamSynchronize(s) != hipSuccess && !st) st = fail(ctx, FMX_EHIP, "PageRank");
    (void)hipEventDestroy(ev);
    (void)hipFree(buf);
    return st;
}

// NMF by Lee-Seung multiplicative updates, matrix/libmatrix-algs/NMF.cpp:
// 164-230 (update_lee) and 259-316 (NMF), with H kept transposed (tH, m x k
// row-major: the reference's L_COL k x m H byte for byte).  Per iteration:
//   tD  = tH * (W^T W)                      (:168-173)
//   tH  = max(tH .* (A^T W), eps) ./ (tD + eps)   (:176-193)
//   D2  = W * (tH^T tH)                     (:201-208)
//   W   = max(W .* (A tH), eps) ./ (D2 + eps)     (:211-224)
//   WtW = W^T W                             (:227-228)
// and after iterations 0, 5, 10, ... the distance ||A - W H||_F^2 =
// nnz - 2 tr((A^T W)^T tH) + tr((tH WtW)^T tH) (Fnorm, :110-126).  The SpMMs
// are FP32 (FP64 sums rounded once), the Gram and k x k products accumulate
// in FP64 (the reference: FP32 BLAS), the update is FP32.
fmx_status fmx_nmf(fmx_ctx *ctx, const fmx_spm *A, const fmx_spm *At, int k, int max_iters, float *W, float *tH,
                   double *dist, void *stream)
{
    if (!ctx || !A || !W || !tH) return fail(ctx, FMX_EINVAL, "null argument");
    if (A->esz) return fail(ctx, FMX_EUNSUPPORTED, "can only handle binary sparse matrix");
    if (!At) {
        if (A->nrows != A->ncols) return fail(ctx, FMX_EDIM, "a non-square matrix needs its transpose");
        At = A;
    }
    if (At->esz) return fail(ctx, FMX_EUNSUPPORTED, "can only handle binary sparse matrix");
    if (At->nrows != A->ncols || At->ncols != A->nrows) return fail(ctx, FMX_EDIM, "At is not A's transpose");
    if (k < 1 || k > 64) return fail(ctx, FMX_EDIM, "NMF rank must be in [1, 64]");
    if (max_iters < 0) return fail(ctx, FMX_EINVAL, "max_iters must be >= 0");
    FMX_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = (hipStream_t)stream;
    const uint64_t n = A->nrows, m = A->ncols;
    const float eps = 10e-9f;
    float *buf = nullptr;
    double *g = nullptr;
    const uint64_t big = std::max(n, m) * (uint64_t)k;
    FMX_HIP(ctx, dev_malloc(ctx, (void **)&buf, 2 * big * sizeof(float)));
    if (dev_malloc(ctx, (void **)&g, 2 * (size_t)k * k * sizeof(double)) != hipSuccess) {
        (void)hipFree(buf);
        return fail(ctx, FMX_ENOMEM, "NMF Gram buffers");
    }
    float *P = buf, *Q = buf + big;  // (m|n) x k products; the distance's tH W^T W
    double *G = g, *G2 = g + (size_t)k * k;
    std::vector<double> h1((size_t)k * k), h2((size_t)k * k);
    auto upd = [&](float *X, const double *den, uint64_t rows) {
        const UpdShape f(k);
        const uint64_t tiles = (rows + f.rows() - 1) / f.rows();
        const dim3 grid((uint32_t)std::min<uint64_t>(tiles, (uint64_t)ctx->num_cus * 8));
        if (!tiles) return FMX_OK;
        if (k % 4 == 0 && (uintptr_t)X % 16 == 0)
            hipLaunchKernelGGL(nmf_update<true>, grid, dim3(kT), f.lds(), s, X, P, den, rows, k, eps);
        else
            hipLaunchKernelGGL(nmf_update<false>, grid, dim3(kT), f.lds(), s, X, P, den, rows, k, eps);
        return hipGetLastError() == hipSuccess ? FMX_OK : fail(ctx, FMX_EHIP, "NMF update launch");
    };
    fmx_status st = gram(ctx, FMX_F32, FMX_GRAM_F64, n, k, k, W, k, W, k, G, s);  // W^T W
    for (int it = 0; !st && it < max_iters; it++) {
        if (!st) st = fmx_spmm(ctx, At, FMX_F32, k, W, k, P, k, s);
        if (!st) st = upd(tH, G, m);
        if (!st) st = gram(ctx, FMX_F32, FMX_GRAM_F64, m, k, k, tH, k, tH, k, G2, s);  // H H^T
        if (!st) st = fmx_spmm(ctx, A, FMX_F32, k, tH, k, P, k, s);
        if (!st) st = upd(W, G2, n);
        if (!st) st = gram(ctx, FMX_F32, FMX_GRAM_F64, n, k, k, W, k, W, k, G, s);
        if (!st && dist && it % 5 == 0) {
            st = fmx_spmm(ctx, At, FMX_F32, k, W, k, P, k, s);                            // A^T W
            if (!st) st = gram(ctx, FMX_F32, FMX_GRAM_F64, m, k, k, P, k, tH, k, G2, s);  // (A^T W)^T tH
            if (!st && hipMemcpyAsync(h1.data(), G2, h1.size() * 8, hipMemcpyDeviceToHost, s) != hipSuccess)
                st = fail(ctx, FMX_EHIP, "NMF distance");
            if (!st) st = gemm_tall(ctx, FMX_F32, m, k, k, 1.0, tH, k, G, 0.0, Q, k, s);  // tH W^T W
            if (!st) st = gram(ctx, FMX_F32, FMX_GRAM_F64, m, k, k, Q, k, tH, k, G2, s);
            if (!st && (hipMemcpyAsync(h2.data(), G2, h2.size() * 8, hipMemcpyDeviceToHost, s) != hipSuccess ||
                        hipStreamSynchronize(s) != hipSuccess))
                st = fail(ctx, FMX_EHIP, "NMF distance");
            if (!st) {
                double t1 = 0, t2 = 0;
                for (int j = 0; j < k; j++) {
                    t1 += h1[(size_t)j * k + j];
                    t2 += h2[(size_t)j * k + j];
                }
                dist[it / 5] = (double)A->nnz - 2.0 * t1 + t2;
            }
        }
    }
    (void)hipStreamSynchronize(s);
    (void)hipFree(buf);
    (void)hipFree(g);
    return st;
}

}  // extern "C"
