// gnn.hip -- the learned warm start: a 3-layer message-passing network that
// predicts the starting block of the block Krylov eigensolver.
//
// No reference counterpart (the reference starts Anasazi from a random block,
// matrix/eigensolver/FM_MultiVector.h:164-168).  Network, for the normalised
// adjacency N = D^-1/2 A D^-1/2:
//   H0 = X0 (n x 16: log(1+deg), 8 uniform features, 7 zeros)
//   Agg_l = N H_l                      (an SpMM with its output rows scaled;
//                                       the product before it also writes D^-1/2 H_l)
//   H_{l+1} = relu(H_l Ws_l + Agg_l Wn_l + b_l),  l = 0, 1, 2  (hidden 64)
//   Y = H_3 Wo                         (n x 16)
// Dense products run as v_mfma_f32_16x16x32_bf16 with BF16 operands (weights
// and activations rounded to BF16) and FP32 accumulation; a plain-FP32 mode
// exists for gradient checking.  Weight gradients are Gram products (BF16
// MFMA, or FP64), the bias gradient a column sum in the same kernel.
// Parameters, flat FP32: per layer Ws (din x 64), Wn (din x 64), b (64);
// then Wo (64 x 16); din = 16, 64, 64 (19,648 values).
#include <algorithm>
#include <cmath>
#include <vector>

#include "dense.h"
#include "small.h"

namespace fmx {
namespace {

constexpr int kIn = 16, kHid = 64, kOut = 16, kLayers = 3;
constexpr int kT = 256;
constexpr int kKMax = 128;      // max inner dimension
constexpr int kPad = 8;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned short f2bf(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7F800000u) == 0x7F800000u) return (unsigned short)(u >> 16);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

int din_of(int l) { return l == 0 ? kIn : kHid; }

size_t layer_off(int l)
{
    size_t o = 0;
    for (int i = 0; i < l; i++) o += 2ull * din_of(i) * kHid + kHid;
    return o;
}

// What a dense product's epilogue does with out[r][c] = sum_k A[r][k] B[k][c],
// A = [A1 | A2] (n x K), in this order: adds bias[c], adds add[r][c], clears a
// negative value (relu), clears it where gate[r][c] is not positive (the ReLU's
// backward step); then stores the value to out and, times scale[r], to outs.
// Every matrix of it is n x dout without gaps; a null pointer leaves its step
// out.
struct Epilogue {
    const float *bias = nullptr, *add = nullptr, *gate = nullptr;
    const double *scale = nullptr;
    int relu = 0;
    float *out = nullptr, *outs = nullptr;
};

// N floats moved by one load or store, at any float's address.
template <int N>
struct FV {
    float v[N];
};
using F4 = FV<4>;

__device__ __forceinline__ bf16x8 to_bf16(const F4 &a, const F4 &b)
{
    bf16x8 r;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        r[i] = (__bf16)a.v[i];
        r[i + 4] = (__bf16)b.v[i];
    }
    return r;
}

// BF16 MFMA form, K = d1 + d2 <= 32 * KS, dout = 16 * NT; B = W (K x dout) or
// W^T (W dout x K, wtrans).  Bound by the operands' bytes: each wave takes 16
// rows at a time straight from memory into the MFMA operand (a lane's 8
// consecutive k of one row are two 16-byte loads; rounded to BF16 by the
// hardware's pair conversion), B stays in registers for the whole kernel, and
// output tile t of lane p is column NT * p + t, so that a lane stores NT
// consecutive columns.  131,072 rows, 128 -> 64: 46 us with both operands
// staged in LDS by 4-byte loads and 11 us for the scaled copy in a kernel of
// its own, 37 us together like this (100 MB moved, 2.7 TB/s); 64 -> 64 20 us.
template <int KS, int NT>
__global__ void __launch_bounds__(kT) gnn_mfma_kernel(const float *A1, int d1, const float *A2, int d2,
                                                      const float *W, int wtrans, Epilogue ep, uint64_t n)
{
    constexpr int KP = KS * 32, DO = NT * 16, LD = KP + kPad;
    __shared__ unsigned short Bt[DO * LD];
    const int K = d1 + d2;
    // (DO * KP is a multiple of 2 * kT; consecutive threads read consecutive
    // words of W, several in flight)
    constexpr int PER = DO * KP / kT, STEP = PER < 8 ? PER : 8;
    for (int i0 = 0; i0 < PER; i0 += STEP) {
        float v[STEP];
#pragma unroll
        for (int i = 0; i < STEP; i++) {
            const int e = (i0 + i) * kT + threadIdx.x;
            const int c = wtrans ? e / KP : e % DO, k = wtrans ? e % KP : e / DO, kc = k < K ? k : 0;
            v[i] = W[wtrans ? c * K + kc : kc * DO + c];
            if (k >= K) v[i] = 0.f;
        }
#pragma unroll
        for (int i = 0; i < STEP; i++) {
            const int e = (i0 + i) * kT + threadIdx.x;
            const int c = wtrans ? e / KP : e % DO, k = wtrans ? e % KP : e / DO;
            Bt[c * LD + k] = f2bf(v[i]);
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, p = lane & 15, kg = (lane >> 4) * 8;
    bf16x8 b[KS][NT];
#pragma unroll
    for (int s = 0; s < KS; s++)
#pragma unroll
        for (int t = 0; t < NT; t++) b[s][t] = *(const bf16x8 *)(Bt + (NT * p + t) * LD + s * 32 + kg);
    FV<NT> bias{};
    if (ep.bias) bias = *(const FV<NT> *)(ep.bias + NT * p);
    const uint64_t waves = (uint64_t)gridDim.x * (kT / 64);
    for (uint64_t r0 = (blockIdx.x * (uint64_t)(kT / 64) + (threadIdx.x >> 6)) * 16; r0 < n; r0 += waves * 16) {
        const uint64_t ar = r0 + p < n ? r0 + p : n - 1;  // rows past the end are not stored
        F4 x[KS][2];
#pragma unroll
        for (int s = 0; s < KS; s++) {
            const int k = s * 32 + kg;
            // (d1 is a multiple of 8, so a lane's k all lie in one operand)
            const float *src = k < d1 ? A1 + ar * d1 + k : A2 + ar * d2 + (k - d1);
            if (k < K) {
                x[s][0] = *(const F4 *)src;
                x[s][1] = *(const F4 *)(src + 4);
            } else {
                x[s][0] = x[s][1] = F4{{0.f, 0.f, 0.f, 0.f}};
            }
        }
        floatx4 acc[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KS; s++) {
            const bf16x8 a = to_bf16(x[s][0], x[s][1]);
#pragma unroll
            for (int t = 0; t < NT; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[s][t], acc[t], 0, 0, 0);
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint64_t row = r0 + (lane >> 4) * 4 + q;
            if (row >= n) continue;
            const uint64_t at = row * DO + NT * p;
            FV<NT> y, ys;
#pragma unroll
            for (int t = 0; t < NT; t++) y.v[t] = acc[t][q];
            if (ep.bias) {
#pragma unroll
                for (int t = 0; t < NT; t++) y.v[t] += bias.v[t];
            }
            if (ep.add) {
                const FV<NT> x = *(const FV<NT> *)(ep.add + at);
#pragma unroll
                for (int t = 0; t < NT; t++) y.v[t] += x.v[t];
            }
            if (ep.relu) {
#pragma unroll
                for (int t = 0; t < NT; t++) y.v[t] = y.v[t] > 0.f ? y.v[t] : 0.f;
            }
            if (ep.gate) {
                const FV<NT> x = *(const FV<NT> *)(ep.gate + at);
#pragma unroll
                for (int t = 0; t < NT; t++) y.v[t] = x.v[t] > 0.f ? y.v[t] : 0.f;
            }
            if (ep.out) *(FV<NT> *)(ep.out + at) = y;
            if (ep.outs) {
                const double d = ep.scale[row];
#pragma unroll
                for (int t = 0; t < NT; t++) ys.v[t] = (float)((double)y.v[t] * d);
                *(FV<NT> *)(ep.outs + at) = ys;
            }
        }
    }
}

// FP32 form: 32-row tiles keep the operands in 48 KiB.
__global__ void __launch_bounds__(kT) gnn_f32_kernel(const float *A1, int d1, const float *A2, int d2, const float *W,
                                                     int wtrans, int dout, Epilogue ep, uint64_t n)
{
    constexpr int kR = 32;
    __shared__ float As[kR * (kKMax + 1)];
    __shared__ float Bs[kKMax * kHid];
    const int K = d1 + d2;
    for (int e = threadIdx.x; e < K * dout; e += kT) {
        const int k = e / dout, c = e - k * dout;
        Bs[e] = wtrans ? W[(size_t)c * K + k] : W[(size_t)k * dout + c];
    }
    for (uint64_t r0 = blockIdx.x * (uint64_t)kR; r0 < n; r0 += (uint64_t)gridDim.x * kR) {
        __syncthreads();
        for (int e = threadIdx.x; e < kR * K; e += kT) {
            const int r = e / K, k = e - r * K;
            const uint64_t row = r0 + r;
            float v = 0.f;
            if (row < n) v = k < d1 ? A1[row * d1 + k] : A2[row * d2 + (k - d1)];
            As[r * (kKMax + 1) + k] = v;
        }
        __syncthreads();
        for (int o = threadIdx.x; o < kR * dout; o += kT) {
            const int r = o / dout, c = o - r * dout;
            const uint64_t row = r0 + r;
            if (row >= n) continue;
            float v = 0.f;
            for (int k = 0; k < K; k++) v = fmaf(As[r * (kKMax + 1) + k], Bs[k * dout + c], v);
            const uint64_t at = row * dout + c;
            if (ep.bias) v += ep.bias[c];
            if (ep.add) v += ep.add[at];
            if (ep.relu) v = v > 0.f ? v : 0.f;
            if (ep.gate) v = ep.gate[at] > 0.f ? v : 0.f;
            if (ep.out) ep.out[at] = v;
            if (ep.outs) ep.outs[at] = (float)((double)v * ep.scale[row]);
        }
    }
}

// ---- weight gradients ----------------------------------------------------------
// partial[y][block] = A_y^T Z over the block's rows (ka = 16 TI by kb = 16 TJ,
// BF16 MFMA, FP32 accumulation; y = blockIdx.y picks A0 or A1) and, with
// bpartial and y = 0, the column sums of Z in FP64.  Bound by the operands'
// bytes: the rows are the MFMA's K dimension, and a lane's 8 rows of a 32-row
// step come straight from memory, TI (TJ) consecutive columns per load, so
// that 16 lanes read whole rows; tile t of lane p is then column TI * p + t.
// Blocks of 128-row steps, few enough that their partials stay a small part
// of the traffic.  131,072 rows, 64 x 64: 200 us for one A from operands
// staged and transposed in LDS by 4-byte loads in 128 blocks, 22 us for both
// like this, and 6 us to add the partials up; the column sums took 17 + 121 us
// in kernels of their own.
template <int TI, int TJ>
__global__ void __launch_bounds__(kT) gnn_grad_kernel(const float *A0, const float *A1, const float *Z, uint64_t n,
                                                      uint64_t rows_per_blk, float *partial, double *bpartial)
{
    constexpr int KA = 16 * TI, KB = 16 * TJ, NOUT = KA * KB;
    __shared__ float red[2][NOUT];
    __shared__ double bred[kT / 64][KB];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, p = lane & 15, rg = (lane >> 4) * 8;
    const float *A = blockIdx.y ? A1 : A0;
    const bool bias = bpartial && blockIdx.y == 0;
    floatx4 acc[TI][TJ];
    double bs[TJ];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < TJ; j++) bs[j] = 0.0;
    const uint64_t b0 = blockIdx.x * rows_per_blk, b1 = min(n, b0 + rows_per_blk);
    for (uint64_t r0 = b0 + w * 32; r0 < b1; r0 += 32 * (kT / 64)) {
        FV<TI> a[8];
        FV<TJ> z[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint64_t r = r0 + rg + i, rc = r < b1 ? r : b1 - 1;
            a[i] = *(const FV<TI> *)(A + rc * KA + TI * p);
            z[i] = *(const FV<TJ> *)(Z + rc * KB + TJ * p);
            if (r >= b1) {
#pragma unroll
                for (int t = 0; t < TI; t++) a[i].v[t] = 0.f;
#pragma unroll
                for (int t = 0; t < TJ; t++) z[i].v[t] = 0.f;
            }
        }
        if (bias)
#pragma unroll
            for (int i = 0; i < 8; i++)
#pragma unroll
                for (int t = 0; t < TJ; t++) bs[t] += (double)z[i].v[t];
        bf16x8 zb[TJ];
#pragma unroll
        for (int t = 0; t < TJ; t++)
#pragma unroll
            for (int i = 0; i < 8; i++) zb[t][i] = (__bf16)z[i].v[t];
#pragma unroll
        for (int ti = 0; ti < TI; ti++) {
            bf16x8 ab;
#pragma unroll
            for (int i = 0; i < 8; i++) ab[i] = (__bf16)a[i].v[ti];
#pragma unroll
            for (int tj = 0; tj < TJ; tj++)
                acc[ti][tj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ab, zb[tj], acc[ti][tj], 0, 0, 0);
        }
    }
    // the block's four waves combine as (w0 + w2) + (w1 + w3)
    auto each = [&](auto fn) {
#pragma unroll
        for (int ti = 0; ti < TI; ti++)
#pragma unroll
            for (int tj = 0; tj < TJ; tj++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    fn(acc[ti][tj][q], (TI * ((lane >> 4) * 4 + q) + ti) * KB + TJ * p + tj);
    };
    if (w >= 2) each([&](float v, int o) { red[w - 2][o] = v; });
    if (bias) {
#pragma unroll
        for (int t = 0; t < TJ; t++) {
            bs[t] += __shfl_xor(bs[t], 16, 64);
            bs[t] += __shfl_xor(bs[t], 32, 64);
            if (lane < 16) bred[w][TJ * p + t] = bs[t];
        }
    }
    __syncthreads();
    if (w < 2) {
#pragma unroll
        for (int ti = 0; ti < TI; ti++)
#pragma unroll
            for (int tj = 0; tj < TJ; tj++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int o = (TI * ((lane >> 4) * 4 + q) + ti) * KB + TJ * p + tj;
                    acc[ti][tj][q] += red[w][o];
                    if (w == 1) red[1][o] = acc[ti][tj][q];
                }
    }
    __syncthreads();
    if (w == 0) {
        float *out = partial + ((uint64_t)blockIdx.y * gridDim.x + blockIdx.x) * NOUT;
        each([&](float v, int o) { out[o] = v + red[1][o]; });
    }
    if (bias && threadIdx.x < KB) {
        double t = 0.0;
        for (int q = 0; q < kT / 64; q++) t += bred[q][threadIdx.x];
        bpartial[(uint64_t)blockIdx.x * KB + threadIdx.x] = t;
    }
}

// out[o] = the sum of nblk partials of output o, in FP64: 16 interleaved
// segments (q, q + 16, ...), each in block order, then the segments in order.
// Outputs 0 .. na - 1 are pa's (FP32), the nb behind them pb's (FP64).
template <int SEG>
__device__ __forceinline__ double seg_sum(double mine, double *red)
{
    red[threadIdx.x] = mine;
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x < kT / SEG)
        for (int q = 0; q < SEG; q++) t += red[q * (kT / SEG) + threadIdx.x];
    return t;
}

__global__ void __launch_bounds__(kT) gnn_grad_reduce(const float *pa, int ny, int nout, const double *pb, int nb,
                                                      int nblk, float *out)
{
    __shared__ double red[kT];
    const int o = blockIdx.x * 16 + (threadIdx.x & 15), sg = threadIdx.x >> 4;
    double s = 0.0;
    if (o < ny * nout) {
        const float *p = pa + (uint64_t)(o / nout) * nblk * nout + o % nout;
        for (int b = sg; b < nblk; b += 16) s += (double)p[(uint64_t)b * nout];
    } else if (o < ny * nout + nb) {
        for (int b = sg; b < nblk; b += 16) s += pb[(uint64_t)b * nb + (o - ny * nout)];
    }
    const double t = seg_sum<16>(s, red);
    if (threadIdx.x < 16 && o < ny * nout + nb) out[o] = (float)t;
}

__global__ void __launch_bounds__(kT) colsum_kernel(const float *A, uint64_t n, int k, uint64_t rpb,
                                                    double *partial)
{
    const int per = kT / k;
    const int c = threadIdx.x % k, rr = threadIdx.x / k;
    double s = 0.0;
    if (rr < per) {
        const uint64_t r0 = blockIdx.x * rpb, r1 = min(n, r0 + rpb);
        for (uint64_t r = r0 + rr; r < r1; r += per) s += (double)A[r * k + c];
    }
    __shared__ double red[kT];
    red[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x < k) {
        double t = 0.0;
        for (int q = 0; q < per; q++) t += red[q * k + threadIdx.x];
        partial[(uint64_t)blockIdx.x * k + threadIdx.x] = t;
    }
}

__global__ void __launch_bounds__(kT) f64_to_f32(const double *a, float *b, int n)
{
    for (int i = blockIdx.x * kT + threadIdx.x; i < n; i += gridDim.x * kT) b[i] = (float)a[i];
}

__global__ void __launch_bounds__(kT) adam_kernel(uint64_t np, float *p, const float *g, float *m, float *v,
                                                  float lr, float b1, float b2, float eps, float c1, float c2)
{
    for (uint64_t i = blockIdx.x * (uint64_t)kT + threadIdx.x; i < np; i += (uint64_t)gridDim.x * kT) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.f - b1) * gi;
        const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    }
}

// X0[v] = [log(1 + deg_v), 8 x uniform[-1, 1), 7 x 0]
__global__ void __launch_bounds__(kT) features_kernel(const float *deg, uint64_t n, uint64_t seed, float *X0)
{
    for (uint64_t e = blockIdx.x * (uint64_t)kT + threadIdx.x; e < n * kIn; e += (uint64_t)gridDim.x * kT) {
        const uint64_t v = e / kIn;
        const int j = (int)(e - v * kIn);
        float x = 0.f;
        if (j == 0) {
            x = logf(1.f + deg[v]);
        } else if (j <= 8) {
            uint64_t z = seed + (v * 8 + j) * 0x9E3779B97F4A7C15ULL;
            z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
            z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
            z ^= z >> 31;
            x = (float)((double)(z >> 11) * (1.0 / 9007199254740992.0) * 2.0 - 1.0);
        }
        X0[e] = x;
    }
}

uint32_t grid_n(fmx_ctx *ctx, uint64_t work)
{
    uint64_t b = (work + kT - 1) / kT;
    uint64_t cap = (uint64_t)ctx->num_cus * 16;
    return (uint32_t)(b < 1 ? 1 : (b > cap ? cap : b));
}

// [A1 | A2] B with the epilogue; dout is 16 or 64, d1 and d2 multiples of 16.
fmx_status gemm(fmx_ctx *ctx, int mode, const float *A1, int d1, const float *A2, int d2, const float *W, int wtrans,
                int dout, const Epilogue &ep, uint64_t n, hipStream_t s)
{
    if (!n) return FMX_OK;
    const int K = d1 + d2;
    if (mode != 0) {
        const uint32_t grid = (uint32_t)std::min<uint64_t>((n + 31) / 32, (uint64_t)ctx->num_cus * 8);
        hipLaunchKernelGGL(gnn_f32_kernel, dim3(grid), dim3(kT), 0, s, A1, d1, A2, d2, W, wtrans, dout, ep, n);
        FMX_HIP(ctx, hipGetLastError());
        return FMX_OK;
    }
    // at most four blocks per CU: a wave's B then serves several row tiles
    const uint32_t grid = (uint32_t)std::min<uint64_t>((n + 63) / 64, (uint64_t)ctx->num_cus * 4);
#define FMX_GNN(KS, NT)                                                                                        \
    hipLaunchKernelGGL((gnn_mfma_kernel<KS, NT>), dim3(grid), dim3(kT), 0, s, A1, d1, A2, d2, W, wtrans, ep, n)
    if (dout == 64) {
        if (K <= 32) FMX_GNN(1, 4);
        else if (K <= 64) FMX_GNN(2, 4);
        else FMX_GNN(4, 4);
    } else {
        if (K <= 32) FMX_GNN(1, 1);
        else if (K <= 64) FMX_GNN(2, 1);
        else FMX_GNN(4, 1);
    }
#undef FMX_GNN
    FMX_HIP(ctx, hipGetLastError());
    return FMX_OK;
}

// out = N X for d columns, XS being X with its rows scaled already; the sums
// are rounded before and after the outer scaling
fmx_status norm_agg(fmx_ctx *ctx, const fmx_spm *spm, const double *dinv, const float *XS, int d, float *out,
                    hipStream_t s)
{
    return spmm_exec(ctx, spm, FMX_F32, d, nullptr, dinv, XS, d, out, d, 0, false, s, true);
}

// out (FP32) = A0^T Z, then A1^T Z, then (bias) the column sums of Z; A0 and
// A1 (or NULL) are n x ka, Z n x kb.
fmx_status grads(fmx_ctx *ctx, int mode, uint64_t n, int ka, int kb, const float *A0, const float *A1, const float *Z,
                 bool bias, float *out, hipStream_t s)
{
    const int nout = ka * kb, ny = A1 ? 2 : 1, nb = bias ? kb : 0;
    if (mode != 0) {
        double *g64 = nullptr, *part = nullptr;
        const uint32_t nblk = 512;
        FMX_HIP(ctx, dev_malloc(ctx, (void **)&g64, ((size_t)nout + (size_t)nblk * kHid) * sizeof(double)));
        part = g64 + nout;
        fmx_status st = FMX_OK;
        for (int y = 0; y < ny && !st; y++) {
            st = gram(ctx, FMX_F32, FMX_GRAM_F64, n, ka, kb, y ? A1 : A0, ka, Z, kb, g64, s);
            if (st) break;
            hipLaunchKernelGGL(f64_to_f32, dim3(16), dim3(kT), 0, s, g64, out + y * nout, nout);
        }
        if (!st && bias) {
            hipLaunchKernelGGL(colsum_kernel, dim3(nblk), dim3(kT), 0, s, Z, n, kb, (n + nblk - 1) / nblk, part);
            hipLaunchKernelGGL(gnn_grad_reduce, dim3((nb + 15) / 16), dim3(kT), 0, s, nullptr, 0, nout, part, nb,
                               (int)nblk, out + ny * nout);
        }
        if (!st && hipGetLastError() != hipSuccess) st = fail(ctx, FMX_EHIP, "gradient launch");
        (void)hipStreamSynchronize(s);
        (void)hipFree(g64);
        return st;
    }
    // 256 blocks, more where the rows' bytes dwarf the partials'
    const uint64_t blocks = std::min<uint64_t>((n + 127) / 128, std::max<uint64_t>(256, std::min<uint64_t>(n / 2048, 1024)));
    const uint64_t rpb = blocks ? ((n + blocks - 1) / blocks + 127) / 128 * 128 : 128;
    const uint32_t nblk = (uint32_t)std::max<uint64_t>(1, (n + rpb - 1) / rpb);
    const size_t fb = (size_t)ny * nblk * nout * sizeof(float);
    StreamScratch::Lease ws;
    fmx_status st = ctx_scratch(ctx, s, fb + (size_t)nblk * kb * sizeof(double), ws);
    if (st) return st;
    float *pa = (float *)ws.ptr;
    double *pb = bias ? (double *)((char *)ws.ptr + fb) : nullptr;
#define FMX_GRAD(TI, TJ)                                                                                       \
    hipLaunchKernelGGL((gnn_grad_kernel<TI, TJ>), dim3(nblk, ny), dim3(kT), 0, s, A0, A1, Z, n, rpb, pa, pb)
    if (kb == 64) {
        if (ka == 64) FMX_GRAD(4, 4);
        else FMX_GRAD(1, 4);
    } else {
        FMX_GRAD(4, 1);
    }
#undef FMX_GRAD
    FMX_HIP(ctx, hipGetLastError());
    hipLaunchKernelGGL(gnn_grad_reduce, dim3((ny * nout + nb + 15) / 16), dim3(kT), 0, s, pa, ny, nout, pb, nb,
                       (int)nblk, out);
    FMX_HIP(ctx, hipGetLastError());
    return FMX_OK;
}

}  // namespace
}  // namespace fmx

using namespace fmx;

extern "C" {

uint64_t fmx_gnn_param_count(void) { return layer_off(kLayers) + (uint64_t)kHid * kOut; }
uint64_t fmx_gnn_acts_floats(uint64_t n) { return n * (uint64_t)(kIn + 5 * kHid); }
uint64_t fmx_gnn_work_floats(uint64_t n) { return n * (uint64_t)(4 * kHid); }

fmx_status fmx_gnn_features(fmx_ctx *ctx, const fmx_spm *spm, uint64_t seed, float *X0, double *dinv,
                            void *stream)
{
    if (!ctx || !spm || !X0 || !dinv) return fail(ctx, FMX_EINVAL, "null argument");
    FMX_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = (hipStream_t)stream;
    const uint64_t n = spm->nrows;
    float *ones = nullptr, *deg = nullptr;
    FMX_HIP(ctx, dev_malloc(ctx, (void **)&ones, n * sizeof(float)));
    FMX_HIP(ctx, dev_malloc(ctx, (void **)&deg, n * sizeof(float)));
    std::vector<float> h1(n, 1.0f);
    fmx_status st = FMX_OK;
    if (hipMemcpyAsync(ones, h1.data(), n * 4, hipMemcpyHostToDevice, s) != hipSuccess) st = FMX_EHIP;
    if (!st) st = fmx_spmm(ctx, spm, FMX_F32, 1, ones, 1, deg, 1, s);
    if (!st) st = degree_inv_sqrt(ctx, deg, n, dinv, s);
    if (!st) {
        hipLaunchKernelGGL(features_kernel, dim3(grid_n(ctx, n * kIn)), dim3(kT), 0, s, deg, n, seed, X0);
        if (hipGetLastError() != hipSuccess) st = FMX_EHIP;
    }
    (void)hipStreamSynchronize(s);
    (void)hipFree(ones);
    (void)hipFree(deg);
    return st;
}

fmx_status fmx_gnn_forward(fmx_ctx *ctx, const fmx_spm *spm, const double *dinv, const float *P,
                           const float *X0, float *acts, float *Y, float *work, int mode, void *stream)
{
    if (!ctx || !spm || !dinv || !P || !X0 || !acts || !Y || !work) return fail(ctx, FMX_EINVAL, "null argument");
    if (mode != 0 && mode != 1) return fail(ctx, FMX_EINVAL, "mode is 0 (BF16 MFMA) or 1 (FP32)");
    FMX_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = (hipStream_t)stream;
    const uint64_t n = spm->nrows;
    const float *H = X0;
    float *a = acts, *T = work;  // T: the next aggregation's operand, D^-1/2 H
    fmx_status st = row_scale(ctx, FMX_F32, n, kIn, dinv, X0, kIn, T, kIn, s);
    for (int l = 0; l < kLayers && !st; l++) {
        const int d = din_of(l);
        float *Agg = a;
        a += n * d;
        float *Hn = a;
        a += n * kHid;
        st = norm_agg(ctx, spm, dinv, T, d, Agg, s);
        if (st) return st;
        const float *Wl = P + layer_off(l);
        Epilogue ep;
        ep.bias = Wl + 2 * (size_t)d * kHid;
        ep.relu = 1;
        ep.out = Hn;
        if (l + 1 < kLayers) {
            ep.scale = dinv;
            ep.outs = T;
        }
        st = gemm(ctx, mode, H, d, Agg, d, Wl, 0, kHid, ep, n, s);
        H = Hn;
    }
    if (st) return st;
    Epilogue ep;
    ep.out = Y;
    return gemm(ctx, mode, H, kHid, nullptr, 0, P + layer_off(kLayers), 0, kOut, ep, n, s);
}

fmx_status fmx_gnn_backward(fmx_ctx *ctx, const fmx_spm *spm, const double *dinv, const float *P,
                            const float *X0, const float *acts, const float *dY, float *G, float *work, int mode,
                            void *stream)
{
    if (!ctx || !spm || !dinv || !P || !X0 || !acts || !dY || !G || !work) return fail(ctx, FMX_EINVAL, "null argument");
    if (mode != 0 && mode != 1) return fail(ctx, FMX_EINVAL, "mode is 0 (BF16 MFMA) or 1 (FP32)");
    FMX_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = (hipStream_t)stream;
    const uint64_t n = spm->nrows;
    // activations: per layer Agg_l (n x din), H_{l+1} (n x 64)
    const float *Agg[kLayers], *Hs[kLayers + 1];
    Hs[0] = X0;
    const float *a = acts;
    for (int l = 0; l < kLayers; l++) {
        Agg[l] = a;
        a += n * din_of(l);
        Hs[l + 1] = a;
        a += n * kHid;
    }
    float *dZ = work, *next = work + n * kHid, *T2 = work + 2 * n * kHid, *T3 = work + 3 * n * kHid;
    const float *Wo = P + layer_off(kLayers);
    fmx_status st = grads(ctx, mode, n, kHid, kOut, Hs[kLayers], nullptr, dY, false, G + layer_off(kLayers), s);
    {
        // dZ_3 = (dY Wo^T) where H_3 > 0  (Wo is 64 x 16 = dout x K)
        Epilogue ep;
        ep.gate = Hs[kLayers];
        ep.out = dZ;
        if (!st) st = gemm(ctx, mode, dY, kOut, nullptr, 0, Wo, 1, kHid, ep, n, s);
    }
    for (int l = kLayers - 1; l >= 0 && !st; l--) {
        const int d = din_of(l);
        const float *Wl = P + layer_off(l);
        st = grads(ctx, mode, n, d, kHid, Hs[l], Agg[l], dZ, true, G + layer_off(l), s);
        if (st || l == 0) break;
        // dZ_l = (dZ Ws^T + N (dZ Wn^T)) where H_l > 0; Ws, Wn are d x 64 = dout x K
        Epilogue ea;
        ea.scale = dinv;
        ea.outs = T2;
        st = gemm(ctx, mode, dZ, kHid, nullptr, 0, Wl + (size_t)d * kHid, 1, d, ea, n, s);
        if (!st) st = norm_agg(ctx, spm, dinv, T2, d, T3, s);
        Epilogue eb;
        eb.add = T3;
        eb.gate = Hs[l];
        eb.out = next;
        if (!st) st = gemm(ctx, mode, dZ, kHid, nullptr, 0, Wl, 1, d, eb, n, s);
        std::swap(dZ, next);
    }
    if (hipStreamSynchronize(s) != hipSuccess && !st) st = FMX_EHIP;
    return st ? fail(ctx, st, "gnn backward failed") : FMX_OK;
}

fmx_status fmx_subspace_loss(fmx_ctx *ctx, uint64_t n, int k, const float *Y, const float *U, double *loss,
                             float *dY, void *stream)
{
    if (!ctx || !Y || !U || !loss || k <= 0 || k > 64) return fail(ctx, FMX_EINVAL, "bad argument");
    FMX_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t s = (hipStream_t)stream;
    double *dG = nullptr, *dC = nullptr, *dM = nullptr;
    FMX_HIP(ctx, dev_malloc(ctx, (void **)&dG, (size_t)k * k * sizeof(double)));
    FMX_HIP(ctx, dev_malloc(ctx, (void **)&dC, (size_t)k * k * sizeof(double)));
    FMX_HIP(ctx, dev_malloc(ctx, (void **)&dM, 2 * (size_t)k * k * sizeof(double)));
    std::vector<double> G(k * k), C(k * k), Gi(k * k), B(k * k), M1(k * k), M2(k * k), T(k * k);
    fmx_status st = gram(ctx, FMX_F32, FMX_GRAM_F64, n, k, k, Y, k, Y, k, dG, s);
    if (!st) st = gram(ctx, FMX_F32, FMX_GRAM_F64, n, k, k, U, k, Y, k, dC, s);
    if (!st && hipMemcpyAsync(G.data(), dG, k * k * 8, hipMemcpyDeviceToHost, s) != hipSuccess) st = FMX_EHIP;
    if (!st && hipMemcpyAsync(C.data(), dC, k * k * 8, hipMemcpyDeviceToHost, s) != hipSuccess) st = FMX_EHIP;
    if (!st && hipStreamSynchronize(s) != hipSuccess) st = FMX_EHIP;
    if (!st) {
        // Gi = G^-1 (Gauss-Jordan, partial pivoting; k x k on the host)
        std::vector<double> M(2 * k * k);
        for (int i = 0; i < k; i++)
            for (int j = 0; j < 2 * k; j++) M[i * 2 * k + j] = j < k ? G[i * k + j] : (j - k == i);
        for (int c = 0; c < k && !st; c++) {
            int p = c;
            for (int r = c + 1; r < k; r++) if (fabs(M[r * 2 * k + c]) > fabs(M[p * 2 * k + c])) p = r;
            if (M[p * 2 * k + c] == 0.0) { st = fail(ctx, FMX_EINVAL, "Y has rank < k"); break; }
            for (int j = 0; j < 2 * k; j++) std::swap(M[c * 2 * k + j], M[p * 2 * k + j]);
            const double dv = M[c * 2 * k + c];
            for (int j = 0; j < 2 * k; j++) M[c * 2 * k + j] /= dv;
            for (int r = 0; r < k; r++) {
                if (r == c) continue;
                const double f = M[r * 2 * k + c];
                if (f != 0.0) for (int j = 0; j < 2 * k; j++) M[r * 2 * k + j] -= f * M[c * 2 * k + j];
            }
        }
        if (!st) {
            for (int i = 0; i < k; i++) for (int j = 0; j < k; j++) Gi[i * k + j] = M[i * 2 * k + k + j];
            for (int i = 0; i < k; i++) for (int j = 0; j < k; j++) {
                double v = 0; for (int t = 0; t < k; t++) v += C[t * k + i] * C[t * k + j];
                B[i * k + j] = v;
            }
            double tr = 0;
            for (int i = 0; i < k; i++) for (int j = 0; j < k; j++) tr += Gi[i * k + j] * B[j * k + i];
            *loss = k - tr;
            for (int i = 0; i < k; i++) for (int j = 0; j < k; j++) {
                double a1 = 0, a2 = 0;
                for (int t = 0; t < k; t++) { a1 += C[i * k + t] * Gi[t * k + j]; a2 += Gi[i * k + t] * B[t * k + j]; }
                M1[i * k + j] = a1;
                T[i * k + j] = a2;
            }
            for (int i = 0; i < k; i++) for (int j = 0; j < k; j++) {
                double v = 0; for (int t = 0; t < k; t++) v += T[i * k + t] * Gi[t * k + j];
                M2[i * k + j] = v;
            }
        }
    }
    if (!st && dY) {
        if (hipMemcpyAsync(dM, M1.data(), k * k * 8, hipMemcpyHostToDevice, s) != hipSuccess ||
            hipMemcpyAsync(dM + k * k, M2.data(), k * k * 8, hipMemcpyHostToDevice, s) != hipSuccess)
            st = FMX_EHIP;
        if (!st) st = gemm_tall(ctx, FMX_F32, n, k, k, -2.0, U, k, dM, 0.0, dY, k, s);
        if (!st) st = gemm_tall(ctx, FMX_F32, n, k, k, 2.0, Y, k, dM + k * k, 1.0, dY, k, s);
    }
    (void)hipStreamSynchronize(s);
    (void)hipFree(dG);
    (void)hipFree(dC);
    (void)hipFree(dM);
    return st;
}

fmx_status fmx_adam(fmx_ctx *ctx, uint64_t np, float *params, const float *grads, float *m, float *v, float lr,
                    float beta1, float beta2, float eps, int step, void *stream)
{
    if (!ctx || !params || !grads || !m || !v || step < 1) return fail(ctx, FMX_EINVAL, "bad argument");
    FMX_HIP(ctx, hipSetDevice(ctx->device));
    const float c1 = 1.f - powf(beta1, (float)step), c2 = 1.f - powf(beta2, (float)step);
    hipLaunchKernelGGL(adam_kernel, dim3(grid_n(ctx, np)), dim3(kT), 0, (hipStream_t)stream, np, params, grads, m,
                       v, lr, beta1, beta2, eps, c1, c2);
    FMX_HIP(ctx, hipGetLastError());
    return FMX_OK;
}

}  // extern "C"
