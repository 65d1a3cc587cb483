// devprim.hip -- hand-written device primitives for tile construction.
//
//   * scan_exclusive: tile reduce -> recursive scan of tile sums -> tile scan
//     (4096 values per 256-thread block, wave scans by DPP-free shuffles);
//   * radix_sort_u64: stable LSD radix sort, 8-bit digits; per pass a digit
//     histogram per tile of keys, an exclusive scan of each digit's counts
//     over the tiles, and a scatter that ranks equal digits inside each wave
//     with ballots (so equal keys keep their order: the sort is stable);
//   * max_u32_pair: max of two id arrays.
#include "devprim.h"

namespace fmx {
namespace {

constexpr int kT = 256;          // threads per block
constexpr int kI = 16;           // items per thread
constexpr int kTile = kT * kI;   // 4096

template <typename T>
__device__ __forceinline__ T shfl_up_t(T v, int d)
{
    if constexpr (sizeof(T) == 8) {
        uint32_t lo = (uint32_t)v, hi = (uint32_t)((uint64_t)v >> 32);
        lo = __shfl_up(lo, d, 64);
        hi = __shfl_up(hi, d, 64);
        return (T)(((uint64_t)hi << 32) | lo);
    } else {
        return (T)__shfl_up((uint32_t)v, d, 64);
    }
}

// Exclusive scan of one value per thread over the block; returns the block total.
template <typename T, int NT = kT>
__device__ __forceinline__ T block_exclusive(T v, T *lds_waves, T &total)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    T inc = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        T o = shfl_up_t(inc, d);
        if (lane >= d) inc += o;
    }
    if (lane == 63) lds_waves[w] = inc;
    __syncthreads();
    T off = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < NT / 64; i++) {
        T x = lds_waves[i];
        if (i < w) off += x;
        tot += x;
    }
    __syncthreads();
    total = tot;
    return off + inc - v;
}

template <typename T>
__global__ void __launch_bounds__(kT) scan_reduce(const T *in, uint64_t n, T *partials)
{
    __shared__ T wl[kT / 64];
    const uint64_t base = (uint64_t)blockIdx.x * kTile;
    T s = 0;
#pragma unroll
    for (int i = 0; i < kI; i++) {
        uint64_t idx = base + (uint64_t)i * kT + threadIdx.x;
        if (idx < n) s += in[idx];
    }
    T tot;
    (void)block_exclusive(s, wl, tot);
    if (threadIdx.x == 0) partials[blockIdx.x] = tot;
}

template <typename T>
__global__ void __launch_bounds__(kT) scan_tile(const T *in, T *out, uint64_t n, const T *carries,
                                                 T *d_total)
{
    __shared__ T wl[kT / 64];
    const uint64_t base = (uint64_t)blockIdx.x * kTile + (uint64_t)threadIdx.x * kI;
    T v[kI];
    T s = 0;
    // a thread's 16 values as 16-byte words where they are whole and aligned
    // (every caller's arrays are; a tile's start is): the
    // scans of counts and flags of a 16.8 M edge build 430 -> 168 us
    constexpr int kV = 16 / sizeof(T);
    const bool whole = base + kI <= n && (((uintptr_t)in | (uintptr_t)out) & 15) == 0;
    if (whole) {
#pragma unroll
        for (int i = 0; i < kI; i += kV) {
            const uint4 q = *(const uint4 *)(in + base + i);
            __builtin_memcpy(v + i, &q, 16);
        }
    } else {
#pragma unroll
        for (int i = 0; i < kI; i++) v[i] = base + i < n ? in[base + i] : T(0);
    }
#pragma unroll
    for (int i = 0; i < kI; i++) s += v[i];
    T tot;
    T run = block_exclusive(s, wl, tot);
    if (carries) run += carries[blockIdx.x];
#pragma unroll
    for (int i = 0; i < kI; i++) {
        const T x = v[i];
        v[i] = run;
        run += x;
    }
    if (whole) {
#pragma unroll
        for (int i = 0; i < kI; i += kV) {
            uint4 q;
            __builtin_memcpy(&q, v + i, 16);
            *(uint4 *)(out + base + i) = q;
        }
    } else {
#pragma unroll
        for (int i = 0; i < kI; i++)
            if (base + i < n) out[base + i] = v[i];
    }
    if (d_total && threadIdx.x == 0) *d_total = tot;
}

template <typename T>
fmx_status scan_rec(fmx_ctx *ctx, const T *in, T *out, uint64_t n, T *d_total, hipStream_t s)
{
    const uint64_t nb = (n + kTile - 1) / kTile;
    if (nb <= 1) {
        hipLaunchKernelGGL(scan_tile<T>, dim3(1), dim3(kT), 0, s, in, out, n, (const T *)nullptr,
                           d_total);
        FMX_HIP(ctx, hipGetLastError());
        return FMX_OK;
    }
    DevBuf<T> partials;
    FMX_HIP(ctx, partials.alloc(ctx, nb));
    hipLaunchKernelGGL(scan_reduce<T>, dim3((uint32_t)nb), dim3(kT), 0, s, in, n, partials.p);
    FMX_HIP(ctx, hipGetLastError());
    fmx_status st = scan_rec<T>(ctx, partials.p, partials.p, nb, d_total, s);
    if (st) return st;
    hipLaunchKernelGGL(scan_tile<T>, dim3((uint32_t)nb), dim3(kT), 0, s, in, out, n,
                       (const T *)partials.p, (T *)nullptr);
    FMX_HIP(ctx, hipGetLastError());
    // outside a construction the partials are freed at once: after the kernels
    if (!ctx->blocks.scopes) FMX_HIP(ctx, hipStreamSynchronize(s));
    return FMX_OK;
}

// ---- radix sort -------------------------------------------------------------
// A pass reads the keys twice and writes them once; it is bound by that and,
// for short lists, by its launches.  Tiles of 8192 keys (512 threads; 4096
// keys and 256 threads with a payload, whose LDS would leave one block per CU
// otherwise): twice the keys of a digit lie together in the output, and the
// histogram is half as long.  One block scans a digit's counts over all tiles,
// and each tile adds the digits before its own itself, so a pass is three
// launches.  A pass over 16.8 M keys: count 28 us, scan 5, scatter 56 (4.8 TB/s);
// with 4096-key tiles, digits counted by LDS atomics a second time and the
// general scan over the whole histogram 32, 30 and 79.
constexpr int kChunks = 16;                            // 64-key chunks per wave
template <bool KV>
constexpr int kSortT = KV ? 256 : 512;                 // threads per tile
template <bool KV>
constexpr int kSortTile = kSortT<KV> / 64 * kChunks * 64;

template <bool KV>
__global__ void __launch_bounds__(kSortT<KV>) rs_count(const uint64_t *keys, uint64_t n, int shift,
                                                       uint64_t *hist, uint32_t nb)
{
    __shared__ uint32_t cnt[256];
    if (threadIdx.x < 256) cnt[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t base = (uint64_t)blockIdx.x * kSortTile<KV>;
#pragma unroll 4
    for (int i = 0; i < kChunks; i++) {
        uint64_t idx = base + (uint64_t)i * kSortT<KV> + threadIdx.x;
        if (idx < n) atomicAdd(&cnt[(keys[idx] >> shift) & 0xFF], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 256) hist[(uint64_t)threadIdx.x * nb + blockIdx.x] = cnt[threadIdx.x];
}

// Block d: the exclusive scan of digit d's counts over the nb tiles, in
// place, and their sum.
constexpr int kScanT = 1024;
__global__ void __launch_bounds__(kScanT) rs_scan(uint64_t *hist, uint32_t nb, uint64_t *total)
{
    __shared__ uint64_t wl[kScanT / 64];
    uint64_t *h = hist + (uint64_t)blockIdx.x * nb;
    uint64_t carry = 0;
    for (uint32_t at = 0; at < nb; at += 4 * kScanT) {
        const uint64_t i0 = (uint64_t)at + 4 * threadIdx.x;
        uint64_t v[4], sum = 0, all;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            v[j] = i0 + j < nb ? h[i0 + j] : 0;
            sum += v[j];
        }
        uint64_t run = carry + block_exclusive<uint64_t, kScanT>(sum, wl, all);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (i0 + j < nb) h[i0 + j] = run;
            run += v[j];
        }
        carry += all;
    }
    if (threadIdx.x == 0) total[blockIdx.x] = carry;
}

// Scatter of one pass; the optional u32 payload (vin -> vout) moves with its
// key.  The tile's keys are first ranked into digit order in LDS (equal
// digits ranked inside each wave with ballots, waves and 64-key chunks in
// order, so equal keys keep their order: the sort is stable), then written
// out in that order, so consecutive threads write consecutive slots of each
// digit's run in the output (coalesced).
template <bool KV>
__global__ void __launch_bounds__(kSortT<KV>) rs_scatter_t(const uint64_t *in, uint64_t *out, const uint32_t *vin,
                                                           uint32_t *vout, uint64_t n, int shift,
                                                           const uint64_t *offs, const uint64_t *total, uint32_t nb)
{
    constexpr int kNT = kSortT<KV>, kWaves = kNT / 64, kKeys = kSortTile<KV>;
    __shared__ uint32_t wcnt[kWaves][256];  // keys of each digit per wave, then their first tile slot
    __shared__ uint32_t dstart[256];        // first tile slot of each digit
    __shared__ uint64_t gstart[256];        // first output slot of this tile's keys of each digit
    __shared__ uint32_t wl[kWaves];
    __shared__ uint64_t wl8[kWaves];
    __shared__ uint64_t sk[kKeys];          // the tile's keys in digit order
    __shared__ uint32_t sv[KV ? kKeys : 1];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < kWaves * 256; i += kNT) (&wcnt[0][0])[i] = 0;
    // wave w owns keys [w*1024, (w+1)*1024) of the tile, 64 at a time, in order
    const uint64_t base = (uint64_t)blockIdx.x * kKeys + (uint64_t)w * (kChunks * 64);
    uint64_t k[kChunks];
    uint32_t pv[KV ? kChunks : 1];
    uint32_t rank[kChunks];  // among the wave's keys of its digit
#pragma unroll
    for (int c = 0; c < kChunks; c++) {
        uint64_t idx = base + (uint64_t)c * 64 + lane;
        k[c] = idx < n ? in[idx] : 0;
        if constexpr (KV) pv[c] = idx < n ? vin[idx] : 0u;
    }
    uint64_t dtot = 0, doff = 0;
    if (threadIdx.x < 256) {
        dtot = total[threadIdx.x];
        doff = offs[(uint64_t)threadIdx.x * nb + blockIdx.x];
    }
    __syncthreads();
    const uint64_t lt = (1ull << lane) - 1ull;
#pragma unroll
    for (int c = 0; c < kChunks; c++) {
        const uint64_t idx = base + (uint64_t)c * 64 + lane;
        const bool valid = idx < n;
        const uint32_t d = (uint32_t)(k[c] >> shift) & 0xFFu;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bm = __ballot(valid && bit);
            peers &= bit ? bm : ~bm;
        }
        const uint32_t before = wcnt[w][d];
        rank[c] = before + __popcll(peers & lt);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (valid && (peers & lt) == 0) wcnt[w][d] = before + __popcll(peers);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    {
        const int d = threadIdx.x;  // one digit per thread
        uint32_t tot = 0, all;
        uint64_t all8;
        if (d < 256) {
#pragma unroll
            for (int ww = 0; ww < kWaves; ww++) tot += wcnt[ww][d];
        }
        uint32_t run = block_exclusive<uint32_t, kNT>(tot, wl, all);
        const uint64_t first = block_exclusive<uint64_t, kNT>(dtot, wl8, all8);
        if (d < 256) {
            dstart[d] = run;
#pragma unroll
            for (int ww = 0; ww < kWaves; ww++) {
                const uint32_t c = wcnt[ww][d];
                wcnt[ww][d] = run;
                run += c;
            }
            gstart[d] = first + doff;
        }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kChunks; c++) {
        if (base + (uint64_t)c * 64 + lane < n) {
            const uint32_t lpos = wcnt[w][(uint32_t)(k[c] >> shift) & 0xFFu] + rank[c];
            sk[lpos] = k[c];
            if constexpr (KV) sv[lpos] = pv[c];
        }
    }
    __syncthreads();
    const uint64_t t0 = (uint64_t)blockIdx.x * kKeys;
    const uint32_t nt = (uint32_t)min((uint64_t)kKeys, n - t0);
    for (uint32_t j = threadIdx.x; j < nt; j += kNT) {
        const uint64_t key = sk[j];
        const uint32_t d = (uint32_t)(key >> shift) & 0xFFu;
        const uint64_t pos = gstart[d] + (j - dstart[d]);
        out[pos] = key;
        if constexpr (KV) vout[pos] = sv[j];
    }
}

template <bool KV>
fmx_status sort_passes(fmx_ctx *ctx, uint64_t *&a, uint64_t *&b, uint32_t *&va, uint32_t *&vb, uint64_t n, int from,
                       int bits, hipStream_t s)
{
    const uint64_t nb64 = (n + kSortTile<KV> - 1) / kSortTile<KV>;
    if (nb64 >= (1ull << 32) / 256) return fail(ctx, FMX_EUNSUPPORTED, "too many keys to sort");
    const uint32_t nb = (uint32_t)nb64;
    DevBuf<uint64_t> hist;
    FMX_HIP(ctx, hist.alloc(ctx, (uint64_t)nb * 256 + 256));
    uint64_t *total = hist.p + (uint64_t)nb * 256;
    for (int shift = from; shift < bits; shift += 8) {
        hipLaunchKernelGGL(rs_count<KV>, dim3(nb), dim3(kSortT<KV>), 0, s, a, n, shift, hist.p, nb);
        hipLaunchKernelGGL(rs_scan, dim3(256), dim3(kScanT), 0, s, hist.p, nb, total);
        hipLaunchKernelGGL(rs_scatter_t<KV>, dim3(nb), dim3(kSortT<KV>), 0, s, a, b, va, vb, n, shift, hist.p, total,
                           nb);
        FMX_HIP(ctx, hipGetLastError());
        std::swap(a, b);
        std::swap(va, vb);
    }
    if (!ctx->blocks.scopes) FMX_HIP(ctx, hipStreamSynchronize(s));
    return FMX_OK;
}

// One atomic per block, and few blocks: atomics on one word pass one by one,
// some 5 ns each (16.8 M pairs: 113 us with one per wave of 2048 blocks; 40 us
// like this).
__global__ void __launch_bounds__(kT) max_pair_kernel(const uint32_t *a, const uint32_t *b,
                                                      uint64_t n, uint32_t *out)
{
    __shared__ uint32_t wm[kT / 64];
    uint32_t m = 0;
    const uint64_t step = (uint64_t)gridDim.x * kT;
    uint64_t i = blockIdx.x * (uint64_t)kT + threadIdx.x;
    for (; i + 3 * step < n; i += 4 * step) {
        uint32_t v[8];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            v[2 * t] = a[i + t * step];
            v[2 * t + 1] = b[i + t * step];
        }
#pragma unroll
        for (int t = 0; t < 8; t++) m = max(m, v[t]);
    }
    for (; i < n; i += step) m = max(m, max(a[i], b[i]));
    for (int d = 32; d; d >>= 1) m = max(m, (uint32_t)__shfl_xor(m, d, 64));
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kT / 64; w++) m = max(m, wm[w]);
        atomicMax(out, m);
    }
}

}  // namespace

template <typename T>
fmx_status scan_exclusive(fmx_ctx *ctx, const T *in, T *out, uint64_t n, T *total, hipStream_t s)
{
    DevBuf<T> d_total;
    FMX_HIP(ctx, d_total.alloc(ctx, 1));
    if (n == 0) {
        if (total) *total = 0;
        return FMX_OK;
    }
    fmx_status st = scan_rec<T>(ctx, in, out, n, d_total.p, s);
    if (st) return st;
    if (total) {
        st = pinned_fetch(ctx, total, d_total.p, sizeof(T), 0, s);
        if (st) return st;
    }
    if (total || !ctx->blocks.scopes) FMX_HIP(ctx, hipStreamSynchronize(s));
    if (total) pinned_get(ctx, total, sizeof(T), 0);
    return FMX_OK;
}

template fmx_status scan_exclusive<uint32_t>(fmx_ctx *, const uint32_t *, uint32_t *, uint64_t,
                                             uint32_t *, hipStream_t);
template fmx_status scan_exclusive<uint64_t>(fmx_ctx *, const uint64_t *, uint64_t *, uint64_t,
                                             uint64_t *, hipStream_t);

fmx_status scan_u64_exclusive(fmx_ctx *ctx, const uint64_t *in, uint64_t *out, uint64_t n, uint64_t *total,
                              hipStream_t s)
{
    return scan_exclusive<uint64_t>(ctx, in, out, n, total, s);
}

fmx_status radix_sort_u64(fmx_ctx *ctx, uint64_t *keys, uint64_t *tmp, uint64_t n, int from, int bits,
                          uint64_t **sorted, hipStream_t s)
{
    uint32_t *dummy = nullptr;
    return radix_sort_u64_kv(ctx, keys, tmp, nullptr, nullptr, n, from, bits, sorted, &dummy, s);
}

fmx_status radix_sort_u64_kv(fmx_ctx *ctx, uint64_t *keys, uint64_t *tmp, uint32_t *vals, uint32_t *vtmp,
                             uint64_t n, int from, int bits, uint64_t **sorted, uint32_t **sorted_vals,
                             hipStream_t s)
{
    *sorted = keys;
    *sorted_vals = vals;
    if (n < 2 || bits <= from) return FMX_OK;
    fmx_status st = vals ? sort_passes<true>(ctx, keys, tmp, vals, vtmp, n, from, bits, s)
                         : sort_passes<false>(ctx, keys, tmp, vals, vtmp, n, from, bits, s);
    if (st) return st;
    *sorted = keys;
    *sorted_vals = vals;
    return FMX_OK;
}

fmx_status max_u32_pair(fmx_ctx *ctx, const uint32_t *a, const uint32_t *b, uint64_t n,
                        uint32_t *out, hipStream_t s)
{
    DevBuf<uint32_t> d;
    FMX_HIP(ctx, d.alloc(ctx, 1));
    FMX_HIP(ctx, hipMemsetAsync(d.p, 0, sizeof(uint32_t), s));
    uint64_t blocks = (n + kT - 1) / kT;
    if (blocks > (uint64_t)ctx->num_cus * 4) blocks = (uint64_t)ctx->num_cus * 4;
    if (blocks == 0) blocks = 1;
    hipLaunchKernelGGL(max_pair_kernel, dim3((uint32_t)blocks), dim3(kT), 0, s, a, b, n, d.p);
    FMX_HIP(ctx, hipGetLastError());
    fmx_status st = pinned_fetch(ctx, out, d.p, sizeof(uint32_t), 0, s);
    if (st) return st;
    FMX_HIP(ctx, hipStreamSynchronize(s));
    pinned_get(ctx, out, sizeof(uint32_t), 0);
    return FMX_OK;
}

}  // namespace fmx
