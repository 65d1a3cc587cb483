// image_dev.hip -- walks of an image resident in HBM, on the device: the
// gather-order relabelling of an uploaded image, the column ranking that a
// device build shares, and the cuts of a device-built image's work plans.
//
// decode_lists: every non-zero as (row, column[, value]) in stream order
// (block rows ascending; in each block row its tiles in directory order; in
// each tile the SCSR rows, then the COO entries):
//   tile_origin   each tile's block row (one thread per block row);
//   tile_count    each tile's non-zero count, from its header;
//   scan          each tile's first output position;
//   decode        one thread per tile walks its words and writes its
//                 non-zeros (and counts each column's uses, atomically, when
//                 asked).
//
// rank_columns: the nhot most used columns become 0..nhot-1 in descending
// order of use (ties by column) and every other column c becomes nhot + c:
//   rank          sort keys ((2^31 - uses) << 32 | column): descending use,
//                 ascending column among equals;
//   cut           the first rank at which the running sum of uses reaches
//                 the wanted share (or the uses reach 0) is nhot;
//   new ids       of all columns, and the list of the hot ones in new order.
// gather_order_lists: decode_lists' lists with the columns relabelled so.
//
// plan_cuts: the split items of a work plan, whose ranges come as fractions
// of their block row, moved to where an item may start (one wave per item:
// a binary search of the directory, then a search back for the row in
// force, 512 words at a time).
#include "devprim.h"

namespace fmx {
namespace {

constexpr int kT = 256;
constexpr uint64_t kMaxUses = 1ull << 31;  // non-zeros of a gather-order image stay below 2^31

// image words are 2-byte aligned (tiles start at even byte offsets)
__device__ __forceinline__ uint32_t ld16(const uint8_t *p) { return *(const uint16_t *)p; }
__device__ __forceinline__ uint32_t ld32(const uint8_t *p) { return ld16(p) | (ld16(p + 2) << 16); }

__global__ void __launch_bounds__(kT) tile_origin(const uint32_t *brow_dir, uint64_t nbr, uint32_t *tbr)
{
    for (uint64_t br = blockIdx.x * (uint64_t)kT + threadIdx.x; br < nbr; br += (uint64_t)gridDim.x * kT)
        for (uint32_t t = brow_dir[br]; t < brow_dir[br + 1]; t++) tbr[t] = (uint32_t)br;
}

__global__ void __launch_bounds__(kT) tile_count(const uint8_t *img, const int64_t *offs, const uint2 *dir,
                                                 const uint32_t *tbr, uint64_t ntiles, uint32_t *tnnz)
{
    for (uint64_t t = blockIdx.x * (uint64_t)kT + threadIdx.x; t < ntiles; t += (uint64_t)gridDim.x * kT)
        tnnz[t] = ld32(img + offs[tbr[t]] + 2ull * dir[t].x + 8);
}

__global__ void __launch_bounds__(kT) decode(const uint8_t *img, const int64_t *offs, const uint2 *dir,
                                             const uint32_t *tbr, const uint32_t *tpos, uint64_t ntiles,
                                             uint64_t H, uint64_t W, uint32_t esz, uint32_t *rows,
                                             uint32_t *cols, uint8_t *vals, uint32_t *uses)
{
    for (uint64_t t = blockIdx.x * (uint64_t)kT + threadIdx.x; t < ntiles; t += (uint64_t)gridDim.x * kT) {
        const uint64_t br = tbr[t];
        const uint8_t *p = img + offs[br] + 2ull * dir[t].x;
        const uint32_t nnz = ld32(p + 8);
        if (!nnz) continue;
        const uint32_t nrow = ld16(p + 12), ncoo = ld16(p + 14);
        const uint32_t scsr_words = (nrow - ncoo) + (nnz - ncoo);
        const uint8_t *w = p + 16, *coo = w + 2ull * scsr_words + 2, *vp = coo + 4ull * ncoo;
        const uint32_t r0 = (uint32_t)(br * H), c0 = (uint32_t)((uint64_t)dir[t].y * W);
        uint64_t o = tpos[t];
        uint32_t e = 0, r = r0;
        auto put = [&](uint32_t row, uint32_t col) {
            rows[o] = row;
            cols[o] = col;
            if (uses) atomicAdd(&uses[col], 1u);
            for (uint32_t b = 0; b < esz; b++) vals[o * esz + b] = vp[(uint64_t)e * esz + b];
            o++;
            e++;
        };
        for (uint32_t i = 0; i < scsr_words; i++) {
            const uint32_t v = ld16(w + 2ull * i);
            if (v & 0x8000u) r = r0 + (v & 0x7FFFu);
            else put(r, c0 + v);
        }
        for (uint32_t i = 0; i < ncoo; i++) put(r0 + (ld16(coo + 4ull * i) & 0x7FFFu), c0 + ld16(coo + 4ull * i + 2));
    }
}

__global__ void __launch_bounds__(kT) rank_keys(const uint32_t *uses, uint64_t ncols, uint64_t *keys)
{
    for (uint64_t c = blockIdx.x * (uint64_t)kT + threadIdx.x; c < ncols; c += (uint64_t)gridDim.x * kT)
        keys[c] = ((kMaxUses - uses[c]) << 32) | c;
}

__global__ void __launch_bounds__(kT) ranked_uses(const uint64_t *keys, uint64_t ncols, uint64_t *u, uint64_t *nhot)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) *nhot = ncols;  // what cut leaves if every rank is hot
    for (uint64_t i = blockIdx.x * (uint64_t)kT + threadIdx.x; i < ncols; i += (uint64_t)gridDim.x * kT)
        u[i] = kMaxUses - (keys[i] >> 32);
}

// Rank i is hot while the uses before it fall short of the share and it has
// uses itself; both conditions hold on a prefix of the ranks, so nhot is the
// first rank that fails (ncols if none does): the one rank that fails while
// its predecessor passes writes it.
__global__ void __launch_bounds__(kT) cut(const uint64_t *keys, const uint64_t *before, uint64_t ncols,
                                          uint64_t target_permille, uint64_t *nhot)
{
    auto hot = [&](uint64_t i) { return before[i] * 1000 < target_permille && (keys[i] >> 32) < kMaxUses; };
    for (uint64_t i = blockIdx.x * (uint64_t)kT + threadIdx.x; i < ncols; i += (uint64_t)gridDim.x * kT)
        if (!hot(i) && (i == 0 || hot(i - 1))) *nhot = i;
}

__global__ void __launch_bounds__(kT) new_ids(uint64_t ncols, uint64_t nhot, uint32_t *newid)
{
    for (uint64_t c = blockIdx.x * (uint64_t)kT + threadIdx.x; c < ncols; c += (uint64_t)gridDim.x * kT)
        newid[c] = (uint32_t)(nhot + c);
}

__global__ void __launch_bounds__(kT) hot_ids(const uint64_t *keys, uint64_t nhot, uint32_t *newid, uint32_t *hot)
{
    for (uint64_t i = blockIdx.x * (uint64_t)kT + threadIdx.x; i < nhot; i += (uint64_t)gridDim.x * kT) {
        const uint32_t c = (uint32_t)(keys[i] & 0xFFFFFFFFu);
        newid[c] = (uint32_t)i;
        hot[i] = c;
    }
}

__global__ void __launch_bounds__(kT) relabel(uint32_t *cols, uint64_t nnz, const uint32_t *newid)
{
    for (uint64_t e = blockIdx.x * (uint64_t)kT + threadIdx.x; e < nnz; e += (uint64_t)gridDim.x * kT)
        cols[e] = newid[cols[e]];
}

// The last tile of the block row whose entries are dir[lo, hi) that starts at
// or before word p (the first starts at word 0).
__device__ __forceinline__ uint32_t tile_before(const uint2 *dir, uint32_t lo, uint32_t hi, uint32_t p)
{
    while (hi - lo > 1) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (dir[mid].x <= p) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Split items (slot != kNone) of a plan: item words [begin, begin + nwords)
// of a block row of rot_begin words, dir_begin its first directory entry.
// Both ends move the same way, so neighbouring items still meet: out of the
// header of the tile they fall in (binary), or to the same fraction of its
// entries' words as they have of the whole tile (weighted: the values behind
// them are only read by their entries).  A weighted item also gets the number
// of its tile's entries before it, the place of its first value.  The row
// in force at an item's first word, kNone if that word is a header
// (row part or COO entry), is that of the nearest header before it: the
// lanes read 512 words back at a time and a ballot finds it (a hub row's part
// can be 32768 words long, and 64 words a step made this the longest part of
// a plan; the word behind the tile header always has the header bit, so the
// search ends inside the tile).
__global__ void __launch_bounds__(kT) fix_items(const uint16_t *img, const uint2 *dir, const uint32_t *vdir,
                                                Item *items, uint32_t n, uint32_t *bad)
{
    const int lane = threadIdx.x & 63;
    const uint32_t i = blockIdx.x * (kT / 64) + (threadIdx.x >> 6);
    if (i >= n) return;
    const Item t = items[i];
    if (t.slot == kNone) return;
    const uint32_t words = t.rot_begin, d0 = t.dir_begin, d1 = t.dir_end;
    uint32_t end[2], tile = d0, inside = 0;  // words of the tile's entries before the item
    for (int e = 0; e < 2; e++) {
        uint32_t p = e ? t.begin + t.nwords : t.begin;
        if (p != 0 && p < words) {
            const uint32_t at = tile_before(dir, d0, d1, p), x = dir[at].x;
            if (vdir) {
                const uint32_t next = at + 1 < d1 ? dir[at + 1].x : words;
                p = x + 8 + (uint32_t)((uint64_t)(p - x) * (vdir[at] - x - 8) / (next - x));
            } else {
                p = max(p, x + 8);
            }
            if (e == 0) {
                tile = at;
                inside = p - (x + 8);
            }
        }
        end[e] = p;
    }
    uint32_t carry = kNone, before = 0;
    if (vdir && inside) {
        // the entries among the `inside` words before the item
        const uint64_t stop = t.brow_word + end[0], start = stop - inside;
#pragma unroll 4
        for (uint64_t g = (start & ~7ull) + lane * 8; g < stop; g += 512) {
            const uint4 v = *(const uint4 *)(img + g);
            const uint32_t x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const uint32_t word = x[j >> 1] >> ((j & 1) * 16);
                before += g + j >= start && g + j < stop && !(word & 0x8000u);
            }
        }
        for (int d = 32; d; d >>= 1) before += __shfl_xor(before, d, 64);
    }
    if (end[0] != 0 && (!vdir || (inside && end[0] < vdir[tile]))) {
        const uint16_t *w = img + t.brow_word;
        const uint32_t q = end[0];
        if (!(w[q] & 0x8000u)) {
            // 8-word groups of the image, aligned as the image is: lane l
            // looks at group `top - l`, whose words before q and inside the
            // block row count
            const uint64_t at = t.brow_word + q;  // first word not looked at
            for (uint64_t top = (at - 1) >> 3;; top -= 64) {
                uint32_t head = 0;
                bool any = false;
                if (top >= (uint64_t)lane && (top - lane) * 8 + 7 >= t.brow_word) {
                    const uint64_t g = (top - lane) * 8;
                    const uint4 v = *(const uint4 *)(img + g);
                    const uint32_t x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const uint32_t word = (x[j >> 1] >> ((j & 1) * 16)) & 0xFFFFu;
                        if (g + j >= t.brow_word && g + j < at && (word & 0x8000u)) {
                            head = word;
                            any = true;
                        }
                    }
                }
                const uint64_t m = __ballot(any);
                if (m) {
                    // the lowest such lane is the nearest group, its last
                    // head the nearest word
                    carry = __shfl(head, __ffsll((unsigned long long)m) - 1, 64) & 0x7FFFu;
                    break;
                }
                if (top < 64 || (top - 63) * 8 <= t.brow_word) break;  // (not reached: the tile has a header)
            }
        }
    }
    if (lane) return;
    if (end[0] > end[1] || end[1] > words || d0 >= d1 || dir[tile].x > end[0]) *bad = 1;
    Item *o = items + i;
    o->begin = o->rot_begin = end[0];
    o->nwords = end[1] - end[0];
    o->dir_begin = o->rot_dir = tile;
    o->carry = carry;
    o->before = before;
}

uint32_t grid_for(fmx_ctx *ctx, uint64_t n)
{
    const uint64_t want = (n + kT - 1) / kT, cap = (uint64_t)ctx->num_cus * 32;
    return (uint32_t)std::max<uint64_t>(1, std::min(want, cap));
}

}  // namespace

fmx_status decode_lists(fmx_ctx *ctx, const fmx_spm *src, uint32_t *rows, uint32_t *cols, void *vals,
                        uint32_t *uses)
{
    hipStream_t s = ctx->stream;
    if (!src->d_image) return fail(ctx, FMX_EINVAL, "internal error: the image is not in HBM");
    if (src->nnz >= (1ull << 32)) return fail(ctx, FMX_EUNSUPPORTED, "more than 2^32 - 1 non-zeros to list");
    const uint64_t nbr = src->nbr, ntiles = src->brow_dir[nbr];
    DevBuf<int64_t> offs;
    DevBuf<uint32_t> bdir, tbr, tnnz;
    FMX_HIP(ctx, offs.alloc(ctx, nbr + 1));
    FMX_HIP(ctx, bdir.alloc(ctx, nbr + 1));
    FMX_HIP(ctx, tbr.alloc(ctx, ntiles));
    FMX_HIP(ctx, tnnz.alloc(ctx, ntiles));
    FMX_HIP(ctx, hipMemcpyAsync(offs.p, src->offs.data(), (nbr + 1) * sizeof(int64_t), hipMemcpyHostToDevice, s));
    FMX_HIP(ctx, hipMemcpyAsync(bdir.p, src->brow_dir.data(), (nbr + 1) * sizeof(uint32_t), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(tile_origin, dim3(grid_for(ctx, nbr)), dim3(kT), 0, s, bdir.p, nbr, tbr.p);
    hipLaunchKernelGGL(tile_count, dim3(grid_for(ctx, ntiles)), dim3(kT), 0, s, src->d_image, offs.p, src->d_dir,
                       tbr.p, ntiles, tnnz.p);
    FMX_HIP(ctx, hipGetLastError());
    uint32_t total = 0;
    fmx_status st = scan_exclusive<uint32_t>(ctx, tnnz.p, tnnz.p, ntiles, &total, s);
    if (st) return st;
    if (total != src->nnz) return fail(ctx, FMX_EINVAL, "internal error: tile counts disagree with the image");
    hipLaunchKernelGGL(decode, dim3(grid_for(ctx, ntiles)), dim3(kT), 0, s, src->d_image, offs.p, src->d_dir, tbr.p,
                       tnnz.p, ntiles, src->H, src->W, (uint32_t)src->esz, rows, cols, (uint8_t *)vals, uses);
    FMX_HIP(ctx, hipGetLastError());
    FMX_HIP(ctx, hipStreamSynchronize(s));  // the directory copies above read host memory
    return FMX_OK;
}

fmx_status rank_columns(fmx_ctx *ctx, const uint32_t *uses, uint64_t ncols, uint64_t nnz, uint64_t permille,
                        uint32_t **newid_out, uint32_t **hot_out, uint64_t *nhot_out)
{
    *newid_out = *hot_out = nullptr;
    *nhot_out = 0;
    hipStream_t s = ctx->stream;
    DevBuf<uint64_t> keys, ktmp, before, nhot;
    FMX_HIP(ctx, keys.alloc(ctx, ncols));
    FMX_HIP(ctx, ktmp.alloc(ctx, ncols));
    FMX_HIP(ctx, before.alloc(ctx, ncols));
    FMX_HIP(ctx, nhot.alloc(ctx, 1));
    hipLaunchKernelGGL(rank_keys, dim3(grid_for(ctx, ncols)), dim3(kT), 0, s, uses, ncols, keys.p);
    FMX_HIP(ctx, hipGetLastError());
    uint64_t *sorted = nullptr;
    // by the uses only: the keys start in column order and the sort is stable
    fmx_status st = radix_sort_u64(ctx, keys.p, ktmp.p, ncols, 32, 64, &sorted, s);
    if (st) return st;
    hipLaunchKernelGGL(ranked_uses, dim3(grid_for(ctx, ncols)), dim3(kT), 0, s, sorted, ncols, before.p,
                       nhot.p);
    FMX_HIP(ctx, hipGetLastError());
    st = scan_exclusive<uint64_t>(ctx, before.p, before.p, ncols, nullptr, s);
    if (st) return st;
    hipLaunchKernelGGL(cut, dim3(grid_for(ctx, ncols)), dim3(kT), 0, s, sorted, before.p, ncols, nnz * permille,
                       nhot.p);
    FMX_HIP(ctx, hipGetLastError());
    uint64_t nh = 0;
    st = pinned_fetch(ctx, &nh, nhot.p, sizeof(uint64_t), 0, s);
    if (st) return st;
    FMX_HIP(ctx, hipStreamSynchronize(s));
    pinned_get(ctx, &nh, sizeof(uint64_t), 0);
    if (nh == 0 || nh + ncols > (1ull << 32)) return FMX_OK;  // no hot columns, or ids past 32 bits
    DevBuf<uint32_t> newid, hot;
    FMX_HIP(ctx, newid.alloc(ctx, ncols));
    // (stays with the matrix: of its own size, a kept block may be twice that)
    FMX_HIP(ctx, dev_malloc(ctx, (void **)&hot.p, nh * sizeof(uint32_t)));
    hipLaunchKernelGGL(new_ids, dim3(grid_for(ctx, ncols)), dim3(kT), 0, s, ncols, nh, newid.p);
    hipLaunchKernelGGL(hot_ids, dim3(grid_for(ctx, nh)), dim3(kT), 0, s, sorted, nh, newid.p, hot.p);
    FMX_HIP(ctx, hipGetLastError());
    *newid_out = newid.release();
    *hot_out = hot.release();
    *nhot_out = nh;
    return FMX_OK;
}

fmx_status gather_order_lists(fmx_ctx *ctx, const fmx_spm *src, uint64_t ncols, uint64_t permille,
                              uint32_t *rows, uint32_t *cols, void *vals, uint32_t **hot_out, uint64_t *nhot_out)
{
    hipStream_t s = ctx->stream;
    *hot_out = nullptr;
    *nhot_out = 0;
    DevBuf<uint32_t> uses, newid;
    FMX_HIP(ctx, uses.alloc(ctx, ncols));
    FMX_HIP(ctx, hipMemsetAsync(uses.p, 0, ncols * sizeof(uint32_t), s));
    fmx_status st = decode_lists(ctx, src, rows, cols, vals, uses.p);
    if (!st) st = rank_columns(ctx, uses.p, ncols, src->nnz, permille, &newid.p, hot_out, nhot_out);
    if (st || !*nhot_out) return st;
    hipLaunchKernelGGL(relabel, dim3(grid_for(ctx, src->nnz)), dim3(kT), 0, s, cols, src->nnz, newid.p);
    FMX_HIP(ctx, hipGetLastError());
    FMX_HIP(ctx, hipStreamSynchronize(s));
    return FMX_OK;
}

fmx_status plan_cuts(fmx_ctx *ctx, const fmx_spm *s, Item *items, uint32_t n)
{
    if (!s->d_image) return fail(ctx, FMX_EINVAL, "internal error: the image is not in HBM");
    uint32_t *bad = (uint32_t *)((char *)ctx->pinned + kPinnedFlag);
    *(volatile uint32_t *)bad = 0;
    hipLaunchKernelGGL(fix_items, dim3((n + kT / 64 - 1) / (kT / 64)), dim3(kT), 0, ctx->stream,
                       (const uint16_t *)s->d_image, s->d_dir, s->esz ? s->d_vdir : nullptr, items, n, bad);
    FMX_HIP(ctx, hipGetLastError());
    return FMX_OK;
}

}  // namespace fmx
