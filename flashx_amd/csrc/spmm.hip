// spmm.hip -- gfx950 SpMM over the reference's 2D tile image.
//
// Reference semantics: block_spmm_task_impl::run_on_block with row_part_func
// and coo_func (matrix/sparse_matrix.h:219-375): for every non-zero (r, c) of
// a tile, Y[r][0..k) += X[c][0..k) (binary matrix, value 1).
//
// Execution model (one wave = one work item, no cross-wave sharing):
//   * an item is a contiguous word range of one block row (tile headers and
//     all) plus a band of <= Hs output rows kept in LDS;
//   * the range is decoded 512 words at a time (a "chunk", 16-byte aligned),
//     lane l owning 8 consecutive words.  A header is 8 words and a tile at
//     least 11, so a lane's entries belong to one tile, the last one that
//     starts at or before its first word, and two 8-bit masks (row heads and
//     entries) describe its words.  The row in effect at a lane's first word
//     and its first queue position are wave scans (DPP), and the (global
//     column, band row) entries go to an LDS queue in stream order;
//   * the queue is drained with vector gathers of X rows (16 bytes per lane,
//     L lanes per non-zero).  Lane group g takes 8 consecutive entries, so a
//     run of one row (a row part of a tile) is summed in registers and reaches
//     the band with one LDS add per element at each row change;
//   * the next chunk's words are requested behind the first gathers; a wave's
//     own decode and gathers alternate, and the other resident waves (five
//     per SIMD, as LDS allows) keep gathers in flight meanwhile;
//   * the band is written to Y once (rows without non-zeros are 0), or to a
//     partial slot when a power-law band was split over several items; split
//     bands are summed slot by slot, in stream order, by spmm_reduce.
// Each band is owned by exactly one wave, so results do not depend on timing.
// FP32 data accumulate in an FP64 band and are rounded once on write-out.
#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "fmx_internal.h"

namespace fmx {
namespace {

constexpr int kWPB = 1;  // waves per workgroup: one item, so LDS packs per wave

struct SpmmArgs {
    const uint16_t *img;
    const uint2 *dir;
    const Item *items;
    const void *X;
    void *Y;
    void *partial;
    int64_t ldx;
    int64_t ldy;
    uint32_t nitems;
    uint32_t hs;
    uint32_t wave_bytes;
    uint32_t band_bytes;
    uint32_t band_stride;
    int log2w;
    int k;
    uint64_t ncols;
    const uint32_t *vdir;  // weighted images: values-region word of each tile
    int vwords;            // weighted images: u16 words per value (2 or 4)
    const double *rscale;  // floating-point data: Y row r is scaled by rscale[r] (or null)
    int ycol;              // Y column-major: element (r, j) at Y[j * ldy + r]
    int round_first;       // a scaled row's sum is rounded to T before it is scaled
    int low_bands;         // bands are lower than tiles: entries outside an item's band are met
    const void *Xhot;      // gather-order images: rows of columns < nhot (leading dimension k)
    uint64_t nhot;         // columns c >= nhot are row c - nhot of X
    const void *Xcold;     // narrow forms: X - nhot rows, so that row c of it is column c >= nhot
    uint32_t xstride;      // narrow forms: bytes from row to row of X (and Xhot)
};

// Narrow: the columns fit 24 bits, the operand 32-bit byte offsets and the
// band 8-bit row numbers (narrow_ok).  A queue entry is then one word, and a
// row's address one 24-bit multiply-add onto a scalar base, instead of a
// 64-bit product per gather.
constexpr int kRowShift = 24;

// Where element colb / sizeof(T) of row gcol of the gathered operand lies:
// with HOT (a gather-order image) in the dense hot block for the first nhot
// columns and in X for the others, else in X.
template <typename T, bool HOT, bool NARROW>
__device__ __forceinline__ const T *xrow(const SpmmArgs &a, uint32_t gcol, uint32_t colb)
{
    if constexpr (NARROW) {
        const uint32_t off = __umul24(gcol, a.xstride) + colb;
        if constexpr (!HOT) return (const T *)((const char *)a.X + off);
        const char *base = gcol < (uint32_t)a.nhot ? (const char *)a.Xhot : (const char *)a.Xcold;
        return (const T *)(base + off);
    } else {
        const T *p;
        if constexpr (!HOT) p = (const T *)a.X + (uint64_t)gcol * a.ldx;
        else p = gcol < a.nhot ? (const T *)a.Xhot + (uint64_t)gcol * (uint32_t)a.k
                               : (const T *)a.X + (uint64_t)(gcol - a.nhot) * a.ldx;
        return (const T *)((const char *)p + colb);
    }
}

template <typename T, int E, bool ALIGNED = true>
struct alignas(ALIGNED ? sizeof(T) * E : sizeof(T)) Vec {
    T v[E];
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t rdlane(uint32_t v, int l)
{
    return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}

__device__ __forceinline__ uint32_t uni(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}

template <typename T>
__device__ __forceinline__ void lds_add(T *p, T v)
{
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Orders this wave's LDS writes before its later LDS reads.  LDS executes one
// wave's instructions in order, so only compiler reordering must be stopped;
// a fence would also wait for every outstanding global load.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
}

// Inclusive scans over the wave's lanes on DPP moves (no LDS trip): within
// rows of 16 lanes, then row 15's total into the next row and lane 31's into
// the upper half.  Lanes without a source keep the identity.
template <typename OP>
__device__ __forceinline__ int wave_scan(int v, int identity, OP op)
{
    v = op(v, __builtin_amdgcn_update_dpp(identity, v, 0x111, 0xf, 0xf, false));  // row_shr:1
    v = op(v, __builtin_amdgcn_update_dpp(identity, v, 0x112, 0xf, 0xf, false));  // row_shr:2
    v = op(v, __builtin_amdgcn_update_dpp(identity, v, 0x114, 0xf, 0xf, false));  // row_shr:4
    v = op(v, __builtin_amdgcn_update_dpp(identity, v, 0x118, 0xf, 0xf, false));  // row_shr:8
    v = op(v, __builtin_amdgcn_update_dpp(identity, v, 0x142, 0xa, 0xf, false));  // row_bcast:15
    v = op(v, __builtin_amdgcn_update_dpp(identity, v, 0x143, 0xc, 0xf, false));  // row_bcast:31
    return v;
}
__device__ __forceinline__ int wave_sum(int v) { return wave_scan(v, 0, [](int a, int b) { return a + b; }); }
__device__ __forceinline__ int wave_max(int v, int least)
{
    return wave_scan(v, least, [](int a, int b) { return a > b ? a : b; });
}

// LDS accumulator type: FP32 data accumulate in FP64 (ds_add_f64 is fast on
// gfx950 where ds_add_f32 is not, and the sum is then rounded once).
template <typename T> struct AccOf { using type = T; };
template <> struct AccOf<float> { using type = double; };

template <typename T, int K>
struct Lanes {
    static constexpr int S = sizeof(T);
    static constexpr int VB = (K * S < 16) ? K * S : 16;  // bytes per lane
    static constexpr int E = VB / S;                       // elements per lane
    static constexpr int L = K / E;                        // lanes per non-zero
    static constexpr int NZP = 64 / L;                     // non-zeros per pass
};

// Compiled row forms: K > 0 is a width of K columns, one of the powers of two
// above; K < 0 is any width of at least -K columns, -K elements per lane
// (Row below); K = 0 walks flat (entry, element) pairs, one element per lane
// and step: rows wider than 64 lanes hold, and the sequential mode's runtime
// widths (never in gather order).
template <typename T, int K>
constexpr int row_elems()
{
    if constexpr (K > 0) return Lanes<T, K>::E;
    else return K < 0 ? -K : 1;
}

// This lane's share of the rows in a batch: L lanes take one row, lane q of
// them the E columns from byte colb with one load, and nzp rows go side by
// side.  Element i is added at band column off[i]: the lanes of one add touch
// consecutive words.  With a width that is no multiple of E the last lane's
// load starts early, so that it ends with the row; the columns it shares with
// its neighbour go to the band row's spare word, and so does everything of
// the lanes left over (64 mod L, and beyond 32 rows), which repeat lane 0's
// load.  The loads then need only T's alignment (the hardware takes 16 bytes
// at any dword).
template <typename T, int K>
struct Row {
    static constexpr int E = row_elems<T, K>();
    uint32_t g, nzp, colb, off[E];
    bool on = true;  // the lane has a share
    __device__ __forceinline__ Row(int k, int lane)
    {
        if constexpr (K > 0) {
            using C = Lanes<T, K>;
            const uint32_t q = lane % C::L;
            g = lane / C::L;
            nzp = C::NZP;
            colb = q * E * sizeof(T);
#pragma unroll
            for (int i = 0; i < E; i++) off[i] = i * C::L + q;
        } else if constexpr (K < 0) {
            const uint32_t L = ((uint32_t)k + E - 1) / E;
            nzp = min(64 / L, 32u);
            g = lane / L;
            const uint32_t q = lane - g * L;
            const uint32_t col0 = min(q * E, (uint32_t)k - E), skip = q * E - col0;
            on = g < nzp;
#pragma unroll
            for (uint32_t i = 0; i < (uint32_t)E; i++) off[i] = !on || i < skip ? E * L : (i - skip) * L + q;
            if (!on) g = 0;
            colb = on ? col0 * sizeof(T) : 0;
        }
    }
};

// Band column of output column c in the order of Row::off.
template <typename T, int K>
__device__ __forceinline__ uint32_t band_col(uint32_t c, uint32_t k)
{
    if constexpr (K == 0) return c;
    constexpr uint32_t E = row_elems<T, K>();
    const uint32_t L = K > 0 ? (uint32_t)(K > 0 ? K : 1) / E : (k + E - 1) / E;
    return (c % E) * L + c / E;
}

constexpr int kP = 8;        // consecutive queue entries of a lane group per batch
constexpr int kChunk = 512;  // words per chunk: 8 per lane
constexpr int kWin = 64;     // directory window: a chunk meets at most (512 - 1) / 11 + 1 tile starts
constexpr uint32_t kNoWord = 0x7FFFFFFFu;  // past every word of a block row

// Queue entry e lives at slot e + e/8: the 8-entry segments of the lane
// groups then start in different LDS banks.  The flat form (K = 0) reads in
// order.  Whole batches are drained, so the slots past the last entry are
// filled up: batches of at most 32 rows side by side (K < 0) end at entry 672
// at the latest.
template <int K>
__device__ __forceinline__ uint32_t qslot(uint32_t e) { return K ? e + e / kP : e; }
template <int K>
constexpr int queue_slots() { return K > 0 ? kChunk + kChunk / kP + 1 : K < 0 ? 672 + 672 / kP + 1 : kChunk + 1; }

// A wave's LDS: the band, the queue's columns, values and rows, the window,
// the lanes' tile flags and the window's value words.
struct Layout {
    uint32_t val, row, win, flag, wval, bytes;
};
template <int K, bool WEIGHTED, bool NARROW>
__host__ __device__ __forceinline__ Layout lds_layout(uint32_t band_bytes)
{
    constexpr uint32_t QS = queue_slots<K>();
    Layout l;
    l.val = band_bytes + QS * 4;
    l.row = l.val + (WEIGHTED ? QS * 4 : 0);
    l.win = (l.row + (NARROW ? 0 : QS * 2) + 7) & ~7u;
    l.flag = l.win + (kWin + 1) * 8;
    l.wval = l.flag + 64 * 4;
    l.bytes = (l.wval + (WEIGHTED ? kWin * 4 : 0) + 15) & ~15u;
    return l;
}

// Entry slots: the column, and the band row (`dump`, the row past the band,
// for an entry outside it, whose column is 0 then).
template <bool NARROW>
struct Queue {
    uint32_t *col;
    uint16_t *row;
    __device__ __forceinline__ void put(uint32_t sl, uint32_t c, uint32_t r) const
    {
        if constexpr (NARROW) {
            col[sl] = r << kRowShift | c;
        } else {
            col[sl] = c;
            row[sl] = (uint16_t)r;
        }
    }
    __device__ __forceinline__ void get(uint32_t sl, uint32_t &c, uint32_t &r) const
    {
        c = col[sl];
        if constexpr (NARROW) {
            r = c >> kRowShift;
            c &= (1u << kRowShift) - 1;
        } else {
            r = row[sl];
        }
    }
};

// ---------------------------------------------------------------------------
// Decode.  A stored tile is >= 11 words (16-byte header, one entry, end
// marker; a 16-byte stub only for an empty block row, which is an item by
// itself).

struct ItemCtx {
    uint64_t bw;          // absolute word index of the block row
    int32_t begin, pend;  // item words [begin, pend), relative to the block row
    uint32_t sb_base, rows, dump;
    int log2w;
    uint32_t last_col;
};

// One directory entry of the window per lane, and (weighted) its values word.
struct Window {
    uint2 e;
    uint32_t v;
    bool live;  // inside the block row
};

__device__ __forceinline__ int32_t clamp8(int32_t x) { return x < 0 ? 0 : x > 8 ? 8 : x; }

// Decodes the chunk starting at absolute word c (8-word aligned) from this
// lane's 8 words in wreg and the directory window, whose entry 0 holds the
// chunk's first item word.  Writes the chunk's entries in stream order and
// returns their number; carry becomes the row in effect after the chunk.
// Weighted images (W): a tile's values follow its COO region, one per
// non-zero in stream order (SCSR values, then COO values,
// sparse_matrix_format.h:233-241).  Words at or past the values region are
// not entries, and the value of an entry is as many values behind the
// region's start as entries of its tile come before it: those decoded in the
// chunk before the tile's first lane do not count, and c0 of window tile 0's
// lie before this chunk (in earlier ones, or before the item).  tiles: how many
// tiles of the window have lanes in this chunk; qt: the entry that the value
// positions of lane 63's tile count from.
template <int K, bool W, bool NARROW>
__device__ __forceinline__ uint32_t decode_chunk(const ItemCtx &ic, uint64_t c, const uint32_t *wreg,
                                                 const Window &w, uint2 *win, uint32_t *flag, uint32_t *wval, int c0,
                                                 int vwords, int &carry, const Queue<NARROW> &q, uint32_t *qval,
                                                 int lane, int &tiles, int &qt)
{
    const int32_t cb = (int32_t)((int64_t)c - (int64_t)ic.bw);
    const int32_t p0 = cb + lane * 8;
    // Window tile t rules the lanes from the first one whose words start at
    // or behind it (tile 0: from lane 0); no two tiles begin with one lane.
    // Lanes leave their tile's mark there, valid in this chunk only.
    win[lane] = w.live ? w.e : make_uint2(kNoWord, 0u);
    if constexpr (W) wval[lane] = w.v;
    const int32_t f = lane == 0 ? 0 : ((int32_t)w.e.x - cb + 7) >> 3;
    if (w.live && f < 64) flag[f] = (uint32_t)cb;
    wave_sync();
    const bool begins = flag[lane] == (uint32_t)cb;
    const uint64_t bm = __ballot(begins);
    const uint32_t j = __builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u)) +
                       (begins ? 0u : ~0u);
    const uint2 t = win[j];
    int32_t stop = (int32_t)win[j + 1].x;
    stop = stop < ic.pend ? stop : ic.pend;
    uint32_t tv = 0;
    if constexpr (W) {
        tv = wval[j];
        stop = stop < (int32_t)tv ? stop : (int32_t)tv;
    }
    // this lane's item words behind the tile's header and before its end
    const int32_t from = (int32_t)t.x + 8 > ic.begin ? (int32_t)t.x + 8 : ic.begin;
    const int32_t lo = clamp8(from - p0), hi = clamp8(stop - p0);
    const uint32_t body = hi > lo ? ((1u << (hi - lo)) - 1u) << lo : 0u;
    // bit i: word i has the head bit (the top bytes of four words side by
    // side, their top bits weighted 1, 2, 4, 8 by a dot product)
    const uint32_t y0 = __builtin_amdgcn_perm(wreg[1], wreg[0], 0x07050301u);
    const uint32_t y1 = __builtin_amdgcn_perm(wreg[3], wreg[2], 0x07050301u);
    const uint32_t hb = __builtin_amdgcn_udot4((y1 >> 7) & 0x01010101u, 0x80402010u,
                                               __builtin_amdgcn_udot4((y0 >> 7) & 0x01010101u, 0x08040201u, 0u, false),
                                               false);
    const uint32_t heads = body & hb, ents = body & ~hb;
    // the last head's row, scanned together with its lane: the nearest lane
    // below with a head gives the row in effect at this lane's first word
    const int last = 31 - __clz((int)heads);
    const uint32_t w01 = last & 2 ? wreg[1] : wreg[0], w23 = last & 2 ? wreg[3] : wreg[2];
    const uint32_t lw = (last & 4 ? w23 : w01) >> ((last & 1) * 16);
    const int key = wave_max(heads ? (lane << 16) | (int)(lw & 0x7FFFu) : -1, -1);
    const int below = __builtin_amdgcn_update_dpp(-1, key, 0x138, 0xf, 0xf, false);  // wave_shr:1
    int r = below >= 0 ? below & 0x7FFF : carry;
    const int top = (int)rdlane((uint32_t)key, 63);
    if (top >= 0) carry = top & 0x7FFF;
    const int cnt = __popc(ents);
    const int incl = wave_sum(cnt);
    const uint32_t qn = rdlane((uint32_t)incl, 63);
    uint32_t o = (uint32_t)(incl - cnt);
    uint32_t vw = 0;
    if constexpr (W) {
        // (the counts never fall, so the latest tile start has the largest)
        int q0 = wave_max(begins ? incl - cnt : 0, 0);
        q0 = j == 0 ? -c0 : q0;
        vw = tv + (uint32_t)((int)o - q0) * (uint32_t)vwords;
        tiles = __popcll(bm);
        qt = (int)rdlane((uint32_t)q0, 63);
    }
    const uint32_t colbase = t.y << ic.log2w;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t word = (wreg[i >> 1] >> ((i & 1) * 16)) & 0xFFFFu;
        if (heads & (1u << i)) r = (int)(word & 0x7FFFu);
        if (ents & (1u << i)) {
            const uint32_t br = (uint32_t)r - ic.sb_base;  // no row in effect: r = -1, past any band
            const bool keep = br < ic.rows;
            const uint32_t gcol = min(colbase | word, ic.last_col);
            const uint32_t sl = qslot<K>(o);
            q.put(sl, keep ? gcol : 0u, keep ? br : ic.dump);
            if constexpr (W) {
                qval[sl] = vw;
                vw += (uint32_t)vwords;
            }
            o++;
        }
    }
    return qn;
}

// This lane's words of chunk c, clamped to the aligned 8-word group holding
// the item's last word lastw (always inside the image allocation, whose size
// is a multiple of 4096 bytes).  The image is streamed once: non-temporal
// loads, so it does not displace X in L2.
__device__ __forceinline__ void load_words(const uint16_t *img, uint64_t c, uint64_t lastw, int lane, uint32_t *wreg)
{
    const uint64_t last8 = lastw & ~7ull;
    uint64_t g = c + (uint64_t)lane * 8;
    g = g < last8 ? g : last8;
    const u32x4 v = __builtin_nontemporal_load((const u32x4 *)(img + g));
    wreg[0] = v.x;
    wreg[1] = v.y;
    wreg[2] = v.z;
    wreg[3] = v.w;
}

// Directory entry ct + lane (clamped); `live` marks one inside the block row.
template <bool W>
__device__ __forceinline__ void load_window(const SpmmArgs &a, uint32_t ct, uint32_t dlast, int lane, Window &w)
{
    const uint32_t t = ct + lane;
    w.live = t <= dlast;
    w.e = a.dir[t < dlast ? t : dlast];
    if constexpr (W) w.v = a.vdir[t < dlast ? t : dlast];
}

// Drains (K != 0): gathers of P consecutive entries per lane group, summed in
// registers per row run, added to the band at row changes.
template <typename T, int K>
__device__ __forceinline__ void load_row(Vec<T, row_elems<T, K>()> &v, const T *p)
{
    if constexpr (K > 0) {
        v = *(const Vec<T, row_elems<T, K>()> *)p;
    } else {
        const Vec<T, row_elems<T, K>(), false> u = *(const Vec<T, row_elems<T, K>(), false> *)p;
#pragma unroll
        for (int i = 0; i < row_elems<T, K>(); i++) v.v[i] = u.v[i];
    }
}

// The batch of entries from `base` (a multiple of 8): lane group g's are
// g * 8 .. g * 8 + 7 of it.
template <typename T, int K, bool HOT, bool NARROW>
__device__ __forceinline__ void gather_batch(const SpmmArgs &a, const Row<T, K> &row, const Queue<NARROW> &q,
                                             uint32_t base, Vec<T, row_elems<T, K>()> *v, uint32_t *rr)
{
    uint32_t gcs[kP];
    const uint32_t s0 = qslot<K>(base) + row.g * (kP + 1);
#pragma unroll
    for (int pp = 0; pp < kP; pp++) q.get(s0 + pp, gcs[pp], rr[pp]);
    // every queue read before the first gather, every gather before the first use
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int pp = 0; pp < kP; pp++) load_row<T, K>(v[pp], xrow<T, HOT, NARROW>(a, gcs[pp], row.colb));
    __builtin_amdgcn_sched_barrier(0);
}

// Fills the slots from entry qn up to entry `end` with row-less entries.
template <int K, bool NARROW>
__device__ __forceinline__ void fill_queue(const Queue<NARROW> &q, uint32_t *qval, uint32_t qn, uint32_t end,
                                           uint32_t dump, int lane)
{
    for (uint32_t e = qn + lane; e < end; e += 64) {
        q.put(qslot<K>(e), 0u, dump);
        if (qval) qval[qslot<K>(e)] = 0u;  // a safe address
    }
    wave_sync();
}

// Whether lanes without a share of a batch are kept from adding: at runtime
// widths, which can leave 31 of 64 lanes over, and where many entries go side
// by side.  Elsewhere the mask costs more than it saves (FP32 k = 64, few
// non-zeros: 3%).
template <typename T, int K>
constexpr bool stays_out()
{
    if constexpr (K > 0) return Lanes<T, K>::NZP >= 16;
    else return true;
}

// Adds a batch to the band, run by run; elem(pp, i) is entry pp's element i
// in the accumulator's type (times its value).  Lane groups without an entry
// (`some` is false, in a chunk's last batch) and lanes without a share of a row
// stay out, and single adds (!RUNS) of entries outside the band are left out
// where there are any: all of those go to one row, whose adds the LDS takes
// one after the other (2^20 evenly picked columns, 4 edges a vertex, FP64 k = 1
// in 32-row tiles: 151 us with them, 52 without).
template <typename T, int K, typename A, bool RUNS, typename F>
__device__ __forceinline__ void accumulate_batch(A *band, uint32_t S, const Row<T, K> &row, const uint32_t *rr,
                                                 bool some, bool low_bands, uint32_t dump, F elem)
{
    constexpr int E = row_elems<T, K>();
    if (stays_out<T, K>() && (!some || !row.on)) return;
    if constexpr (!RUNS) {
        if (low_bands) {
#pragma unroll
            for (int pp = 0; pp < kP; pp++) {
                if (rr[pp] == dump) continue;
                A *dst = band + __umul24(rr[pp], S);
#pragma unroll
                for (int i = 0; i < E; i++) lds_add(dst + row.off[i], elem(pp, i));
            }
        } else {
#pragma unroll
            for (int pp = 0; pp < kP; pp++) {
                A *dst = band + __umul24(rr[pp], S);
#pragma unroll
                for (int i = 0; i < E; i++) lds_add(dst + row.off[i], elem(pp, i));
            }
        }
    } else {
        A acc[E];
        uint32_t cur = rr[0];
#pragma unroll
        for (int i = 0; i < E; i++) acc[i] = elem(0, i);
#pragma unroll
        for (int pp = 1; pp < kP; pp++) {
            if (rr[pp] != cur) {
                A *dst = band + __umul24(cur, S);
#pragma unroll
                for (int i = 0; i < E; i++) lds_add(dst + row.off[i], acc[i]);
                cur = rr[pp];
#pragma unroll
                for (int i = 0; i < E; i++) acc[i] = elem(pp, i);
            } else {
#pragma unroll
                for (int i = 0; i < E; i++) acc[i] += elem(pp, i);
            }
        }
        A *dst = band + __umul24(cur, S);
#pragma unroll
        for (int i = 0; i < E; i++) lds_add(dst + row.off[i], acc[i]);
    }
}

// ---------------------------------------------------------------------------
// Sequential mode: every output element is the left-to-right sum of its
// row's products in stream order, one rounding per addition, starting from
// the zeroed band -- the reference's own order (row_part_func / coo_func,
// matrix/sparse_matrix.h:219-331, `dest_row[j] += src_row[j] * data` per
// non-zero, tiles in ascending block column).  Within a tile a row's columns
// ascend and tiles ascend, so this is each row's ascending-column sum, the
// same for every tile shape.  Lane groups hold consecutive queue entries, so
// they add in group order: group g reads the band after group g-1 wrote it
// (one wave's LDS accesses execute in program order).  A run of one row
// inside a group is chained in registers, which is the same sequence of
// roundings.
template <typename T, int K>
__device__ __forceinline__ void accumulate_batch_seq(T *band, uint32_t S, int lane, uint32_t entries,
                                                     const Vec<T, Lanes<T, K>::E> *v, const uint32_t *rr)
{
#pragma clang fp contract(off)
    using C = Lanes<T, K>;
    const int q = lane % C::L;
    const int g = lane / C::L;
    // (the groups with entries, where there may be many without)
    const int groups = C::NZP >= 32 && entries < C::NZP * kP ? (int)(entries + kP - 1) / kP : C::NZP;
    for (int gg = 0; gg < groups; gg++) {
        if (g == gg) {
            T acc[C::E];
            uint32_t cur = rr[0];
            T *at = band + cur * S + q;
#pragma unroll
            for (int i = 0; i < C::E; i++) acc[i] = at[i * C::L];
#pragma unroll
            for (int pp = 0; pp < kP; pp++) {
                if (rr[pp] != cur) {
#pragma unroll
                    for (int i = 0; i < C::E; i++) at[i * C::L] = acc[i];
                    cur = rr[pp];
                    at = band + cur * S + q;
#pragma unroll
                    for (int i = 0; i < C::E; i++) acc[i] = at[i * C::L];
                }
#pragma unroll
                for (int i = 0; i < C::E; i++) acc[i] = acc[i] + v[pp].v[i];
            }
#pragma unroll
            for (int i = 0; i < C::E; i++) at[i * C::L] = acc[i];
        }
        wave_sync();
    }
}

// One value of type T from the u16-aligned values region (u16 loads, so no
// alignment beyond 2 bytes is assumed).
template <typename T>
__device__ __forceinline__ T load_value(const uint16_t *p)
{
    if constexpr (sizeof(T) == 4) {
        const uint32_t u = (uint32_t)p[0] | ((uint32_t)p[1] << 16);
        return __builtin_bit_cast(T, u);
    } else {
        const uint64_t u = (uint64_t)p[0] | ((uint64_t)p[1] << 16) | ((uint64_t)p[2] << 32) |
                           ((uint64_t)p[3] << 48);
        return __builtin_bit_cast(T, u);
    }
}

// Runtime width: flat (entry, element) pairs, one element per lane; weighted
// images (V) multiply it by the entry's value.
template <typename T, typename V, typename A, bool NARROW>
__device__ __forceinline__ void drain_generic(const SpmmArgs &a, A *band, uint32_t S, const Queue<NARROW> &q,
                                              const uint32_t *qval, const uint16_t *vimg, uint32_t qn, int lane)
{
    const uint32_t k = (uint32_t)a.k;
    const uint32_t tot = qn * k;
    for (uint32_t base = 0; base < tot; base += 64 * kP) {
        A v[kP];
        uint32_t dst[kP];
#pragma unroll
        for (int pp = 0; pp < kP; pp++) {
            const uint32_t f = base + pp * 64 + lane;
            const uint32_t fc = f < tot ? f : tot - 1;
            const uint32_t e = fc / k, j = fc - e * k;
            uint32_t gc, qr;
            q.get(e, gc, qr);
            v[pp] = (A)*xrow<T, false, NARROW>(a, gc, j * sizeof(T));
            if constexpr (!std::is_void<V>::value) v[pp] *= (A)load_value<V>(vimg + qval[e]);
            dst[pp] = f < tot && qr != a.hs ? qr * S + j : 0xFFFFFFFFu;
        }
#pragma unroll
        for (int pp = 0; pp < kP; pp++)
            if (dst[pp] != 0xFFFFFFFFu) lds_add(band + dst[pp], v[pp]);
    }
}

// Sequential mode at runtime widths: lane j owns output column j (of each
// 64-column slice) and adds the queue's entries in order.  Weighted images
// multiply each gathered element by the entry's value of type V first,
// rounded in T, as `src_row[j] * data` is.
template <typename T, typename V, bool NARROW>
__device__ __forceinline__ void drain_generic_seq(const SpmmArgs &a, T *band, uint32_t S, const Queue<NARROW> &q,
                                                  const uint32_t *qval, const uint16_t *vimg, uint32_t qn, int lane)
{
#pragma clang fp contract(off)
    const uint32_t k = (uint32_t)a.k;
    for (uint32_t j0 = 0; j0 < k; j0 += 64) {
        const uint32_t j = j0 + (uint32_t)lane;
        const bool act = j < k;
        for (uint32_t e0 = 0; e0 < qn; e0 += kP) {
            T v[kP];
            uint32_t dst[kP];
#pragma unroll
            for (int pp = 0; pp < kP; pp++) {
                const uint32_t e = e0 + pp;
                const uint32_t ec = e < qn ? e : qn - 1;
                uint32_t gc, qr;
                q.get(ec, gc, qr);
                v[pp] = *xrow<T, false, NARROW>(a, gc, (act ? j : 0u) * sizeof(T));
                if constexpr (!std::is_void<V>::value) v[pp] = v[pp] * (T)load_value<V>(vimg + qval[ec]);
                dst[pp] = (e < qn && act) ? qr * S + j : 0xFFFFFFFFu;
            }
#pragma unroll
            for (int pp = 0; pp < kP; pp++)
                if (dst[pp] != 0xFFFFFFFFu) band[dst[pp]] = band[dst[pp]] + v[pp];
        }
    }
}

// A row's sum times its output scale: rounded to T once, by the caller's
// store, or (round_first) also before the scaling.
template <typename T, typename A>
__device__ __forceinline__ A scaled(int round_first, A sum, double scale)
{
    return (A)((round_first ? (double)(T)sum : (double)sum) * scale);
}

// The output scales of a band's first 128 rows, requested when the item
// starts so that their latency is hidden by the item's work.
struct RowScale {
    double v[2];
};

template <typename T>
__device__ __forceinline__ RowScale prefetch_rscale(const SpmmArgs &a, uint64_t row0, uint32_t rows, int lane)
{
    RowScale rs{{1.0, 1.0}};
    if constexpr (std::is_floating_point<T>::value) {
        if (a.rscale) {
#pragma unroll
            for (int h = 0; h < 2; h++)
                if ((uint32_t)(h * 64 + lane) < rows) rs.v[h] = a.rscale[row0 + h * 64 + lane];
        }
    }
    return rs;
}

// Writes the band to Y, or to its partial slot.  With row scales, the
// scales of bands of at most 128 rows are staged in scratch LDS (the drained
// queue), so the write loop waits on no global load.
template <typename T, int K, typename A>
__device__ __forceinline__ void write_band(const SpmmArgs &a, const A *band, uint32_t S, uint64_t row0,
                                           uint32_t rows, uint32_t slot, int lane, const RowScale &rs,
                                           double *scratch)
{
    const uint32_t k = K > 0 ? K : (uint32_t)a.k;
    auto bcol = [&](uint32_t cc) -> uint32_t { return band_col<T, K>(cc, k); };
    if (slot == kNone) {
        T *dst = (T *)a.Y + row0 * (uint64_t)a.ldy;
        bool staged = false;
        if constexpr (std::is_floating_point<T>::value) {
            if (a.rscale && rows <= 128) {
                wave_sync();
#pragma unroll
                for (int h = 0; h < 2; h++)
                    if ((uint32_t)(h * 64 + lane) < rows) scratch[h * 64 + lane] = rs.v[h];
                wave_sync();
                staged = true;
            }
        }
        if (a.ycol) {
            // column-major Y: lanes run down a column, so the stores of one
            // column are consecutive
            T *dc = (T *)a.Y + row0;
            for (uint32_t i = lane; i < rows * k; i += 64) {
                const uint32_t cc = i / rows, r = i - cc * rows;
                A v = band[r * S + bcol(cc)];
                if constexpr (std::is_floating_point<T>::value)
                    if (a.rscale) v = scaled<T>(a.round_first, v, staged ? scratch[r] : a.rscale[row0 + r]);
                __builtin_nontemporal_store((T)v, &dc[cc * (uint64_t)a.ldy + r]);
            }
            return;
        }
        for (uint32_t i = lane; i < rows * k; i += 64) {
            const uint32_t r = i / k, cc = i - r * k;
            A v = band[r * S + bcol(cc)];
            if constexpr (std::is_floating_point<T>::value)
                if (a.rscale) v = scaled<T>(a.round_first, v, staged ? scratch[r] : a.rscale[row0 + r]);
            // written once and not read here: non-temporal
            __builtin_nontemporal_store((T)v, &dst[r * (uint64_t)a.ldy + cc]);
        }
    } else {
        A *dst = (A *)a.partial + (uint64_t)slot * a.hs * k;
        for (uint32_t i = lane; i < rows * k; i += 64) {
            const uint32_t r = i / k, cc = i - r * k;
            dst[i] = band[r * S + bcol(cc)];
        }
    }
}

struct ItemState {
    ItemCtx ic;
    uint32_t dlast, slot, ct;
    uint64_t row0;
    int carry;
    int32_t begin, end, rot;  // the whole item, and where processing starts
    uint32_t dir_begin, rot_dir;
    int item_carry;
    int c0, item_c0;  // weighted: entries of the first tile before the segment / the item
};

// Segment 0 is [rot, end) and segment 1 is [begin, rot) (empty without a
// rotation).  A rotated start is a tile start, where no row is carried in.
__device__ __forceinline__ bool select_segment(ItemState &st, int seg)
{
    if (seg == 0) {
        st.ic.begin = st.rot;
        st.ic.pend = st.end;
        st.ct = st.rot_dir;
        st.carry = st.rot == st.begin ? st.item_carry : -1;
        st.c0 = st.rot == st.begin ? st.item_c0 : 0;
        return true;
    }
    if (st.rot == st.begin) return false;
    st.ic.begin = st.begin;
    st.ic.pend = st.rot;
    st.ct = st.dir_begin;
    st.carry = st.item_carry;
    st.c0 = st.item_c0;
    return true;
}

__device__ __forceinline__ ItemState item_state(const SpmmArgs &a, const Item &it)
{
    ItemState s;
    s.ic.bw = it.brow_word;
    s.ic.begin = (int32_t)it.begin;
    s.ic.pend = (int32_t)(it.begin + it.nwords);  // nwords >= 1
    s.ic.sb_base = it.sb_base;
    s.ic.rows = it.rows;
    s.ic.dump = a.hs;
    s.ic.log2w = a.log2w;
    s.ic.last_col = (uint32_t)(a.ncols - 1);
    s.dlast = it.dir_end - 1;
    s.row0 = ((uint64_t)it.row0_hi << 32) | it.row0_lo;
    s.slot = it.slot;
    s.carry = (it.carry == kNone) ? -1 : (int)it.carry;
    s.ct = it.dir_begin;
    s.begin = (int32_t)it.begin;
    s.end = (int32_t)(it.begin + it.nwords);
    s.rot = (int32_t)it.rot_begin;
    s.dir_begin = it.dir_begin;
    s.rot_dir = it.rot_dir;
    s.item_carry = s.carry;
    s.item_c0 = (int)it.before;
    return s;
}

// ---------------------------------------------------------------------------
// The SpMM kernel: chunks of 512 words, each decoded and then drained batch
// by batch.  The next chunk's words and window are requested behind the
// first batch's gathers, so their latency overlaps the gathers'; the gathers
// of one wave are not overlapped with its own decode, other resident waves
// fill that gap.
// V: the type of a weighted image's values, void for a binary one.
// SEQ: the sequential mode (accumulate_batch_seq): the band holds T and
// every element is summed in the reference's order; the plan of such a call
// neither splits nor rotates items.
template <typename T, typename V, int K, bool SEQ, bool HOT, bool NARROW>
__device__ __forceinline__ void spmm_body(const SpmmArgs &a)
{
    constexpr bool W = !std::is_void<V>::value;
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63;
    const uint32_t wv = uni(threadIdx.x >> 6);
    const uint32_t item_id = blockIdx.x * kWPB + wv;
    if (item_id >= a.nitems) return;

    unsigned char *wbase = smem + wv * a.wave_bytes;
    using A = typename std::conditional<SEQ, T, typename AccOf<T>::type>::type;
    const Layout l = lds_layout<K, W, NARROW>(a.band_bytes);
    A *band = (A *)wbase;
    const Queue<NARROW> q{(uint32_t *)(wbase + a.band_bytes), (uint16_t *)(wbase + l.row)};
    uint32_t *qval = W ? (uint32_t *)(wbase + l.val) : nullptr;
    uint2 *win = (uint2 *)(wbase + l.win);
    uint32_t *flag = (uint32_t *)(wbase + l.flag);
    uint32_t *wval = W ? (uint32_t *)(wbase + l.wval) : nullptr;

    ItemState st = item_state(a, a.items[item_id]);
    const RowScale rs = prefetch_rscale<T>(a, st.row0, st.ic.rows, lane);
    const Row<T, K> row(a.k, lane);
    const uint32_t S = a.band_stride;
    for (uint32_t i = lane; i < st.ic.rows * S; i += 64) band[i] = A(0);
    if (lane == 0) win[kWin] = make_uint2(kNoWord, 0u);
    const uint16_t *vimg = a.img + st.ic.bw;

    for (int seg = 0; seg < 2; seg++) {
    if (!select_segment(st, seg)) break;
    flag[lane] = kNoWord;
    const uint64_t abs_end = st.ic.bw + (uint64_t)st.ic.pend;
    const uint64_t lastw = abs_end - 1;
    uint64_t c = (st.ic.bw + (uint64_t)st.ic.begin) & ~7ull;
    int c0 = st.c0;  // weighted: entries of window tile 0 before this chunk
    uint32_t wreg[4];
    Window w;
    load_words(a.img, c, lastw, lane, wreg);
    load_window<W>(a, st.ct, st.dlast, lane, w);

    while (c < abs_end) {
        int tiles = 0, qt = 0;
        const uint32_t qn = decode_chunk<K, W, NARROW>(st.ic, c, wreg, w, win, flag, wval, c0, a.vwords, st.carry, q,
                                                       qval, lane, tiles, qt);
        uint64_t cn = c + kChunk;
        wave_sync();
        // the next chunk's words and window (this chunk's are in LDS now),
        // whose entry 0 is this window's last tile starting at or before it
        auto fetch_next = [&]() {
            if (cn < abs_end) {
                uint32_t pn = (uint32_t)((int64_t)cn - (int64_t)st.ic.bw);
                int adv = __popcll(__ballot(w.live && w.e.x <= pn));
                if constexpr (W) {
                    // from inside a tile's values to the next tile (with
                    // cuts inside tiles, R-MAT scale 14 FP32 k = 16 weighted
                    // 41 -> 14 us, scale 20 in gather order 298 -> 183)
                    if (adv < 64 && pn >= rdlane(w.v, adv - 1)) {
                        const bool more = (__ballot(w.live) >> adv) & 1;
                        const uint64_t to = more ? (st.ic.bw + rdlane(w.e.x, adv)) & ~7ull : abs_end;
                        if (to > cn) {
                            cn = to < abs_end ? to : abs_end;
                            if (cn == abs_end) return;
                            pn = (uint32_t)((int64_t)cn - (int64_t)st.ic.bw);
                            adv = __popcll(__ballot(w.live && w.e.x <= pn));
                        }
                    }
                }
                // that tile has entries in this chunk if lanes of it began here
                if constexpr (W) c0 = adv > tiles ? 0 : (int)qn - qt;
                st.ct += (uint32_t)adv - 1;
                load_words(a.img, cn, lastw, lane, wreg);
                load_window<W>(a, st.ct, st.dlast, lane, w);
            }
        };
        if constexpr (K != 0) {
            // requested behind the first batch's gathers: a wait for the
            // gathers need not wait for these, and their latency overlaps
            // the gathers' instead of preceding them
            constexpr int E = row_elems<T, K>();
            const uint32_t batch = row.nzp * kP;
            bool fetched = false;
            for (uint32_t base = 0; base < qn; base += batch) {
                if (base + batch > qn) fill_queue<K>(q, qval, qn, base + batch, st.ic.dump, lane);
                Vec<T, E> v[kP];
                uint32_t rr[kP];
                typename std::conditional<W, V, int>::type vals[kP];
                if constexpr (W) {
                    const uint32_t s0 = qslot<K>(base) + row.g * (kP + 1);
#pragma unroll
                    for (int pp = 0; pp < kP; pp++) vals[pp] = load_value<V>(vimg + qval[s0 + pp]);
                }
                gather_batch<T, K, HOT, NARROW>(a, row, q, base, v, rr);
                if (!fetched) {
                    fetch_next();
                    fetched = true;
                }
                const bool some = base + row.g * kP < qn;
                if constexpr (SEQ) {
                    if constexpr (W) {
                        // products rounded in T, then added in order
#pragma clang fp contract(off)
#pragma unroll
                        for (int pp = 0; pp < kP; pp++)
#pragma unroll
                            for (int i = 0; i < E; i++) v[pp].v[i] = v[pp].v[i] * (T)vals[pp];
                    }
                    accumulate_batch_seq<T, K>(band, S, lane, qn - base, v, rr);
                } else if constexpr (W) {
                    accumulate_batch<T, K, A, true>(band, S, row, rr, some, a.low_bands, st.ic.dump,
                                                    [&](int pp, int i) { return (A)v[pp].v[i] * (A)vals[pp]; });
                } else {
                    // 8-byte data: each entry adds straight into the band.
                    // Run sums save few LDS adds (rows average 2.4 entries
                    // per tile on R-MAT) and their divergent branches cost
                    // more than that for E <= 2 (FP64 k = 16: 1.17 ms
                    // against 1.34 ms with run sums)
                    accumulate_batch<T, K, A, sizeof(T) != 8>(band, S, row, rr, some, a.low_bands, st.ic.dump,
                                                              [&](int pp, int i) { return (A)v[pp].v[i]; });
                }
            }
            if (!fetched) fetch_next();
        } else {
            fetch_next();
            if (qn) {
                if constexpr (SEQ) drain_generic_seq<T, V>(a, band, S, q, qval, vimg, qn, lane);
                else drain_generic<T, V, A>(a, band, S, q, qval, vimg, qn, lane);
            }
        }
        wave_sync();
        c = cn;
    }
    }
    write_band<T, K, A>(a, band, S, st.row0, st.ic.rows, st.slot, lane, rs, (double *)(wbase + a.band_bytes));
}

template <typename T, int K, bool SEQ, bool HOT, bool NARROW>
__global__ void __launch_bounds__(64 * kWPB) __attribute__((amdgpu_waves_per_eu(5, 5))) spmm_lane(SpmmArgs a)
{
    spmm_body<T, void, K, SEQ, HOT, NARROW>(a);
}

template <typename T, typename V, int K, bool SEQ, bool HOT, bool NARROW>
__global__ void __launch_bounds__(64 * kWPB) __attribute__((amdgpu_waves_per_eu(4, 4))) spmm_lane_w(SpmmArgs a)
{
    spmm_body<T, V, K, SEQ, HOT, NARROW>(a);
}

// Y rows of a split band = partial slots summed in stream order: one element
// per thread, four slots' loads in flight (a block per split that walked its
// elements and slots one load at a time took 26 us after each rank-20 SpMM of
// 260,000 vertices; 5 us like this).
template <typename T, typename A>
__global__ void __launch_bounds__(256) spmm_reduce(const Split *splits, const A *partial,
                                                    uint32_t hs, uint32_t k, T *Y, int64_t ldy,
                                                    const double *rscale, int ycol, int round_first)
{
    const Split sp = splits[blockIdx.x];
    const uint32_t i = blockIdx.y * 256 + threadIdx.x;
    if (i >= sp.rows * k) return;
    const uint64_t step = (uint64_t)hs * k;
    const A *p = partial + (uint64_t)sp.slot_begin * step + i;
    A acc = p[0];
    uint32_t s = 1;
    for (; s + 4 <= sp.nslots; s += 4) {
        A v[4];
#pragma unroll
        for (int t = 0; t < 4; t++) v[t] = p[(s + t) * step];
#pragma unroll
        for (int t = 0; t < 4; t++) acc += v[t];
    }
    for (; s < sp.nslots; s++) acc += p[s * step];
    const uint32_t r = i / k, c = i - r * k;
    if constexpr (std::is_floating_point<T>::value)
        if (rscale) acc = scaled<T>(round_first, acc, rscale[sp.row0 + r]);
    if (ycol) Y[c * (uint64_t)ldy + sp.row0 + r] = (T)acc;
    else Y[(sp.row0 + r) * (uint64_t)ldy + c] = (T)acc;
}

// Gathers in flight per lane group (kP): eight 16-byte gathers per lane keep
// spmm_lane at 86 VGPRs at most (FP32 k = 16: 77).  More resident waves with short batches put more
// gathers in flight than fewer waves with long ones: on R-MAT scale 22, FP32
// k = 16, 64x32768 tiles, 0.93 ms against 1.30 ms for 512-entry batches
// overlapped with the next decode at two waves per SIMD (the best earlier
// schedule), and 57 ms against 92 ms on scale 27, FP32 k = 32.

// Raises a kernel's dynamic LDS limit once per process.
template <void (*KERN)(SpmmArgs)>
fmx_status allow_lds(fmx_ctx *ctx)
{
    static bool done = false;
    if (!done) {
        FMX_HIP(ctx, hipFuncSetAttribute((const void *)KERN, hipFuncAttributeMaxDynamicSharedMemorySize,
                                         160 * 1024));
        done = true;
    }
    return FMX_OK;
}

template <void (*KERN)(SpmmArgs)>
fmx_status launch_items(fmx_ctx *ctx, const SpmmArgs &a, hipStream_t stream)
{
    const uint32_t lds = a.wave_bytes * kWPB;
    if (lds > ctx->lds_per_block) return fail(ctx, FMX_EUNSUPPORTED, "band does not fit in LDS");
    fmx_status st = allow_lds<KERN>(ctx);
    if (st) return st;
    const uint32_t blocks = (a.nitems + kWPB - 1) / kWPB;
    if (blocks) {
        hipLaunchKernelGGL(KERN, dim3(blocks), dim3(64 * kWPB), lds, stream, a);
        FMX_HIP(ctx, hipGetLastError());
    }
    return FMX_OK;
}

template <typename T, int K, bool SEQ, bool HOT, bool NARROW>
fmx_status launch_n(fmx_ctx *ctx, SpmmArgs a, int vprim, hipStream_t stream)
{
    // the band and its dump row
    a.band_bytes = (uint32_t)(((uint64_t)(a.hs + 1) * a.band_stride *
                                   sizeof(typename std::conditional<SEQ, T, typename AccOf<T>::type>::type) + 15) & ~15ull);
    a.wave_bytes = a.vdir ? lds_layout<K, true, NARROW>(a.band_bytes).bytes
                          : lds_layout<K, false, NARROW>(a.band_bytes).bytes;
    if (a.vdir) {
        // the stored values are of type T, or float with FP64 dense data
        // (spmm_creator<double, float>)
        if constexpr (std::is_same<T, double>::value)
            if (vprim == 8) return launch_items<spmm_lane_w<double, float, K, SEQ, HOT, NARROW>>(ctx, a, stream);
        return launch_items<spmm_lane_w<T, T, K, SEQ, HOT, NARROW>>(ctx, a, stream);
    }
    return launch_items<spmm_lane<T, K, SEQ, HOT, NARROW>>(ctx, a, stream);
}

// The narrow forms' limits; with a hot block its rows and X's are one stride
// apart.
template <typename T>
bool narrow_ok(const SpmmArgs &a)
{
    const uint64_t stride = (uint64_t)a.ldx * sizeof(T);
    return a.ncols <= (1u << kRowShift) && a.hs < 256 && stride < (1u << 24) &&
           a.ncols * stride + (uint64_t)a.k * sizeof(T) < (1ull << 32) && (!a.nhot || a.ldx == a.k);
}

template <typename T, int K, bool SEQ, bool HOT>
fmx_status launch_k(fmx_ctx *ctx, SpmmArgs a, int vprim, hipStream_t stream)
{
    if (narrow_ok<T>(a)) {
        a.xstride = (uint32_t)(a.ldx * sizeof(T));
        a.Xcold = (const char *)a.X - (size_t)a.nhot * a.xstride;
        return launch_n<T, K, SEQ, HOT, true>(ctx, a, vprim, stream);
    }
    return launch_n<T, K, SEQ, HOT, false>(ctx, a, vprim, stream);
}

// Elements per lane of the runtime-width form for rows of k elements (0: the
// flat form).  Four 4-byte or two 8-byte elements make 16-byte loads; three
// 4-byte columns take two lanes of two.
template <typename T>
int runtime_elems(int k)
{
    const int e = sizeof(T) == 8 || k < 4 ? 2 : 4;
    return k >= e && k <= 64 * e ? e : 0;
}

// Rows of a width without a form of its own, or not aligned for it.  The flat
// form spends a division, a 4- or 8-byte load and an LDS add on each element,
// this one a third of a load and an add per row run: 700,001 vertices x 10
// FP32 columns 140 -> 115 us with the restaging of X, four NMF sweeps of rank
// 20 over 260,000 vertices 2.63 -> 2.08 ms.
template <typename T, bool SEQ, bool HOT>
fmx_status launch_runtime(fmx_ctx *ctx, SpmmArgs a, int vprim, hipStream_t stream)
{
    if constexpr (!SEQ) {
        const int e = runtime_elems<T>(a.k);
        if (e) a.band_stride = (uint32_t)((a.k + e - 1) / e * e + 1);  // whole lanes and a spare word
        if constexpr (sizeof(T) == 4)
            if (e == 4) return launch_k<T, -4, SEQ, HOT>(ctx, a, vprim, stream);
        if (e == 2) return launch_k<T, -2, SEQ, HOT>(ctx, a, vprim, stream);
    }
    // gather-order rows are shorter than 128 bytes, so what is left of them is
    // one column at an address of less than its own alignment
    if constexpr (HOT) return launch_k<T, 1, SEQ, HOT>(ctx, a, vprim, stream);
    else return launch_k<T, 0, SEQ, HOT>(ctx, a, vprim, stream);
}

// HOT (a gather-order image, rows narrower than a 128-byte line) has kernels
// for the widths it is used with; k = 0 asks for the runtime-width form.
template <typename T, bool SEQ, bool HOT>
fmx_status launch_w(fmx_ctx *ctx, SpmmArgs a, int k, int vprim, hipStream_t stream)
{
    constexpr int KMAX = HOT ? (int)(64 / sizeof(T)) : 64;
    if (k > KMAX) k = 0;
    switch (k) {
    case 1: return launch_k<T, 1, SEQ, HOT>(ctx, a, vprim, stream);
    case 2: return launch_k<T, 2, SEQ, HOT>(ctx, a, vprim, stream);
    case 4: return launch_k<T, 4, SEQ, HOT>(ctx, a, vprim, stream);
    case 8: return launch_k<T, 8, SEQ, HOT>(ctx, a, vprim, stream);
    case 16: return launch_k<T, (16 <= KMAX ? 16 : 8), SEQ, HOT>(ctx, a, vprim, stream);
    case 32: return launch_k<T, (32 <= KMAX ? 32 : 8), SEQ, HOT>(ctx, a, vprim, stream);
    case 64: return launch_k<T, (64 <= KMAX ? 64 : 8), SEQ, HOT>(ctx, a, vprim, stream);
    default: return launch_runtime<T, SEQ, HOT>(ctx, a, vprim, stream);
    }
}

template <typename T>
fmx_status launch_t(fmx_ctx *ctx, const fmx_spm *spm, const Plan *plan, int k,
                    const void *X, int64_t ldx, void *Y, int64_t ldy, void *partial,
                    hipStream_t stream, const uint16_t *img, uint32_t item_begin, uint32_t item_end,
                    bool reduce, const double *rscale, uint32_t flags, const void *Xhot, uint64_t nhot)
{
    // integer sums are exact in any order: the sequential mode is the default one
    const bool seq = (flags & FMX_SPMM_SEQ) && std::is_floating_point<T>::value;
    SpmmArgs a;
    a.img = img;
    a.dir = spm->d_dir;
    a.items = plan->d_items + item_begin;
    a.X = X;
    a.Y = Y;
    a.partial = partial;
    a.ldx = ldx;
    a.ldy = ldy;
    a.nitems = item_end - item_begin;
    a.hs = plan->hs;
    // pad band rows by one element to spread the LDS adds over the banks
    static const bool no_pad = getenv("FMX_NO_PAD") != nullptr;  // read once per process
    a.band_stride = (uint32_t)k + ((k >= 4 && !no_pad) ? 1u : 0u);
    a.band_bytes = a.wave_bytes = 0;  // launch_n
    a.log2w = spm->log2w;
    a.k = k;
    a.ncols = spm->ncols;
    a.vdir = spm->esz ? spm->d_vdir : nullptr;
    a.vwords = (int)(spm->esz / 2);
    a.rscale = rscale;
    a.ycol = (flags & FMX_SPMM_Y_COLMAJOR) ? 1 : 0;
    a.round_first = (flags & kSpmmRoundFirst) ? 1 : 0;
    a.low_bands = plan->hs < spm->H;
    a.Xhot = Xhot;
    a.nhot = Xhot ? nhot : 0;
    // 16-byte vector gathers need aligned rows; otherwise the runtime-width path.
    const int vb = (k * (int)sizeof(T) < 16) ? k * (int)sizeof(T) : 16;
    const bool aligned = ((uintptr_t)X % vb == 0) && ((ldx * (int64_t)sizeof(T)) % vb == 0) &&
                         ((uintptr_t)Xhot % vb == 0) && ((k * (int)sizeof(T)) % vb == 0);
    const int kk = aligned ? k : 0;
    fmx_status st;
    if (a.nhot)
        st = launch_w<T, false, true>(ctx, a, kk, spm->prim, stream);  // never with the sequential mode
    else if constexpr (std::is_floating_point<T>::value)
        st = seq ? launch_w<T, true, false>(ctx, a, kk, spm->prim, stream)
                 : launch_w<T, false, false>(ctx, a, kk, spm->prim, stream);
    else
        st = launch_w<T, false, false>(ctx, a, kk, spm->prim, stream);
    if (st) return st;
    if (reduce && plan->nsplits) {
        using A = typename AccOf<T>::type;
        hipLaunchKernelGGL((spmm_reduce<T, A>), dim3(plan->nsplits, (plan->hs * (uint32_t)k + 255) / 256), dim3(256), 0, stream,
                           plan->d_splits, (const A *)partial, plan->hs, (uint32_t)k, (T *)Y, ldy, rscale, a.ycol,
                           a.round_first);
        FMX_HIP(ctx, hipGetLastError());
    }
    return FMX_OK;
}

}  // namespace

// Row-major copies of a dense operand, optionally scaled by pre[i] per row
// (one rounding): out[i * k + j] = X(i, j) * pre[i].  Both are bound by the
// copy's bytes.
//
// A column-major X goes through LDS, 128 rows by up to 32 columns at a time:
// every thread reads down its row's columns (all in flight before the first is
// stored), and the rows are written as one run.  700,001 x 10 FP32: 12 us
// (4.5 TB/s), 20 with a lane for each of 32 columns whether X has them or not.
template <typename T>
__global__ void __launch_bounds__(256) stage_cols(const T *X, int64_t ldx, const double *pre, uint64_t n, uint32_t k,
                                                  T *out)
{
    constexpr int kR = 128, kC = 32;
    __shared__ T tile[kC][kR + 1];
    const uint64_t r0 = (uint64_t)blockIdx.x * kR;
    const uint32_t c0 = blockIdx.y * kC, w = min((uint32_t)kC, k - c0), tid = threadIdx.x;
    const uint32_t rows = (uint32_t)min((uint64_t)kR, n - r0), r = tid % kR, h = tid / kR;
    T v[kC / 2];
#pragma unroll
    for (uint32_t j = 0; j < kC / 2; j++)
        if (2 * j + h < w && r < rows) v[j] = X[(c0 + 2 * j + h) * (uint64_t)ldx + r0 + r];
    [[maybe_unused]] const double p = pre && r < rows ? pre[r0 + r] : 1.0;
#pragma unroll
    for (uint32_t j = 0; j < kC / 2; j++)
        if (2 * j + h < w && r < rows) {
            if constexpr (std::is_floating_point<T>::value)
                if (pre) v[j] = (T)((double)v[j] * p);
            tile[2 * j + h][r] = v[j];
        }
    __syncthreads();
    for (uint32_t e = tid; e < rows * w; e += 256) {
        const uint32_t rr = e / w, c = e - rr * w;
        out[(r0 + rr) * k + c0 + c] = tile[c][rr];
    }
}

// A scaled row-major X: V elements a thread, 16 bytes where rows, stride and
// base allow (260,000 x 16 FP32: 8 us, 13.5 one element at a time with a lane
// for each of 32 columns).
template <typename T, int V>
__global__ void __launch_bounds__(256) stage_rows(const T *X, int64_t ldx, const double *pre, uint64_t n, uint32_t k,
                                                  T *out)
{
    struct alignas(V * sizeof(T)) Piece {
        T v[V];
    };
    const uint32_t kv = k / V;
    const uint64_t tot = n * kv;
    for (uint64_t e = blockIdx.x * 256ull + threadIdx.x; e < tot; e += (uint64_t)gridDim.x * 256) {
        const uint64_t i = tot >> 32 ? e / kv : (uint32_t)e / kv;
        Piece q = *(const Piece *)(X + i * ldx + (e - i * kv) * V);
        const double p = pre[i];
#pragma unroll
        for (int j = 0; j < V; j++) q.v[j] = (T)((double)q.v[j] * p);
        *(Piece *)(out + e * V) = q;
    }
}

template <typename T>
fmx_status stage_typed(fmx_ctx *ctx, uint64_t n, int k, const void *X, int64_t ldx, bool xcol, const double *pre,
                       void *out, hipStream_t stream)
{
    if (xcol) {
        const dim3 grid((unsigned)((n + 127) / 128), (unsigned)((k + 31) / 32));
        hipLaunchKernelGGL(stage_cols<T>, grid, dim3(256), 0, stream, (const T *)X, ldx, pre, n, (uint32_t)k, (T *)out);
    } else if constexpr (std::is_floating_point<T>::value) {
        constexpr int kV = 16 / sizeof(T);
        const bool wide = k % kV == 0 && ldx % kV == 0 && (uintptr_t)X % 16 == 0;
        const uint64_t pieces = n * (uint64_t)(wide ? k / kV : k);
        const dim3 grid((unsigned)std::min<uint64_t>((pieces + 255) / 256, (uint64_t)ctx->num_cus * 64));
        if (wide)
            hipLaunchKernelGGL((stage_rows<T, kV>), grid, dim3(256), 0, stream, (const T *)X, ldx, pre, n, (uint32_t)k,
                               (T *)out);
        else
            hipLaunchKernelGGL((stage_rows<T, 1>), grid, dim3(256), 0, stream, (const T *)X, ldx, pre, n, (uint32_t)k,
                               (T *)out);
    }
    FMX_HIP(ctx, hipGetLastError());
    return FMX_OK;
}

// (only a column-major or a scaled X is restaged, and only floating-point
// data is scaled)
fmx_status stage_dense_rows(fmx_ctx *ctx, fmx_dtype dt, uint64_t n, int k, const void *X, int64_t ldx, bool xcol,
                            const double *pre, void *out, hipStream_t stream)
{
    if (n == 0) return FMX_OK;
    switch (dt) {
    case FMX_I32: return stage_typed<int32_t>(ctx, n, k, X, ldx, xcol, nullptr, out, stream);
    case FMX_I64:
    case FMX_U64: return stage_typed<int64_t>(ctx, n, k, X, ldx, xcol, nullptr, out, stream);
    case FMX_F32: return stage_typed<float>(ctx, n, k, X, ldx, xcol, pre, out, stream);
    case FMX_F64: return stage_typed<double>(ctx, n, k, X, ldx, xcol, pre, out, stream);
    default: return fail(ctx, FMX_ETYPE, "wrong matrix type in spmm");
    }
}

// out[i][0..k) = X[hot[i]][0..k): rows of V-sized pieces, a row's pieces on
// consecutive lanes.
template <typename V>
__global__ void __launch_bounds__(256) stage_hot(const V *X, uint64_t ldx_v, const uint32_t *hot, uint64_t nhot,
                                                  uint32_t kv, V *out)
{
    const uint64_t tot = nhot * kv;
    for (uint64_t e = blockIdx.x * 256ull + threadIdx.x; e < tot; e += (uint64_t)gridDim.x * 256) {
        const uint64_t i = e / kv, j = e - i * kv;
        out[e] = X[(uint64_t)hot[i] * ldx_v + j];
    }
}

fmx_status stage_hot_rows(fmx_ctx *ctx, fmx_dtype dt, uint64_t nhot, int k, const void *X, int64_t ldx,
                          const uint32_t *hot, void *out, hipStream_t stream)
{
    if (nhot == 0) return FMX_OK;
    const uint64_t rb = (uint64_t)k * elem_size(dt), lb = (uint64_t)ldx * elem_size(dt);
    const uint64_t blocks = std::min<uint64_t>((nhot * k + 255) / 256, (uint64_t)ctx->num_cus * 32);
    // the widest piece that divides the row, the stride and the base
    if (rb % 16 == 0 && lb % 16 == 0 && (uintptr_t)X % 16 == 0)
        hipLaunchKernelGGL(stage_hot<uint4>, dim3((unsigned)blocks), dim3(256), 0, stream, (const uint4 *)X, lb / 16,
                           hot, nhot, (uint32_t)(rb / 16), (uint4 *)out);
    else if (rb % 8 == 0 && lb % 8 == 0 && (uintptr_t)X % 8 == 0)
        hipLaunchKernelGGL(stage_hot<uint2>, dim3((unsigned)blocks), dim3(256), 0, stream, (const uint2 *)X, lb / 8,
                           hot, nhot, (uint32_t)(rb / 8), (uint2 *)out);
    else
        hipLaunchKernelGGL(stage_hot<uint32_t>, dim3((unsigned)blocks), dim3(256), 0, stream, (const uint32_t *)X,
                           lb / 4, hot, nhot, (uint32_t)(rb / 4), (uint32_t *)out);
    FMX_HIP(ctx, hipGetLastError());
    return FMX_OK;
}

fmx_status launch_spmm(fmx_ctx *ctx, const fmx_spm *spm, const Plan *plan, fmx_dtype dt,
                       int k, const void *X, int64_t ldx, void *Y, int64_t ldy,
                       void *partial, hipStream_t stream, const uint16_t *img,
                       uint32_t ib, uint32_t ie, bool reduce, const double *rscale, uint32_t flags,
                       const void *Xhot, uint64_t nhot)
{
    if (rscale && dt != FMX_F32 && dt != FMX_F64) return fail(ctx, FMX_ETYPE, "row scaling needs FP data");
    switch (dt) {
    case FMX_I32: return launch_t<int32_t>(ctx, spm, plan, k, X, ldx, Y, ldy, partial, stream, img, ib, ie, reduce, rscale, flags, Xhot, nhot);
    // size_t sums wrap exactly as long sums do: one kernel serves both
    case FMX_I64:
    case FMX_U64: return launch_t<int64_t>(ctx, spm, plan, k, X, ldx, Y, ldy, partial, stream, img, ib, ie, reduce, rscale, flags, Xhot, nhot);
    case FMX_F32: return launch_t<float>(ctx, spm, plan, k, X, ldx, Y, ldy, partial, stream, img, ib, ie, reduce, rscale, flags, Xhot, nhot);
    case FMX_F64: return launch_t<double>(ctx, spm, plan, k, X, ldx, Y, ldy, partial, stream, img, ib, ie, reduce, rscale, flags, Xhot, nhot);
    default: return fail(ctx, FMX_ETYPE, "wrong matrix type in spmm");
    }
}

}  // namespace fmx
