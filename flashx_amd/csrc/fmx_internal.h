// fmx_internal.h -- shared host/device declarations of libfmx.
//
// Layout of a matrix in HBM:
//   image    : the reference-format tile image, byte for byte (4096-byte
//              header + block rows; matrix/sparse_matrix_format.h:213-240).
//   dir      : one {start, bc} pair per stored tile, in image order; `start`
//              is the tile's first u16 word relative to its block row.
//   plans    : per sub-band height Hs, a list of work items (contiguous word
//              ranges of one block row) and the partial-band reduction list.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <map>
#include <memory>
#include <string>
#include <thread>
#include <utility>
#include <vector>

#include "../../include/fmx.h"

namespace fmx {

constexpr uint32_t kNone = 0xFFFFFFFFu;
constexpr uint64_t kHeaderBytes = 4096;

// One unit of SpMM work: words [begin, begin+nwords) of a block row, whose
// non-zeros with tile-relative rows in [sb_base, sb_base + rows) accumulate
// into one LDS band.  `carry` is the tile-relative row in force at `begin`
// when the range starts inside a row part (kNone otherwise).
struct Item {
    uint64_t brow_word;   // absolute u16 index of the block row's first word
    uint32_t begin;       // first word, relative to the block row
    uint32_t nwords;
    uint32_t dir_begin;   // directory index of the tile holding `begin`
    uint32_t dir_end;     // one past the block row's last directory entry
    uint32_t row0_lo;     // first output row of the band (low / high 32 bits)
    uint32_t row0_hi;
    uint32_t sb_base;     // tile-relative row of band row 0
    uint32_t rows;        // rows in the band
    uint32_t carry;
    uint32_t slot;        // partial-band slot, kNone = write Y directly
    uint32_t rot_begin;   // the item is processed from this word (a tile start, or begin) ...
    uint32_t rot_dir;     // ... whose directory index this is, to its end, then from begin
    uint32_t before;      // weighted: entries of the tile holding `begin` that lie before it
    uint32_t pad;
};
static_assert(sizeof(Item) == 64, "Item layout");

// A band split over several items: Y rows [row0, row0+rows) are the ordered
// sum of partial slots [slot_begin, slot_begin+nslots).
struct Split {
    uint64_t row0;
    uint32_t rows;
    uint32_t slot_begin;
    uint32_t nslots;
    uint32_t pad;
};
static_assert(sizeof(Split) == 24, "Split layout");

struct Plan {
    uint32_t hs = 0;            // band height (rows)
    uint32_t nitems = 0;
    uint32_t nslots = 0;
    uint32_t nsplits = 0;
    Item *d_items = nullptr;
    Split *d_splits = nullptr;  // in d_items' allocation
    // streamed matrices: the items of chunk c are [chunk_items[c], chunk_items[c+1])
    std::vector<uint32_t> chunk_items;
    ~Plan();
};

// Device blocks of constructions (inside a BlockScope), kept for reuse: a
// build makes and drops some hundred buffers, and hipMalloc + hipFree take
// 25 us from 4 MB and 360 us from 256 MB (a build of 16.8 M edges spent 11 of
// its 16.5 ms in them).  Everything that uses them runs on the context's
// stream, so a block may be handed on while kernels that use it are still
// queued.  While a scope is open every block is kept, and kRest bytes when it
// is closed: first the blocks that the latest build did not use go back, then
// its largest.  All of them go back when one of the library's allocations
// fails, with fmx_ctx_trim and with the context, which one host thread uses at
// a time.  kRest is what other allocators of the process (torch's) have to do
// without; 2 GB (8 GB: 13.0 ms at 2^26 edges, none: 17.7) hold what builds of up
// to 2^24 edges use, among blocks of other sizes too: with 1 GB, builds of
// 2^20 vertices, 16 edges each, took 4.5 ms by themselves and 5.0 to 5.9 after
// larger ones, whose blocks they take over.
// Blocks outside a scope are allocated and freed as they come.
class BlockCache {
public:
    ~BlockCache() { trim(0); }
    hipError_t get(size_t bytes, void **p, size_t *got);
    void put(void *p, size_t bytes);
    void trim(size_t most);
    int scopes = 0;
    static constexpr size_t kRest = size_t(2) << 30;

private:
    struct Block {
        size_t bytes;
        void *p;
        uint64_t build;  // that used it last
    };
    std::vector<Block> free_;
    size_t held_ = 0;
    uint64_t build_ = 0;
    friend struct BlockScope;
};

struct BlockScope {
    BlockCache &c;
    explicit BlockScope(BlockCache &cache) : c(cache)
    {
        if (c.scopes++ == 0) c.build_++;
    }
    ~BlockScope() { if (--c.scopes == 0) c.trim(BlockCache::kRest); }
};

// The context's pinned host memory: counts that a kernel writes and the host
// reads, a kernel's error flag, an image's header page, and a staging area
// for small copies.
constexpr size_t kPinnedCounts = 0, kPinnedFlag = 4096, kPinnedHeader = 8192, kPinnedStage = 12288,
                 kPinnedBytes = kPinnedStage + (2 << 20);

// A stream in the order of whose work a buffer may be used again.  The
// handle hipStreamPerThread is another stream in every host thread.
struct StreamKey {
    hipStream_t s = nullptr;
    std::thread::id thread;
    StreamKey() = default;
    explicit StreamKey(hipStream_t stream) : s(stream)
    {
        if (s == hipStreamPerThread) thread = std::this_thread::get_id();
    }
    bool operator==(const StreamKey &o) const { return s == o.s && thread == o.thread; }
};

// Scratch of captured calls: a buffer for each capture, stream in it and
// purpose, allocated for them and shared with nothing else.  Replays may
// overlap any later call and each other, and two streams of one capture are
// branches that run side by side; the captured calls of one stream run in
// order and share.  How long a graph lives is not known (user objects are
// released too early or never on ROCm 7.2), so a buffer lives as long as its
// owner, without which the graph cannot be replayed: the matrix, or for
// dense operations the context.
class GraphScratch {
public:
    GraphScratch() = default;
    GraphScratch(const GraphScratch &) = delete;
    GraphScratch &operator=(const GraphScratch &) = delete;
    ~GraphScratch();
    fmx_status get(fmx_ctx *ctx, const void *purpose, hipStream_t s, unsigned long long graph, size_t bytes,
                   void **out);

private:
    struct Buf {
        const void *purpose;
        StreamKey stream;
        unsigned long long graph;  // hipStreamGetCaptureInfo's id
        void *ptr;
        size_t bytes;
    };
    std::vector<Buf> bufs_;
};

// Scratch of one purpose for calls on several streams: a buffer for each
// stream that uses it, so that calls of one context on different streams do
// not share one.  At most kStreams of them are kept; a further stream takes
// the longest unused one, its work queued behind the call that used it last
// (the device waits, not the host).  A call under stream capture takes its
// buffer from `graphs`.
class StreamScratch {
public:
    // A call's hold on its buffer, to the end of the call that queued the
    // work on it.
    struct Lease {
        void *ptr = nullptr;
        StreamScratch *from = nullptr;
        StreamKey stream;
        Lease() = default;
        Lease(const Lease &) = delete;
        Lease &operator=(const Lease &) = delete;
        ~Lease();
    };
    StreamScratch() = default;
    StreamScratch(const StreamScratch &) = delete;
    StreamScratch &operator=(const StreamScratch &) = delete;
    ~StreamScratch();
    fmx_status get(fmx_ctx *ctx, hipStream_t s, size_t bytes, GraphScratch &graphs, Lease &out);
    void clear();  // the device has finished

private:
    static constexpr size_t kStreams = 4;
    struct Buf {
        StreamKey stream;
        uint64_t used = 0;
        void *ptr = nullptr;
        size_t bytes = 0;
        hipEvent_t last = nullptr;  // behind its last call, if marked
        bool marked = false;
    };
    std::vector<Buf> bufs_;
    uint64_t calls_ = 0;
    bool turns_ = false;  // there were more streams than buffers: calls leave marks
};

constexpr size_t kSharedPartials = size_t(64) << 20;

}  // namespace fmx

struct fmx_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    std::string last_error;
    int num_cus = 0;
    size_t lds_per_block = 0;
    fmx::GraphScratch graphs;   // workspaces of captured dense operations
    fmx::StreamScratch ws;      // dense operations' partials
    fmx::StreamScratch xstage;  // a dense operand restaged row-major / pre-scaled
    fmx::StreamScratch xhot;    // the hot rows of X, densely (gather-order images)
    fmx::StreamScratch partial; // partial bands of split items, to kSharedPartials
    void *noalloc_ws = nullptr;  // this device's copy of the fixed scratch (fmx_gram_noalloc)
    size_t noalloc_bytes = 0;
    void *pinned = nullptr;      // pinned host memory (kPinned*)
    fmx::BlockCache blocks;
};

struct fmx_spm {
    fmx_ctx *ctx = nullptr;
    uint64_t nrows = 0, ncols = 0, nnz = 0, H = 0, W = 0, nbr = 0, nbc = 0;
    uint64_t bytes = 0, esz = 0, ntiles = 0;
    int log2h = 0, log2w = 0, prim = 0;
    uint8_t *d_image = nullptr;         // image in HBM (padded to 4 KiB)
    uint2 *d_dir = nullptr;             // tile directory
    uint32_t *d_vdir = nullptr;         // weighted images: values-region word of each tile
    std::vector<uint8_t> h_image;       // host copy used to build plans (resident matrices)
    std::vector<int64_t> offs;          // block-row byte offsets
    std::vector<uint2> dir;             // host directory (empty for an image built on the device)
    std::vector<uint32_t> vdir;         // weighted images: values-region word (block-row relative)
    std::vector<uint32_t> brow_dir;     // first directory index per block row (+1)
    std::map<uint32_t, std::unique_ptr<fmx::Plan>> plans;
    fmx::StreamScratch partial;         // partial bands of split items, above kSharedPartials
    fmx::GraphScratch graphs;           // all scratch of captured multiplies by this matrix
    // Out-of-core form (d_image == nullptr): the image stays in pinned host
    // memory and every SpMM streams it through two HBM staging buffers in
    // chunks of whole block rows; directory and plans stay in HBM.
    uint8_t *h_pinned = nullptr;        // image, padded with zeros to 4 KiB
    uint64_t h_pinned_len = 0;          // bytes given (file or buffer length)
    std::vector<uint64_t> chunk_br;     // first block row of each chunk, then nbr
    std::vector<uint64_t> chunk_lo, chunk_hi;  // 16-byte aligned byte span of each chunk
    uint8_t *d_stage[2] = {nullptr, nullptr};
    uint64_t stage_bytes = 0;
    hipStream_t copy_stream = nullptr;
    hipEvent_t ev_copied[2] = {nullptr, nullptr};
    hipEvent_t ev_free[2] = {nullptr, nullptr};   // last kernel reading each buffer
    bool free_recorded[2] = {false, false};
    hipEvent_t ev_start = nullptr;
    // Resident images with tiles taller than an SpMM band: the same matrix
    // re-cut into short tiles, which every SpMM runs on (retile.cpp).
    std::unique_ptr<fmx_spm> work;
    // Gather order (hotcols.cpp): the matrix with its nhot most used columns
    // relabelled 0..nhot-1 (hot_ids[i] is the original column of new column
    // i) and every other column c relabelled nhot + c.  Default-mode SpMMs
    // run on it with X's hot rows restaged densely first.
    std::unique_ptr<fmx_spm> fast;
    uint32_t *d_hot = nullptr;
    uint64_t nhot = 0;
    uint64_t build_ns = 0;              // device-built: construction kernels' time
    uint64_t edges_in = 0;              // device-built: edges of the input list
    bool streamed() const { return h_pinned != nullptr; }
    const uint8_t *host_image() const { return h_pinned ? h_pinned : h_image.data(); }
    uint64_t host_bytes() const { return h_pinned ? h_pinned_len : h_image.size(); }
    ~fmx_spm();
};

namespace fmx {

// Records `msg` on the context and returns `st`.
fmx_status fail(fmx_ctx *ctx, fmx_status st, const std::string &msg);
fmx_status hip_fail(fmx_ctx *ctx, hipError_t e, const char *what);
int elem_size(fmx_dtype dt);
// hipMalloc that gives the context's kept blocks back if memory is short.
hipError_t dev_malloc(fmx_ctx *ctx, void **p, size_t bytes);
// Queues a copy of `bytes` bytes of device memory to the context's pinned
// staging area, for pinned_get after the stream has been synchronised; larger
// ones go to dst at once (hipMemcpy's pageable copies of some 100 KB take
// three times as long).
fmx_status pinned_fetch(fmx_ctx *ctx, void *dst, const void *src, size_t bytes, size_t at, hipStream_t s);
void pinned_get(fmx_ctx *ctx, void *dst, size_t bytes, size_t at);

// Validates a host image and fills the matrix fields + directory.
fmx_status analyse_image(fmx_ctx *ctx, fmx_spm *spm);
// Device construction (build_tiles.hip); ncols != 0: an n x ncols matrix;
// internal: a work image of another matrix, whose ids are known to be in
// range and which gets no work images of its own.
fmx_status build_impl(fmx_ctx *ctx, const uint32_t *src, const uint32_t *dst, size_t m, uint64_t n,
                      uint32_t log2_h, uint32_t log2_w, uint32_t flags, const void *vals, uint32_t esz,
                      int32_t prim_type, fmx_spm **out, uint64_t ncols, bool internal);
// The gather-order image of a resident matrix (hotcols.cpp): columns
// relabelled so that the most used ones form a dense front block of X.
// stream_chunk != 0: the image is streamed from pinned host memory in
// chunks of that many bytes, as the matrix it belongs to.
fmx_status prepare_fast(fmx_ctx *ctx, fmx_spm *spm, uint64_t stream_chunk = 0);
// The gather order of ncols columns with the given uses (device; image_dev.hip):
// *newid (device, allocated here) maps a column to its new id, *hot lists the
// nhot columns that cover `permille` of the nnz non-zeros in their new order.
// *nhot = 0 (and nothing allocated) when there are none.  On ctx->stream.
fmx_status rank_columns(fmx_ctx *ctx, const uint32_t *uses, uint64_t ncols, uint64_t nnz, uint64_t permille,
                        uint32_t **newid, uint32_t **hot, uint64_t *nhot);
// The share of the non-zeros that the hot columns of a gather-order image
// cover, and its tile height; whether a matrix gets one.
uint64_t hot_permille();
uint32_t fast_log2_rows(const fmx_spm *spm);
bool wants_fast(const fmx_spm *spm);
// The non-zeros of the image in HBM of src (image_dev.hip) in stream order
// into device lists rows, cols (relabelled into gather order) and vals (esz
// bytes each, if weighted); *hot (device, allocated here) lists the nhot
// columns that cover `permille` of the non-zeros, in their new order.
// *nhot = 0 (and nothing allocated) when there are none.
fmx_status gather_order_lists(fmx_ctx *ctx, const fmx_spm *src, uint64_t ncols, uint64_t permille,
                              uint32_t *rows, uint32_t *cols, void *vals, uint32_t **hot, uint64_t *nhot);
// The non-zeros of the image in HBM of src in stream order into device lists
// rows, cols and vals (esz bytes each, if weighted); uses (ncols counters,
// zeroed by the caller, or NULL) counts each column's non-zeros
// (image_dev.hip).
fmx_status decode_lists(fmx_ctx *ctx, const fmx_spm *src, uint32_t *rows, uint32_t *cols, void *vals,
                        uint32_t *uses);
// The split items among the n device items of an image built on the device:
// their ranges' ends move out of tile headers (binary) or to their share of
// a tile's entries (weighted), and dir_begin, carry, before (weighted) and the
// rotation fields are filled in (image_dev.hip).  Sets the flag in ctx->pinned if an item is
// inconsistent; on ctx->stream, not synchronised.
fmx_status plan_cuts(fmx_ctx *ctx, const fmx_spm *s, Item *items, uint32_t n);
fmx_status finish_streamed(fmx_ctx *ctx, fmx_spm *s, uint64_t chunk_bytes, bool whole_file);
// The chunks, staging buffers and directory of an analysed streamed image
// (or of its re-cut work image), without a gather-order image.
fmx_status finish_streamed_chunks(fmx_ctx *ctx, fmx_spm *s, uint64_t chunk_bytes);
fmx_status alloc_pinned(fmx_ctx *ctx, fmx_spm *s, uint64_t len);
// The work image of a resident matrix with tiles taller than the work
// tile height (retile.cpp): built, validated and uploaded into spm->work.
fmx_status prepare_work(fmx_ctx *ctx, fmx_spm *spm);
uint32_t work_rows_for(const fmx_spm *spm);
void retile_image(const fmx_spm *spm, uint32_t h2, std::vector<uint8_t> &img, std::vector<int64_t> &offs);
// Builds (or fetches) the work plan for band height hs.  An ordered plan
// neither splits nor rotates items, so every band is one item walked from
// its first word (the sequential mode needs this).
fmx_status get_plan(fmx_ctx *ctx, fmx_spm *spm, uint32_t hs, bool ordered, Plan **out);
// Band height for element size s and width k.
uint32_t band_rows(const fmx_spm *spm, int k, int s);

// launch_spmm's flag beside FMX_SPMM_*: spmm_exec's round_first.
constexpr uint32_t kSpmmRoundFirst = 1u << 31;

// Launches the SpMM kernel over plan items [item_begin, item_end) with the
// image at img (absolute u16 word w of the image is img[w]) and, if reduce,
// the in-order reduction of the plan's split bands.  flags: the kernels' part of the FMX_SPMM_* flags (FMX_SPMM_SEQ, FMX_SPMM_Y_COLMAJOR).
// Columns below nhot are read from Xhot (nhot x k, leading dimension k),
// column c >= nhot from row c - nhot of X.
fmx_status launch_spmm(fmx_ctx *ctx, const fmx_spm *spm, const Plan *plan,
                       fmx_dtype dt, int k, const void *X, int64_t ldx,
                       void *Y, int64_t ldy, void *partial,
                       hipStream_t stream, const uint16_t *img,
                       uint32_t item_begin, uint32_t item_end, bool reduce,
                       const double *rscale, uint32_t flags, const void *Xhot = nullptr,
                       uint64_t nhot = 0);
// out[i][0..k) = X[hot[i]][0..k) for i < nhot (out has leading dimension k).
fmx_status stage_hot_rows(fmx_ctx *ctx, fmx_dtype dt, uint64_t nhot, int k, const void *X, int64_t ldx,
                          const uint32_t *hot, void *out, hipStream_t stream);

// out (n x k, row-major, leading dimension k) = X, read row- or column-major
// (xcol), times pre[i] per row when pre is given (FP data only).
fmx_status stage_dense_rows(fmx_ctx *ctx, fmx_dtype dt, uint64_t n, int k, const void *X, int64_t ldx, bool xcol,
                            const double *pre, void *out, hipStream_t stream);

// Y = diag(post) A diag(pre) X with FMX_SPMM_* flags; pre / post may be null.
// The weighted-value type may differ from dtype only when mixed is set
// (FP64 dense data with FP32 values, spmm_creator<double, float>).
// round_first: a scaled row's sum is rounded to dtype before post multiplies
// it (and rounded again), as a product followed by a row scaling rounds.
fmx_status spmm_exec(fmx_ctx *ctx, const fmx_spm *spm, fmx_dtype dtype, int k, const double *pre,
                     const double *post, const void *X, int64_t ldx, void *Y, int64_t ldy, uint32_t flags,
                     bool mixed, hipStream_t s, bool round_first = false);

}  // namespace fmx

#define FMX_HIP(ctx, call)                                            \
    do {                                                              \
        hipError_t e_ = (call);                                       \
        if (e_ != hipSuccess) return fmx::hip_fail((ctx), e_, #call); \
    } while (0)
