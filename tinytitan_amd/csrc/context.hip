// Context, error reporting, timing and the three attention entry points of the C ABI.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <new>

#include "chunk_plan.h"
#include "internal.h"

// Split-K partials of tt_hip_attn_decode_noalloc, the entry point for callers that cannot allocate: a fixed
// array in the library's own device image instead of the context's grown-on-demand buffers.  Every GPU the
// library runs on holds its own copy (33 MiB) at its own address until the process ends; host code reaches it
// only through the address hipGetSymbolAddress returns on that device (kept per context), never by this name.
// Layout: [kStaticPartialRows][256] floats of unnormalised O, then [kStaticPartialRows][2] floats of (max, sum).
static __device__ __align__(256) float scratch[tt::kStaticPartialRows * (256 + 2)];

namespace tt {

int hip_fail(tt_hip_ctx *ctx, hipError_t err, const char *what) {
    if (ctx) {
        ctx->last_hip_error = std::string(what) + ": " + hipGetErrorString(err);
    }
    (void)hipGetLastError();  // clear the sticky per-thread error
    return err == hipErrorOutOfMemory ? TT_HIP_ERR_OUT_OF_MEMORY : TT_HIP_ERR_HIP;
}

int ensure_partials(tt_hip_ctx *ctx, size_t rows, int head_dim) {
    // Sized for head_dim 256 so that a context serves every supported head_dim.
    (void)head_dim;
    if (rows <= ctx->part_rows) return TT_HIP_OK;
    if (ctx->capturing) return TT_HIP_ERR_BUSY;  // growing would synchronise and allocate inside a capture
    hipError_t e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, e, "hipStreamSynchronize");
    if (ctx->part_o) (void)hipFree(ctx->part_o);
    if (ctx->part_ml) (void)hipFree(ctx->part_ml);
    ctx->part_o = nullptr;
    ctx->part_ml = nullptr;
    ctx->part_rows = 0;
    ++ctx->generation;
    size_t want = rows + rows / 4;
    e = hipMalloc(reinterpret_cast<void **>(&ctx->part_o), want * 256 * sizeof(float));
    if (e != hipSuccess) return hip_fail(ctx, e, "hipMalloc(split partial O)");
    e = hipMalloc(reinterpret_cast<void **>(&ctx->part_ml), want * 2 * sizeof(float));
    if (e != hipSuccess) {
        (void)hipFree(ctx->part_o);
        ctx->part_o = nullptr;
        return hip_fail(ctx, e, "hipMalloc(split partial m/l)");
    }
    ctx->part_rows = want;
    return TT_HIP_OK;
}

int ensure_stage(tt_hip_ctx *ctx, size_t elems) {
    if (elems <= ctx->stage_elems) return TT_HIP_OK;
    if (ctx->capturing) return TT_HIP_ERR_BUSY;
    hipError_t e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, e, "hipStreamSynchronize");
    if (ctx->stage_k) (void)hipFree(ctx->stage_k);
    if (ctx->stage_v) (void)hipFree(ctx->stage_v);
    ctx->stage_k = ctx->stage_v = nullptr;
    ctx->stage_elems = 0;
    ++ctx->generation;
    const size_t want = elems + elems / 4;
    e = hipMalloc(reinterpret_cast<void **>(&ctx->stage_k), want * sizeof(_Float16));
    if (e != hipSuccess) return hip_fail(ctx, e, "hipMalloc(dequantised K pages)");
    e = hipMalloc(reinterpret_cast<void **>(&ctx->stage_v), want * sizeof(_Float16));
    if (e != hipSuccess) {
        (void)hipFree(ctx->stage_k);
        ctx->stage_k = nullptr;
        return hip_fail(ctx, e, "hipMalloc(dequantised V pages)");
    }
    ctx->stage_elems = want;
    return TT_HIP_OK;
}

// Rows of selection bytes for a chunk whose selection arrives as index lists.
static int ensure_keep_rows(tt_hip_ctx *ctx, size_t bytes) {
    if (bytes <= ctx->keep_rows_bytes) return TT_HIP_OK;
    if (ctx->capturing) return TT_HIP_ERR_BUSY;
    hipError_t e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, e, "hipStreamSynchronize");
    if (ctx->keep_rows) (void)hipFree(ctx->keep_rows);
    ctx->keep_rows = nullptr;
    ctx->keep_rows_bytes = 0;
    ++ctx->generation;
    const size_t want = bytes + bytes / 4;
    e = hipMalloc(reinterpret_cast<void **>(&ctx->keep_rows), want);
    if (e != hipSuccess) return hip_fail(ctx, e, "hipMalloc(selection rows)");
    ctx->keep_rows_bytes = want;
    return TT_HIP_OK;
}

// One workgroup per query row: clear the row's bytes, then set the byte of every listed key the row can see
// (key < min(kv_valid, start + row + 1), as the reference's kernel tests each list entry).  The row stride is a
// multiple of 16 bytes.
__global__ __launch_bounds__(256) void keep_rows_from_indices_kernel(uint8_t *rows, unsigned row_stride, const uint32_t *indices,
                                                                     unsigned index_stride, const uint32_t *counts, int start,
                                                                     int kv_valid) {
    const unsigned row = blockIdx.x;
    uint8_t *mine = rows + (size_t)row * row_stride;
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    for (unsigned at = threadIdx.x * 16u; at < row_stride; at += 256u * 16u) *reinterpret_cast<u4 *>(mine + at) = (u4)0u;
    __syncthreads();
    const unsigned limit = (unsigned)min(kv_valid, start + (int)row + 1);
    const unsigned count = min(counts[row], index_stride);
    const uint32_t *list = indices + (size_t)row * index_stride;
    for (unsigned i = threadIdx.x; i < count; i += 256u) {
        const unsigned key = list[i];
        if (key < limit) mine[key] = 1;
    }
}

// A chunk's per-query index lists (keepIdx[t * stride + i], i < keepCount[t]; the reference's tiled chunk kernel walks
// them entry by entry, sources/TinyTitanCore/Metal/Prefill/prefill.metal:1069-1117) turned into what a tile of `tt`
// tokens walks here: the ascending list of the 32-key blocks that hold a listed key some token of the tile can see
// (key < min(kv_valid, start + row + 1), the reference's test of each entry), where every key range of `split_blocks`
// blocks starts in that list, per entry the keys of the block that any token keeps (`any_keys`), and per entry and token
// the listed keys, as 32 bits each.  One workgroup per
// token tile; its work is the tile's list entries plus one pass over a bitmap of the context's blocks in LDS (a bit
// per block: 4 KiB per million keys) -- nothing of the order rows x context is written or read.  Entries may come in
// any order and repeat: a bit is set once.
// GROUPS: the same with groups of four keys in the place of blocks: the ascending list of group ids, where the ranges start
// in it, and per eight list positions and token one word, four bits a position.
// LDS: bitmap[W], prefix[W], partial[kPlanThreads + 1], chunk[chunk_entries * (tt | 1)] words, W = ceil(ceil(kv_valid / 32) / 32)
// (GROUPS: ceil(ceil(kv_valid / 4) / 32), and an entry is eight positions).
constexpr int kPlanThreads = 1024;  // sixteen wavefronts: the walks are chains of dependent scalar work that only other wavefronts hide
constexpr int kPlanGroupKeys = 400000;  // keys whose groups' bitmap and prefix sums take 25 of the 64 KiB
template <bool GROUPS>
__global__ __launch_bounds__(kPlanThreads) void keep_plan_kernel(const uint32_t *indices, unsigned index_stride, const uint32_t *counts,
                                                                 int start, int q_len, int kv_valid, int tt, int split_blocks,
                                                                 int n_splits, int cap, int chunk_entries, int *ranges, int *blocks,
                                                                 unsigned *bits, bool any_keys) {
    constexpr int T = kPlanThreads, kShift = GROUPS ? 2 : 5;  // keys of a unit: 1 << kShift
    extern __shared__ unsigned plan_lds[];
    const int tile = blockIdx.x, tid = threadIdx.x;
    const int ctx_blocks = (kv_valid + (1 << kShift) - 1) >> kShift, W = (ctx_blocks + 31) >> 5;
    unsigned *bitmap = plan_lds, *prefix = plan_lds + W, *partial = plan_lds + 2 * W;
    const int rows = min(tt, q_len - tile * tt);
    // Every row of the tile has as many threads as the others, every thread a run of `per` neighbouring entries of its row (so
    // that the lanes of a wavefront work on entries far apart, which seldom meet in one word of LDS: the entries of a
    // sorted list that 64 neighbouring lanes hold fall into a handful of words, and their atomics queue up).  A
    // thread's first kHeld entries are asked for at once, beside its row's count and ahead of everything else, and
    // stay in registers for both walks over the lists: one trip to memory for a tile of the usual size.  Entries
    // beyond them are read again per walk, kBatch at a time.  What a tile's workgroup spends its time on is instructions per entry and walk,
    // sixteen wavefronts on four SIMDs: a thread that ran on from one row's list into the next had two dozen, with a place checked for
    // every one it could hold.  128 rows of 16/2 heads with lists of 2,051 cells 11.5 -> 9.2 us, 100 rows of 32/8 17.2 -> 12.4, over 8 bits 12.2 -> 10.2.
    constexpr unsigned kHeld = 18, kBatch = 8;  // (lists of 2,051 cells, tiles of four and of eight tokens: 9 and 17 entries a thread)
    const unsigned row_threads = (unsigned)T / (unsigned)rows, row = min((unsigned)tid / row_threads, (unsigned)rows - 1u);  // (threads over: at the last row's end)
    const unsigned per = (index_stride + row_threads - 1u) / row_threads, mine = ((unsigned)tid - row * row_threads) * per;
    const uint32_t *list = indices + (size_t)(tile * tt + (int)row) * index_stride;
    const unsigned count = min(counts[tile * tt + (int)row], index_stride), limit = (unsigned)min(kv_valid, start + tile * tt + (int)row + 1);
    const unsigned end = min(mine + per, count);
    unsigned held[kHeld];
#pragma unroll
    for (unsigned j = 0; j < kHeld; ++j)
        if (j < per) held[j] = list[min(mine + j, index_stride - 1u)];  // (18 requests of 64 lanes' far apart words where 9 are wanted: 9.4 -> 11.1 us)
    for (int w = tid; w < W; w += T) bitmap[w] = 0u;
    __syncthreads();
    auto for_listed_keys = [&](auto &&use) {  // use(key): every listed key of the thread's that its row can see
        auto place = [&](unsigned j, unsigned key) {
            if (mine + j < end && key < limit) use(key);
        };
#pragma unroll
        for (unsigned j = 0; j < kHeld; ++j) {
            if (j >= per) break;
            place(j, held[j]);
        }
        for (unsigned base = kHeld; base < per; base += kBatch) {
            unsigned keys[kBatch];
#pragma unroll
            for (unsigned j = 0; j < kBatch; ++j) keys[j] = list[min(mine + base + j, index_stride - 1u)];
#pragma unroll
            for (unsigned j = 0; j < kBatch; ++j) place(base + j, keys[j]);
        }
    };
    for_listed_keys([&](unsigned key) { atomicOr(&bitmap[key >> (kShift + 5)], 1u << ((key >> kShift) & 31u)); });
    __syncthreads();
    // exclusive prefix sums of the words' bit counts: a run of words per thread, a scan of the threads' runs inside
    // each wavefront by shuffles, the wavefronts' totals through LDS
    const int per_thread = (W + T - 1) / T, w_begin = tid * per_thread, w_end = min(W, w_begin + per_thread);
    unsigned run = 0;
    for (int w = w_begin; w < w_end; ++w) run += __popc(bitmap[w]);
    unsigned inclusive = run;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned below = __shfl_up(inclusive, off);
        if ((tid & 63) >= off) inclusive += below;
    }
    if ((tid & 63) == 63) partial[tid >> 6] = inclusive;
    __syncthreads();
    unsigned before = 0;
    for (int w = 0; w < (tid >> 6); ++w) before += partial[w];
    if (tid == T - 1) partial[T] = before + inclusive;
    run = before + inclusive - run;
    for (int w = w_begin; w < w_end; ++w) {
        prefix[w] = run;
        run += __popc(bitmap[w]);
    }
    __syncthreads();
    const int n_touched = (int)partial[T];  // at most min(ctx_blocks, listed entries) <= cap
    int *my_blocks = blocks + (size_t)tile * cap * (GROUPS ? 1 : 2);
    for (int w = tid; w < W; w += T) {
        unsigned word = bitmap[w];
        int at = (int)prefix[w];
        while (word) {
            my_blocks[(GROUPS ? 1 : 2) * at++] = w * 32 + (__ffs((int)word) - 1);
            word &= word - 1u;
        }
    }
    for (int s = tid; s <= n_splits; s += T) {
        const long long first = (long long)s * split_blocks * (GROUPS ? 8 : 1);
        int at = n_touched;
        if (first < ctx_blocks) at = (int)(prefix[first >> 5] + __popc(bitmap[first >> 5] & ((1u << (first & 31)) - 1u)));
        ranges[(size_t)tile * (n_splits + 1) + s] = at;
    }
    // The bits, a run of `chunk_entries` list entries at a time: gathered in LDS (atomics there cost a few cycles; in
    // global memory every listed key would be a request of its own to L2, ~8 cycles each and 32 us for a tile's 8,000
    // keys), then written out side by side.
    unsigned *my_bits = bits + (size_t)tile * (GROUPS ? cap >> 3 : cap) * tt;
    const int n_entries = GROUPS ? (n_touched + 7) >> 3 : n_touched;
    unsigned *chunk = plan_lds + 2 * W + T + 1;  // [chunk_entries][pitch]; an odd pitch: a row's entries in all banks
    const int pitch = tt | 1;
    const unsigned per_tt = ((1u << 19) + (unsigned)tt - 1u) / (unsigned)tt;  // i / tt == i * per_tt >> 19 for i < 16,384 and even tt <= 32
    for (int first = 0; first < n_entries; first += chunk_entries) {
        const int here = min(chunk_entries, n_entries - first);
        __syncthreads();  // (the previous run has been written out)
        for (int i = tid; i < here * pitch; i += T) chunk[i] = 0u;
        __syncthreads();
        for_listed_keys([&](unsigned key) {
            const unsigned w = key >> (kShift + 5), bit = (key >> kShift) & 31u;
            const int rank = (int)(prefix[w] + __popc(bitmap[w] & ((1u << bit) - 1u)));
            const int entry = (GROUPS ? rank >> 3 : rank) - first;
            const unsigned at = GROUPS ? 4u * ((unsigned)rank & 7u) + (key & 3u) : key & 31u;
            if (entry >= 0 && entry < here) atomicOr(&chunk[entry * pitch + (int)row], 1u << at);
        });
        __syncthreads();
        for (int i = tid; i < here * tt; i += T) my_bits[(size_t)first * tt + i] = chunk[i + (int)((unsigned)i * per_tt >> 19) * (pitch - tt)];
        if (GROUPS || !any_keys) continue;
        for (int i = tid; i < here; i += T) {
            unsigned any = 0u;
            for (int r = 0; r < tt; ++r) any |= chunk[i * pitch + r];
            my_blocks[2 * (first + i) + 1] = (int)any;
        }
    }
}

// A plain streaming read, the control the decode pass is measured against: one workgroup per CU walks its own
// contiguous share, every thread keeping 16 loads of 16 bytes in flight (64 KiB per workgroup and turn), and
// folds what it read into one word that is stored only if it equals a value it cannot have.
typedef unsigned u4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void calibrate_read_kernel(const u4 *src, unsigned turns, unsigned *sink) {
    const u4 *p = src + (size_t)blockIdx.x * turns * 4096 + threadIdx.x;
    u4 acc = {0u, 0u, 0u, 0u};
    for (unsigned t = 0; t < turns; ++t) {
        u4 x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = __builtin_nontemporal_load(p + (size_t)t * 4096 + i * 256);
#pragma unroll
        for (int i = 0; i < 16; ++i) acc ^= x[i];
    }
    const unsigned folded = acc[0] ^ acc[1] ^ acc[2] ^ acc[3];
    if (folded == 0x9e3779b9u && sink) sink[0] = folded + threadIdx.x;  // practically never: keeps the loads alive
}

static bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// A per-call table of one int per sequence: on the stack for the batch sizes a step has (the decode entry points
// are called once per layer and token and should not touch the heap), on the heap beyond that.
struct IntTable {
    explicit IntTable(int n) {
        if (n > kInline) {
            heap.resize((size_t)n);
            ints = heap.data();
        }
    }
    int *data() { return ints; }
    int &operator[](int i) { return ints[i]; }

private:
    static constexpr int kInline = 64;
    int inline_ints[kInline];
    std::vector<int> heap;
    int *ints = inline_ints;
};

// A chunk's selection as per-query index lists (one sequence): indices[row * stride + i], i < counts[row].
struct KeepLists {
    const uint32_t *indices;
    size_t stride;
    const uint32_t *counts;
};

// Shared body of decode / verify / prefill.
//   kind 0: rows query tokens per sequence, GQA-packed tiles, split-K.
//   kind 1: causal chunk of one sequence.
//   chunk_splits > 1 (kind 1, one sequence): the chunk kernel over chunk_splits key ranges of
//   chunk_split_blocks blocks, then the combine pass.
static int run_attention(tt_hip_ctx *ctx, tt_hip_kv *kv, int kind, int layer, int n_seq, const int *slots,
                         const int *starts, const int *totals, int rows, int n_q_heads, const tt_half *q,
                         long long q_seq_stride, long long q_tok_stride, const tt_half *gate, long long g_seq_stride,
                         long long g_tok_stride, float scale, tt_half *out, long long o_seq_stride,
                         long long o_tok_stride, int chunk_splits = 1, int chunk_split_blocks = 0,
                         const PageSource *pages = nullptr, int window = 0, const uint8_t *keep = nullptr,
                         long long keep_seq_stride = 0, long long keep_row_stride = 0, bool static_partials = false,
                         const KeepLists *lists = nullptr) {
    const int D = kv->head_dim;
    hipError_t e = hipSetDevice(ctx->device);
    if (e != hipSuccess) return hip_fail(ctx, e, "hipSetDevice");
    for (int base = 0; base < n_seq; base += kMaxSeqPerLaunch) {
        const int n = n_seq - base < kMaxSeqPerLaunch ? n_seq - base : kMaxSeqPerLaunch;
        long long total_keys = 0;
        int max_keys = 0, min_keys = totals[base];
        // Keys a tile walks: all of them, or with a sliding window at most the window, the tile's
        // rows and the partial block in front.
        auto walked = [&](int i) {
            const long long reach = (long long)window + rows + 32;
            return window > 0 && totals[base + i] > reach ? (int)reach : totals[base + i];
        };
        min_keys = walked(0);
        for (int i = 0; i < n; ++i) {
            total_keys += walked(i);
            if (walked(i) > max_keys) max_keys = walked(i);
            if (walked(i) < min_keys) min_keys = walked(i);
        }
        LaunchPlan plan{};
        // Lists over quantised pages that the caller has had dequantised: the split-K kernel walks those pages.
        const bool walks_pages = lists && pages;
        const int kv_bits = walks_pages ? 16 : kv->bits;
        const bool small_tiles_ok = kind == 0 && !keep && !lists && chunk_splits <= 1 && !pages;
        int st = plan_launch(ctx, kind, n, n_q_heads, kv->n_kv_heads, D, rows, total_keys, min_keys, max_keys, &plan, kv_bits,
                             small_tiles_ok);
        if (st != TT_HIP_OK) return st;
        if (chunk_splits > 1) {  // the chunk kernel's geometry: 32-row one-head tiles, its own key ranges
            // (a tile that walked past the launched ranges would lose keys, and the combine pass would count a partial result more)
            if (longest_tile_blocks(starts[base], rows, totals[base], window) > (long long)chunk_splits * chunk_split_blocks)
                return TT_HIP_ERR_SHAPE;
            plan.split_len = chunk_split_blocks * 32;
            plan.n_splits_max = chunk_splits;
        }
        // The plan of a launch over lists (its layout: below).
        bool groups = false;
        int cap = 0, ctx_units = 0;
        size_t n_blocks = 0, n_bits = 0;
        if (lists) {
            // Groups of four keys instead of blocks of 32 (fp16 pages, tiles of 32 rows): a turn of the walk then takes eight
            // listed groups instead of one touched block, of which a selection in blocks of four leaves 1.3 to 2 groups
            // wanted at 32k keys and more (one row's list of 2,051 cells each): 128 rows of 16/2 heads of 256 behind 16k keys 74.0 ->
            // 55 us, 32k 101.3 -> 59.6, 131k 163.0 -> 80.7.
            // Where the tile's lists could hold most of the keys, most of a block is wanted and its loads are the better ones.
            // Heads of 256, whose groups lie in lines of their own (kv_layout.h): as long as the lists hold no more than eight
            // ninths of the keys, from 3,200 keys on (by blocks / by groups: 24/2 heads, 300 rows behind 4,500 keys 130 / 126 us, 512
            // behind 9,000 226 / 150, behind 64,000 593 / 212, 40/2 heads, 512 behind 3,500 209 / 185, behind 2,500 171 / 182).  With fewer
            // keys as long as they hold no more than half of them (lists of 256 keys, 24/2 heads, 300 rows behind 2,700 keys 78.7 / 49.1,
            // 128 rows 39.5 / 30.0; of 32 keys, 8/2 heads, 512 rows behind 1,800 38.5 / 28.8; all rows with one list of 64, 16/2 heads, 64
            // rows behind 2,700 26.1 / 27.3).
            // Narrower heads: half of the keys (8k keys, 512 rows: 121.7 against 133.4 us), and a bound on the tiles: many share
            // fetched lines in L2 only while they stay side by side, which the walk over blocks does better (inside the bound 512 rows of
            // heads of 64 behind 131k keys 470 -> 208 us).  The group bitmap has to leave the plan kernel's LDS room for a run of bits.
            const long long entries = (long long)plan.tt * (long long)lists->stride;
            groups = kv_bits == 16 && plan.nt == 32 && totals[base] <= kPlanGroupKeys &&
                     (D == 256 ? 2 * entries <= totals[base] || (9 * entries <= 8ll * totals[base] && totals[base] >= 3200)
                               : 2 * entries <= totals[base] && (long long)plan.n_tiles * D <= 128ll * ctx->n_cus);
            const int unit = groups ? 4 : 32;
            ctx_units = (totals[base] + unit - 1) / unit;
            cap = (int)(entries < ctx_units ? entries : ctx_units);
            if (cap < 1) cap = 1;
            if (groups) cap = (cap + 7) & ~7;
            n_blocks = (size_t)plan.tok_tiles * cap * (groups ? 1 : 2);
            n_bits = (size_t)plan.tok_tiles * (groups ? cap >> 3 : cap) * plan.tt;
        }
        auto list_ranges = [&](int splits) { return ((size_t)plan.tok_tiles * (splits + 1) + 1) & ~(size_t)1; };
        auto list_plan_words = [&](int splits) { return list_ranges(splits) + n_blocks + n_bits; };
        // Lists in tiles of 32 rows: a workgroup has a CU to itself, and the planner's splits -- as many per tile as one round of
        // workgroups holds -- leave CUs idle where the tiles do not divide them: 362 tiles take two rounds, the second of them
        // less than half full, 150 tiles one on 150 CUs.  More splits per tile, over whole rounds, are counted out in keys'
        // worth of walking: a round costs a split's keys and its start and merge, 2 D; a split 13 ns (at D = 256) of partial results
        // written and read, 1.3 keys; a combine that was not there 800.  Up to ten rounds (84 MB of partial results), and
        // a sixteenth better than fewer splits.  16/2 heads of 256, 300 rows behind 30k keys (150 tiles, 1 split -> 3) 273 -> 208 us,
        // over 8 bits 291 -> 224, 180 rows behind 100k (90 tiles, 2 -> 5) 182 -> 163; 24/2 heads, 361 rows behind 13k (362 tiles, 1 -> 2)
        // 293 -> 253, 300 behind 40k (1 -> 3) 511 -> 375; 32/8 of 128, 300 behind 30k (304 tiles, 1 -> 3) 341 -> 245; 16/4 of 64, 300 behind
        // 20k (152 tiles, 1 -> 5) 150 -> 77.  Left alone where it would lose: 400 rows behind 8k keys (200 tiles) 117 against 131 and more;
        // and where there are more than two tiles a CU and a tile walks less than 8192 keys of 64 dims: a CU has several of those at
        // work at once, so that rounds are not waited for (64/8 of 64, 640 tiles: 319 rows behind 4,508 keys 72.9 us -> 79.8 in
        // two splits, behind 6,064 88.9 -> 92.5, behind 9,001 119.4 -> 118.0; 320 tiles: 158 rows behind 5,324 66.3 -> 59.5).
        const bool several_at_work = plan.n_tiles > 2 * ctx->n_cus && (long long)max_keys * D < 8192 * 64;
        if (lists && plan.nt == 32 && ctx->split_override <= 0 && plan.n_splits_max >= 1 && max_keys > 384 && !several_at_work) {
            auto rounds = [&](long long splits) { return (plan.n_tiles * splits + ctx->n_cus - 1) / ctx->n_cus; };
            auto length = [&](int splits) { return ((max_keys + splits - 1) / splits + 127) / 128 * 128; };
            auto cost = [&](int splits) {
                const double merge = splits > 1 ? 800.0 + 1.3 * D / 256 * plan.n_tiles * splits : 0.0;
                return (double)rounds(splits) * (length(splits) + 2 * D) + merge;
            };
            const int before = plan.n_splits_max;
            int best = before;
            for (int splits = before + 1; splits <= before + 8 && rounds(splits) <= 10; ++splits) {
                const size_t part_rows = (size_t)plan.n_tiles * splits * plan.nt;
                // (inside a capture nothing can grow: the planner's splits)
                if (ctx->capturing && (part_rows > ctx->part_rows || list_plan_words(splits) * sizeof(int) > ctx->keep_rows_bytes)) break;
                if (cost(splits) < cost(best) * (15.0 / 16.0)) best = splits;
            }
            if (best > before) {
                plan.split_len = length(best);
                plan.n_splits_max = (max_keys + plan.split_len - 1) / plan.split_len;
                plan.workgroups = (long long)plan.n_splits_max * plan.n_tiles;
            }
        }
        // Unlike lengths: the split length that makes the launch whole rounds of at most n_cus workgroups, counted with every
        // sequence's short last split -- the planner's estimate does not know those, and a workgroup over a round waits for a
        // whole one.  k workgroups a CU take len keys each at a k-th of the memory's rate, or at their own where k are too
        // few to keep it busy (one workgroup of heads of 256, two of 128, four of 64), and 32,768 / D keys' worth of start,
        // merge and partial results each.  32 decode rows of 16/2 heads of 256 behind 511 .. 16,383 keys 67.5 -> 49.6 us, 4
        // verify rows x 6 sequences behind 5,000 .. 30,000 keys 58.6 -> 39.1, 20 decode rows over 8 bits 53.8 -> 47.8, 24 of
        // 32/8 heads of 128 40.1 -> 37.8.  Never shorter splits than the planner's, whose partial results have a bound.
        const bool ragged = kind == 0 && chunk_splits <= 1 && min_keys != max_keys && plan.n_splits_max > 1;
        if (ragged && ctx->split_override <= 0) {
            const long long sat = 256 / D, tails = (long long)n * plan.n_tiles;
            long long best = 0;
            int best_len = 0;
            for (long long k = 1; k <= plan.slots_per_cu * 2; ++k) {
                const long long most = k * ctx->n_cus;
                // (mostly last splits: the planner's rule; 40 sequences behind 30 .. 3,000 keys, 32/8 heads of 128: 26.6 us against 29.3)
                if (3 * tails > most) continue;
                // (a last split is short by half on average)
                long long len = ((total_keys * plan.n_tiles) / (most - tails / 2) + 127) / 128 * 128;
                if (len < 128) len = 128;
                auto workgroups = [&] {
                    int w = 0;
                    for (int i = 0; i < n; ++i) w += std::max((walked(i) + (int)len - 1) / (int)len, 1);
                    return (long long)w * plan.n_tiles;
                };
                while (workgroups() > most) len += std::max(128ll, len / 16 / 128 * 128);
                const long long cost = len * std::max(k, sat) + k * (32768 / D);
                if (best_len == 0 || cost < best) {
                    best = cost;
                    best_len = (int)len;
                }
            }
            if (best_len > plan.split_len) {
                plan.split_len = best_len;
                plan.n_splits_max = (max_keys + best_len - 1) / best_len;
                plan.workgroups = (long long)plan.n_splits_max * plan.n_tiles * n;
            }
        }
        // One selection per sequence: a wavefront keeps the blocks it still has to work on as one 64-bit word, at
        // most 64 per split.  One per query row: as a list, of at most kKeepWindows such words.
        const int keep_blocks = keep_row_stride > 0 ? 64 * kKeepWindows : 64;
        if (keep && plan.split_len > keep_blocks * plan.waves * 32) {
            plan.split_len = keep_blocks * plan.waves * 32;
            plan.n_splits_max = (max_keys + plan.split_len - 1) / plan.split_len;
            plan.workgroups = (long long)plan.n_splits_max * plan.n_tiles * n;
        }
        // A chunk's token tiles over several key ranges: workgroups that share an XCD share the K/V blocks of a range.  Over index lists also with
        // one range: a KV head's tiles, one behind the other on the XCDs, were in all of their L2s (32/8 heads of 128, 256 rows behind 100k keys
        // 644 -> 418 us a sparse layer's step, behind 60k 400 -> 328; 16/2 of 256, 500 rows 418 -> 301 and 291 -> 252).
        plan.xcd_grid = ctx->xcd_grid && chunk_splits <= 1 && plan.tok_tiles > 1 && (plan.n_splits_max > 1 || lists) && !ragged;
        // Pages that the launch reads once -- one tile per KV head, as in a decode step or a verify pass of a few
        // rows -- are loaded non-temporal once there are enough of them that they would not survive in the
        // 256 MiB memory-side cache until the same layer's next step anyway (16 MiB a launch: sixteen layers of it).
        {
            const long long kv_bytes = total_keys * (long long)kv->n_kv_heads * (long long)(kv->block_bytes() / kBlockTokens) * 2;
            plan.stream = plan.tok_tiles == 1 && plan.hsubs == 1 && chunk_splits <= 1 && keep_row_stride == 0 &&
                          (ctx->stream_override < 0 ? kv_bytes >= (16ll << 20) : ctx->stream_override != 0);
            // V operands in pairs where every CU has a workgroup of its own for the whole of a long launch, which is then what the memory
            // gives (8 sequences x 4 rows of 16/2 heads behind 64k keys, 1 GiB, 179.0 -> 173.8 us a step; behind 45,678, 0.7 GiB,
            // 121.2 -> 119.7): there the lines asked for early are worth it.  They are not with less to read (one sequence behind 65,540
            // keys plain / paired 32.5 / 35.5 us, 3 behind 100,003 100.9 / 101.7) nor with idle CUs (20 behind 20,010, 240
            // workgroups, 130.1 / 132.7), and least of all where several tiles walk the same keys (8 rows, 5 behind 65,540 132.2 / 141.3).
            plan.paired = plan.stream && plan.workgroups % ctx->n_cus == 0 && kv_bytes >= (640ll << 20);
        }
        // A sequence's splits: what its own keys need (at least one), packed one sequence after the other.
        int first_split[kMaxSeqPerLaunch];
        size_t total_splits = 0;
        for (int i = 0; i < n; ++i) {
            first_split[i] = (int)total_splits;
            const int mine = chunk_splits > 1 ? chunk_splits : (walked(i) + plan.split_len - 1) / plan.split_len;
            total_splits += (size_t)(mine < 1 ? 1 : mine);
        }
        // Unlike lengths: a grid of (splits of the longest, tiles, sequences) would be full of workgroups that find nothing to
        // do, and the others would not fall evenly on the XCDs (a split count of a multiple of eight sends split i of
        // every sequence to XCD i mod 8).
        // A KV head's token tiles read the same keys: rounded up to a multiple of eight, their workgroups of one split meet on
        // one XCD (20 sequences x 3 verify rows in tiles of 16, 300 .. 9,000 keys: 45.2 -> 21.0 us; 8 rows 59.2 -> 26.7).
        // Not where the workgroups of one token tile find a CU each, the idle ones included: finding the sequence is a load more
        // in front of the first key (5 decode rows of 16/4 heads of 64 behind 81 .. 491 keys over 8 bits 6.54 us, packed 6.78; 24 rows
        // of 16/2 of 256 behind 336 .. 433 10.39 / 11.00; two tiles, 3 rows x 2 sequences of 24/2 of 256, 11.94 against 11.32).
        plan.packed_splits = ragged && (plan.workgroups > ctx->n_cus || plan.tok_tiles > 1) ? (int)total_splits : 0;
        if (plan.packed_splits > 0 && plan.tok_tiles > 1) plan.packed_splits = (plan.packed_splits + 7) & ~7;
        if (plan.n_splits_max > 1) {
            const size_t part_rows = total_splits * plan.n_tiles * plan.nt;
            if (static_partials) {
                if (part_rows > kStaticPartialRows) return TT_HIP_ERR_SCRATCH;
            } else {
                st = ensure_partials(ctx, part_rows, D);
                if (st != TT_HIP_OK) return st;
            }
        }
        SplitKArgs a;
        std::memset(&a, 0, sizeof(a));
        SplitKHot &h = a.hot;
        h.k_layer = walks_pages ? pages->k : kv->k[layer];
        h.v_layer = walks_pages ? pages->v : kv->v[layer];
        h.q = reinterpret_cast<const _Float16 *>(q) + base * q_seq_stride;
        a.gate = gate ? reinterpret_cast<const _Float16 *>(gate) + base * g_seq_stride : nullptr;
        a.out = reinterpret_cast<_Float16 *>(out) + base * o_seq_stride;
        h.part_o = static_partials ? ctx->static_scratch : ctx->part_o;
        h.part_ml = static_partials ? ctx->static_scratch + kStaticPartialRows * 256 : ctx->part_ml;
        h.page_elems = walks_pages ? pages->page_elems : (long long)kv->page_elems();
        h.q_seq_stride = q_seq_stride;
        h.q_tok_stride = q_tok_stride;
        a.g_seq_stride = g_seq_stride;
        a.g_tok_stride = g_tok_stride;
        a.o_seq_stride = o_seq_stride;
        a.o_tok_stride = o_tok_stride;
        h.n_kv_heads = kv->n_kv_heads;
        h.group = n_q_heads / kv->n_kv_heads;
        h.rows = rows;
        h.gh = plan.gh;
        h.gh_inv = (65536 + plan.gh - 1) / plan.gh;
        h.tt = plan.tt;
        h.hsubs = plan.hsubs;
        h.tok_tiles = plan.tok_tiles;
        h.n_tiles = plan.n_tiles;
        h.split_len = plan.split_len;
        h.n_splits_max = plan.n_splits_max;
        const bool aligned = aligned16(h.q) && aligned16(a.out) && (!a.gate || aligned16(a.gate)) && q_seq_stride % 8 == 0 &&
                             q_tok_stride % 8 == 0 && g_seq_stride % 8 == 0 && g_tok_stride % 8 == 0 && o_seq_stride % 8 == 0 &&
                             o_tok_stride % 8 == 0;
        h.flags = (aligned ? kHotAligned : 0) | (plan.xcd_grid ? kHotXcdGrid : 0) | (plan.packed_splits > 0 ? kHotPackedSplits : 0);
        h.scale_log2e = scale * 1.4426950408889634f;
        h.window = window;
        h.ring_blocks = walks_pages ? pages->ring_blocks : kv->ring_blocks();
        a.keep = keep ? keep + base * keep_seq_stride : nullptr;
        a.keep_seq_stride = keep_seq_stride;
        a.keep_row_stride = keep_row_stride;
        // Finding a wavefront's touched blocks up front costs a round of loads in front of its first block.  A decode step gets
        // back that no wavefront reads a block without a kept key, its first one included.  Over fp16 pages of heads of 256 that
        // is worth it from two blocks a wavefront on (2,051 of 40,001 keys, 16/2 heads: 14.9 -> 13.5 us, of 70,001 17.7 -> 14.0, of
        // 131,070 22.3 -> 14.6, of 262,000 30.8 -> 14.9; with one block, at 8,000 keys, 10.3 against 10.7 the other way), over
        // narrower heads and quantised pages, whose blocks are fewer bytes, from about six (block by block / up front: 16/4 of
        // 64 behind 8,428 keys 7.76 / 8.13, 40/8 of 128 over 8 bits behind 20,002, five blocks, 13.5 / 13.8, behind 25,003, seven, 15.9 / 14.9).
        // From 50,000 keys on, of which a selection of two thousand in groups of four touches about one block in four, from four (24/2
        // of 256 over 4 bits behind 55,000 18.6 / 17.4, 16/4 of 64 over 8 bits behind 72,327, five blocks, 14.1 / 12.8).
        // Per-query rows, whose walk reads every row's bytes first: from about eight.  (Those are always word-aligned: the
        // entry point requires it; a single sequence's mask has no stride to mind.)
        const int listed_blocks = keep_row_stride > 0 ? 8 : D == 256 && kv_bits == 16 ? 2 : max_keys >= 50000 ? 4 : 6;
        h.keep_words = a.keep && (uintptr_t)a.keep % 4 == 0 && (n == 1 || keep_seq_stride % 4 == 0) &&
                       plan.split_len >= listed_blocks * plan.waves * 32;
        for (int i = 0; i < n; ++i) {
            a.seq[i].slot = walks_pages ? 0 : slots[base + i];
            a.seq[i].start = starts[base + i];
            a.seq[i].total = totals[base + i];
            a.seq[i].first_split = first_split[i];
        }
        for (int i = n; i < kMaxSeqPerLaunch; ++i) a.seq[i].first_split = 0x7fffffff;  // (behind every split: see kHotPackedSplits)
        if (lists) {
            // The lists' plan, in the context's selection store: [tile][n_splits + 1] range starts, [tile][cap] blocks with
            // the keys any token keeps (pairs of words, on an even word), [tile][cap][tt] bits; a tile's list cannot be longer than the context's blocks or its tokens' entries.
            st = ensure_keep_rows(ctx, list_plan_words(plan.n_splits_max) * sizeof(int));
            if (st != TT_HIP_OK) return st;
            int *ranges = reinterpret_cast<int *>(ctx->keep_rows);
            int *blocks = ranges + list_ranges(plan.n_splits_max);
            unsigned *bits = reinterpret_cast<unsigned *>(blocks + n_blocks);
            // LDS of the plan kernel: two words per 32 units of context and the run of bits it gathers at a time, what that leaves of
            // 64 KiB: every run is another walk over the lists.
            const int words = (ctx_units + 31) / 32;
            const int chunk_words = (65536 / 4) - (2 * words + kPlanThreads + 1);
            const int chunk_entries = chunk_words / (plan.tt | 1);
            if (chunk_entries < 1) return TT_HIP_ERR_CAPACITY;
            const bool by_key = !groups && launch_fetches_by_key(D, kv_bits, plan.n_tiles, (long long)plan.tt * (long long)lists->stride,
                                                                 totals[base], ctx->n_cus);
            const auto kernel = groups ? keep_plan_kernel<true> : keep_plan_kernel<false>;
            hipLaunchKernelGGL(kernel, dim3((unsigned)plan.tok_tiles), dim3(kPlanThreads),
                               (size_t)(2 * words + kPlanThreads + 1 + chunk_entries * (plan.tt | 1)) * sizeof(unsigned), ctx->stream, lists->indices,
                               (unsigned)lists->stride, lists->counts, starts[base], rows, totals[base], plan.tt, plan.split_len / 32,
                               plan.n_splits_max, cap, chunk_entries, ranges, blocks, bits, by_key);
            e = hipGetLastError();
            if (e != hipSuccess) return hip_fail(ctx, e, "keep_plan_kernel launch");
            a.plan_groups = groups;
            a.plan_by_key = by_key;
            a.plan_ranges = ranges;
            a.plan_blocks = blocks;
            a.plan_bits = bits;
            a.plan_cap = cap;
        }
        if (chunk_splits > 1) {
            st = launch_prefill(ctx, kv, layer, slots[base], starts[base], rows, totals[base], n_q_heads, q, q_tok_stride, gate,
                                g_tok_stride, scale, out, o_tok_stride, chunk_splits, chunk_split_blocks, ctx->part_o,
                                ctx->part_ml, pages, window);
            if (st == TT_HIP_OK) st = launch_combine(ctx, plan, D, n, a);
        } else {
            st = launch_splitk(ctx, plan, D, n, a, kv_bits);
        }
        if (st != TT_HIP_OK) return st;
    }
    return TT_HIP_OK;
}

}  // namespace tt

using namespace tt;

// The calls that follow run on `next`, behind what the context has on its present stream: the stores it keeps for its calls -- partial results,
// dequantised pages, the plans of index lists, the key selection's workspace -- are one set, and a call that overlapped another would work in
// them while the other reads them (a list's plan holds places that the attention kernel reads at).  A stream that is being captured
// has no part in that order: what it holds runs when its graph is launched, and its capture would not survive a wait for outside work.
static int change_stream(tt_hip_ctx *ctx, hipStream_t next) {
    if (next == ctx->stream) return TT_HIP_OK;
    auto capturing = [](hipStream_t stream) {
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        if (stream && hipStreamIsCapturing(stream, &status) != hipSuccess) (void)hipGetLastError();
        return status != hipStreamCaptureStatusNone;
    };
    if (hipSetDevice(ctx->device) != hipSuccess) return TT_HIP_ERR_HIP;
    if (!capturing(next) && !capturing(ctx->stream)) {
        hipError_t e = hipEventRecord(ctx->ev_order, ctx->stream);
        if (e == hipSuccess) e = hipStreamWaitEvent(next, ctx->ev_order, 0);
        if (e != hipSuccess) {  // (a stream that its owner has destroyed meanwhile)
            (void)hipGetLastError();
            if (hipDeviceSynchronize() != hipSuccess) (void)hipGetLastError();
        }
    }
    ctx->stream = next;
    return TT_HIP_OK;
}

extern "C" {

tt_hip_ctx *tt_hip_ctx_create(int device, int *out_err) {
    auto fail = [&](int code) -> tt_hip_ctx * {
        if (out_err) *out_err = code;
        return nullptr;
    };
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || device < 0 || device >= count) {
        (void)hipGetLastError();
        return fail(TT_HIP_ERR_NO_DEVICE);
    }
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) return fail(TT_HIP_ERR_HIP);
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) return fail(TT_HIP_ERR_NO_DEVICE);
    if (hipSetDevice(device) != hipSuccess) return fail(TT_HIP_ERR_HIP);
    tt_hip_ctx *ctx = new (std::nothrow) tt_hip_ctx();
    if (!ctx) return fail(TT_HIP_ERR_OUT_OF_MEMORY);
    ctx->device = device;
    ctx->n_cus = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
    if (hipStreamCreateWithFlags(&ctx->own_stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreate(&ctx->ev_begin) != hipSuccess || hipEventCreate(&ctx->ev_end) != hipSuccess ||
        hipEventCreateWithFlags(&ctx->ev_order, hipEventDisableTiming) != hipSuccess) {
        tt_hip_ctx_destroy(ctx);
        return fail(TT_HIP_ERR_HIP);
    }
    ctx->stream = ctx->own_stream;
    // This device's copy of the static scratch array (the device is current).
    if (hipGetSymbolAddress(reinterpret_cast<void **>(&ctx->static_scratch), HIP_SYMBOL(scratch)) != hipSuccess ||
        !ctx->static_scratch) {
        (void)hipGetLastError();
        tt_hip_ctx_destroy(ctx);
        return fail(TT_HIP_ERR_HIP);
    }
    // The kernels' dynamic-LDS limits are properties of the device's copy of the code: set by the first context
    // on a device, found set by every later one.
    static std::mutex configured_lock;
    static bool configured[64] = {};
    {
        std::lock_guard<std::mutex> hold(configured_lock);
        if (device >= 64 || !configured[device]) {
            int st = configure_splitk_kernels(ctx);
            if (st == TT_HIP_OK) st = configure_prefill_kernels(ctx);
            if (st == TT_HIP_OK) st = configure_affine_kernels(ctx);
            if (st != TT_HIP_OK) {
                tt_hip_ctx_destroy(ctx);
                return fail(st);
            }
            if (device < 64) configured[device] = true;
        }
    }
    if (out_err) *out_err = TT_HIP_OK;
    return ctx;
}

void tt_hip_ctx_destroy(tt_hip_ctx *ctx) {
    if (!ctx) return;
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);  // (null: the default stream)
    if (ctx->part_o) (void)hipFree(ctx->part_o);
    if (ctx->part_ml) (void)hipFree(ctx->part_ml);
    if (ctx->stage_k) (void)hipFree(ctx->stage_k);
    if (ctx->stage_v) (void)hipFree(ctx->stage_v);
    if (ctx->select_ws) (void)hipFree(ctx->select_ws);
    if (ctx->keep_rows) (void)hipFree(ctx->keep_rows);
    for (hipEvent_t ev : ctx->prof_events) (void)hipEventDestroy(ev);
    if (ctx->ev_begin) (void)hipEventDestroy(ctx->ev_begin);
    if (ctx->ev_end) (void)hipEventDestroy(ctx->ev_end);
    if (ctx->ev_order) (void)hipEventDestroy(ctx->ev_order);
    if (ctx->own_stream) (void)hipStreamDestroy(ctx->own_stream);
    delete ctx;
}

int tt_hip_ctx_set_stream(tt_hip_ctx *ctx, void *hip_stream) {
    if (!ctx) return TT_HIP_ERR_INVALID_ARGUMENT;
    BusyGuard guard(ctx);
    if (!guard.ok || ctx->capturing) return TT_HIP_ERR_BUSY;
    return change_stream(ctx, hip_stream ? reinterpret_cast<hipStream_t>(hip_stream) : ctx->own_stream);
}

int tt_hip_ctx_set_default_stream(tt_hip_ctx *ctx) {
    if (!ctx) return TT_HIP_ERR_INVALID_ARGUMENT;
    BusyGuard guard(ctx);
    if (!guard.ok || ctx->capturing) return TT_HIP_ERR_BUSY;
    return change_stream(ctx, nullptr);  // the legacy default stream
}

void *tt_hip_ctx_stream(tt_hip_ctx *ctx) { return ctx ? reinterpret_cast<void *>(ctx->stream) : nullptr; }

int tt_hip_sync(tt_hip_ctx *ctx) {
    if (!ctx) return TT_HIP_ERR_INVALID_ARGUMENT;
    hipError_t e = hipStreamSynchronize(ctx->stream);
    return e == hipSuccess ? TT_HIP_OK : hip_fail(ctx, e, "hipStreamSynchronize");
}

int tt_hip_timer_begin(tt_hip_ctx *ctx) {
    if (!ctx) return TT_HIP_ERR_INVALID_ARGUMENT;
    hipError_t e = hipEventRecord(ctx->ev_begin, ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, e, "hipEventRecord");
    ctx->timer_open = true;
    return TT_HIP_OK;
}

int tt_hip_timer_end(tt_hip_ctx *ctx, uint64_t *out_ns) {
    if (!ctx || !out_ns || !ctx->timer_open) return TT_HIP_ERR_INVALID_ARGUMENT;
    ctx->timer_open = false;
    hipError_t e = hipEventRecord(ctx->ev_end, ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, e, "hipEventRecord");
    e = hipEventSynchronize(ctx->ev_end);
    if (e != hipSuccess) return hip_fail(ctx, e, "hipEventSynchronize");
    float ms = 0.0f;
    e = hipEventElapsedTime(&ms, ctx->ev_begin, ctx->ev_end);
    if (e != hipSuccess) return hip_fail(ctx, e, "hipEventElapsedTime");
    *out_ns = (uint64_t)((double)ms * 1.0e6);
    return TT_HIP_OK;
}

int tt_hip_profile_enable(tt_hip_ctx *ctx, int max_launches) {
    if (!ctx || max_launches <= 0 || max_launches > (1 << 20)) return TT_HIP_ERR_INVALID_ARGUMENT;
    BusyGuard guard(ctx);
    if (!guard.ok || ctx->capturing) return TT_HIP_ERR_BUSY;
    if (hipSetDevice(ctx->device) != hipSuccess) return TT_HIP_ERR_HIP;
    while (ctx->prof_events.size() < (size_t)max_launches * 2) {
        hipEvent_t ev = nullptr;
        hipError_t e = hipEventCreate(&ev);
        if (e != hipSuccess) return hip_fail(ctx, e, "hipEventCreate");
        ctx->prof_events.push_back(ev);
    }
    // Calibrate: an empty event pair on the idle stream.
    hipError_t e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, e, "hipStreamSynchronize");
    float best = -1.0f;
    for (int i = 0; i < 16; ++i) {
        (void)hipEventRecord(ctx->prof_events[0], ctx->stream);
        (void)hipEventRecord(ctx->prof_events[1], ctx->stream);
        e = hipEventSynchronize(ctx->prof_events[1]);
        if (e != hipSuccess) return hip_fail(ctx, e, "hipEventSynchronize");
        float ms = 0.0f;
        if (hipEventElapsedTime(&ms, ctx->prof_events[0], ctx->prof_events[1]) == hipSuccess && (best < 0.0f || ms < best))
            best = ms;
    }
    ctx->prof_overhead_ns = best > 0.0f ? (uint64_t)((double)best * 1.0e6) : 0;
    ctx->prof_used = 0;
    ctx->profiling = true;
    return TT_HIP_OK;
}

int tt_hip_profile_event_overhead_ns(tt_hip_ctx *ctx, uint64_t *out_ns) {
    if (!ctx || !out_ns) return TT_HIP_ERR_INVALID_ARGUMENT;
    *out_ns = ctx->prof_overhead_ns;
    return TT_HIP_OK;
}

int tt_hip_profile_disable(tt_hip_ctx *ctx) {
    if (!ctx) return TT_HIP_ERR_INVALID_ARGUMENT;
    ctx->profiling = false;
    return TT_HIP_OK;
}

int tt_hip_profile_read(tt_hip_ctx *ctx, int *out_launches, uint64_t *out_total_ns) {
    if (!ctx || !out_launches || !out_total_ns) return TT_HIP_ERR_INVALID_ARGUMENT;
    BusyGuard guard(ctx);
    if (!guard.ok || ctx->capturing) return TT_HIP_ERR_BUSY;
    hipError_t e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) return hip_fail(ctx, e, "hipStreamSynchronize");
    double total_ms = 0.0;
    for (size_t i = 0; i + 1 < ctx->prof_used; i += 2) {
        float ms = 0.0f;
        e = hipEventElapsedTime(&ms, ctx->prof_events[i], ctx->prof_events[i + 1]);
        if (e != hipSuccess) return hip_fail(ctx, e, "hipEventElapsedTime");
        total_ms += ms;
    }
    *out_launches = (int)(ctx->prof_used / 2);
    *out_total_ns = (uint64_t)(total_ms * 1.0e6);
    ctx->prof_used = 0;
    return TT_HIP_OK;
}

int tt_hip_graph_begin(tt_hip_ctx *ctx) {
    if (!ctx) return TT_HIP_ERR_INVALID_ARGUMENT;
    BusyGuard guard(ctx);
    if (!guard.ok || ctx->capturing) return TT_HIP_ERR_BUSY;
    if (hipSetDevice(ctx->device) != hipSuccess) return TT_HIP_ERR_HIP;
    hipError_t e = hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) return hip_fail(ctx, e, "hipStreamBeginCapture");
    ctx->capturing = true;
    return TT_HIP_OK;
}

int tt_hip_graph_end(tt_hip_ctx *ctx, tt_hip_graph **out_graph) {
    if (!ctx || !out_graph || !ctx->capturing) return TT_HIP_ERR_INVALID_ARGUMENT;
    BusyGuard guard(ctx);
    if (!guard.ok) return TT_HIP_ERR_BUSY;
    ctx->capturing = false;
    hipGraph_t graph = nullptr;
    hipError_t e = hipStreamEndCapture(ctx->stream, &graph);
    if (e != hipSuccess || !graph) return hip_fail(ctx, e, "hipStreamEndCapture");
    hipGraphExec_t exec = nullptr;
    e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    if (e != hipSuccess) {
        (void)hipGraphDestroy(graph);
        return hip_fail(ctx, e, "hipGraphInstantiate");
    }
    tt_hip_graph *g = new (std::nothrow) tt_hip_graph();
    if (!g) {
        (void)hipGraphExecDestroy(exec);
        (void)hipGraphDestroy(graph);
        return TT_HIP_ERR_OUT_OF_MEMORY;
    }
    g->graph = graph;
    g->exec = exec;
    g->ctx = ctx;
    g->generation = ctx->generation;
    *out_graph = g;
    return TT_HIP_OK;
}

int tt_hip_graph_launch(tt_hip_ctx *ctx, tt_hip_graph *graph) {
    if (!ctx || !graph || !graph->exec) return TT_HIP_ERR_INVALID_ARGUMENT;
    BusyGuard guard(ctx);
    if (!guard.ok || ctx->capturing) return TT_HIP_ERR_BUSY;
    // Buffers whose addresses the graph's kernels carry have been released since the capture.
    if (graph->ctx != ctx || graph->generation != ctx->generation) return TT_HIP_ERR_STALE;
    hipError_t e = hipGraphLaunch(graph->exec, ctx->stream);
    return e == hipSuccess ? TT_HIP_OK : hip_fail(ctx, e, "hipGraphLaunch");
}

void tt_hip_graph_destroy(tt_hip_graph *graph) {
    if (!graph) return;
    if (graph->exec) (void)hipGraphExecDestroy(graph->exec);
    if (graph->graph) (void)hipGraphDestroy(graph->graph);
    delete graph;
}

int tt_hip_split_geometry(tt_hip_ctx *ctx, int n_seq, int n_q_heads, int n_kv_heads, int head_dim, int rows,
                          int seq_len, int *out_split_tokens, int *out_splits, int *out_workgroups) {
    if (!ctx || seq_len < 0) return TT_HIP_ERR_INVALID_ARGUMENT;
    LaunchPlan plan{};
    int st = plan_launch(ctx, 0, n_seq, n_q_heads, n_kv_heads, head_dim, rows, (long long)seq_len * n_seq, seq_len, seq_len, &plan, 16, true);
    if (st != TT_HIP_OK) return st;
    if (out_split_tokens) *out_split_tokens = plan.split_len;
    if (out_splits) *out_splits = plan.n_splits_max;
    if (out_workgroups) *out_workgroups = (int)plan.workgroups;
    return TT_HIP_OK;
}

int tt_hip_set_split_tokens(tt_hip_ctx *ctx, int split_tokens) {
    if (!ctx || split_tokens < 0) return TT_HIP_ERR_INVALID_ARGUMENT;
    ctx->split_override = split_tokens;
    return TT_HIP_OK;
}

int tt_hip_set_option(tt_hip_ctx *ctx, int option, int value) {
    if (!ctx) return TT_HIP_ERR_INVALID_ARGUMENT;
    BusyGuard guard(ctx);
    if (!guard.ok || ctx->capturing) return TT_HIP_ERR_BUSY;
    switch (option) {
        case TT_HIP_OPT_KV_STREAM:
            if (value < -1 || value > 1) return TT_HIP_ERR_INVALID_ARGUMENT;
            ctx->stream_override = value;
            return TT_HIP_OK;
        case TT_HIP_OPT_XCD_GRID:
            if (value != 0 && value != 1) return TT_HIP_ERR_INVALID_ARGUMENT;
            ctx->xcd_grid = value != 0;
            return TT_HIP_OK;
        case TT_HIP_OPT_MEASURE_PASS_ONLY:
            if (value != 0 && value != 1) return TT_HIP_ERR_INVALID_ARGUMENT;
            ctx->pass_only = value != 0;
            return TT_HIP_OK;
        default: return TT_HIP_ERR_INVALID_ARGUMENT;
    }
}

int tt_hip_calibrate_read(tt_hip_ctx *ctx, const void *src, size_t bytes, uint32_t *sink, size_t *out_bytes_read) {
    if (!ctx || !src || (reinterpret_cast<uintptr_t>(src) & 15u) != 0) return TT_HIP_ERR_INVALID_ARGUMENT;
    BusyGuard guard(ctx);
    if (!guard.ok) return TT_HIP_ERR_BUSY;
    const size_t per_turn = (size_t)ctx->n_cus * 65536;  // every workgroup reads 64 KiB per turn
    const size_t turns = bytes / per_turn;
    if (turns == 0 || turns > 0xffffffffull) return TT_HIP_ERR_SHAPE;
    if (hipSetDevice(ctx->device) != hipSuccess) return TT_HIP_ERR_HIP;
    launch_profiled(ctx, calibrate_read_kernel, dim3((unsigned)ctx->n_cus), dim3(256), 0u, static_cast<const u4 *>(src),
                    (unsigned)turns, sink);
    const hipError_t e = hipGetLastError();
    if (out_bytes_read) *out_bytes_read = turns * per_turn;
    return e == hipSuccess ? TT_HIP_OK : hip_fail(ctx, e, "calibrate_read_kernel launch");
}

const char *tt_hip_strerror(int status) {
    switch (status) {
        case TT_HIP_OK: return "ok";
        case TT_HIP_ERR_INVALID_ARGUMENT: return "invalid argument";
        case TT_HIP_ERR_SHAPE: return "unsupported shape";
        case TT_HIP_ERR_CURSOR: return "KV cursor mismatch";
        case TT_HIP_ERR_CAPACITY: return "KV capacity exceeded";
        case TT_HIP_ERR_BUSY: return "context busy (re-entered)";
        case TT_HIP_ERR_OUT_OF_MEMORY: return "out of device memory";
        case TT_HIP_ERR_HIP: return "HIP runtime error";
        case TT_HIP_ERR_NO_DEVICE: return "no gfx950 device";
        case TT_HIP_ERR_STALE: return "graph captured before a buffer it uses was reallocated";
        case TT_HIP_ERR_SCRATCH: return "call needs more split scratch than the fixed array of the no-allocation entry point holds";
        default: return "unknown status";
    }
}

const char *tt_hip_last_hip_error(tt_hip_ctx *ctx) { return ctx ? ctx->last_hip_error.c_str() : ""; }

// ---- attention entry points ------------------------------------------------

static int check_common(tt_hip_ctx *ctx, tt_hip_kv *kv, int layer, int n_q_heads, const void *q, const void *out) {
    if (!ctx || !kv || !q || !out) return TT_HIP_ERR_INVALID_ARGUMENT;
    if (kv->ctx != ctx) return TT_HIP_ERR_INVALID_ARGUMENT;
    if (layer < 0 || layer >= kv->n_layers) return TT_HIP_ERR_INVALID_ARGUMENT;
    if (n_q_heads <= 0 || n_q_heads % kv->n_kv_heads != 0) return TT_HIP_ERR_SHAPE;
    return TT_HIP_OK;
}

int tt_hip_attn_decode(tt_hip_ctx *ctx, tt_hip_kv *kv, int layer, int n_seq, const int *slots, const int *seq_lens,
                       int n_q_heads, const tt_half *q, const tt_half *gate, float scale, tt_half *out) {
    return tt_hip_attn_decode_swa(ctx, kv, layer, n_seq, slots, seq_lens, 0, n_q_heads, q, gate, scale, out);
}

int tt_hip_attn_decode_swa(tt_hip_ctx *ctx, tt_hip_kv *kv, int layer, int n_seq, const int *slots, const int *seq_lens,
                           int window, int n_q_heads, const tt_half *q, const tt_half *gate, float scale, tt_half *out) {
    int st = check_common(ctx, kv, layer, n_q_heads, q, out);
    if (st != TT_HIP_OK) return st;
    if (n_seq <= 0 || !slots || !seq_lens || window < 0) return TT_HIP_ERR_INVALID_ARGUMENT;
    IntTable starts(n_seq);
    for (int i = 0; i < n_seq; ++i) {
        if (slots[i] < 0 || slots[i] >= kv->n_slots || seq_lens[i] < 0) return TT_HIP_ERR_INVALID_ARGUMENT;
        const long long first = window > 0 && seq_lens[i] > window ? seq_lens[i] - window : 0;
        if (!kv->holds_keys(first, seq_lens[i])) return TT_HIP_ERR_CAPACITY;
        starts[i] = seq_lens[i] - 1;
    }
    BusyGuard guard(ctx);
    if (!guard.ok) return TT_HIP_ERR_BUSY;
    const long long row = (long long)n_q_heads * kv->head_dim;
    return run_attention(ctx, kv, 0, layer, n_seq, slots, starts.data(), seq_lens, 1, n_q_heads, q, row, row, gate, row,
                         row, scale, out, row, row, 1, 0, nullptr, window);
}

// Same kernels and planner as tt_hip_attn_decode; the partials live in this device's copy of `scratch`
// (reached through the address taken at context creation) and the per-sequence tables on the stack, so the
// call allocates nothing on the device or the host.  Calls on one GPU share the array: they must not overlap.
int tt_hip_attn_decode_noalloc(tt_hip_ctx *ctx, tt_hip_kv *kv, int layer, int n_seq, const int *slots, const int *seq_lens,
                               int n_q_heads, const tt_half *q, const tt_half *gate, float scale, tt_half *out) {
    int st = check_common(ctx, kv, layer, n_q_heads, q, out);
    if (st != TT_HIP_OK) return st;
    if (n_seq <= 0 || !slots || !seq_lens) return TT_HIP_ERR_INVALID_ARGUMENT;
    if (n_seq > kMaxSeqPerLaunch) return TT_HIP_ERR_SCRATCH;  // one launch: its tables travel as kernel arguments
    int starts[kMaxSeqPerLaunch];
    for (int i = 0; i < n_seq; ++i) {
        if (slots[i] < 0 || slots[i] >= kv->n_slots || seq_lens[i] < 0) return TT_HIP_ERR_INVALID_ARGUMENT;
        if (!kv->holds_keys(0, seq_lens[i])) return TT_HIP_ERR_CAPACITY;
        starts[i] = seq_lens[i] - 1;
    }
    BusyGuard guard(ctx);
    if (!guard.ok) return TT_HIP_ERR_BUSY;
    const long long row = (long long)n_q_heads * kv->head_dim;
    return run_attention(ctx, kv, 0, layer, n_seq, slots, starts, seq_lens, 1, n_q_heads, q, row, row, gate, row, row, scale,
                         out, row, row, 1, 0, nullptr, 0, nullptr, 0, 0, /*static_partials=*/true);
}

int tt_hip_attn_decode_keep(tt_hip_ctx *ctx, tt_hip_kv *kv, int layer, int n_seq, const int *slots, const int *seq_lens,
                            const uint8_t *keep_mask, size_t keep_stride, int n_q_heads, const tt_half *q,
                            const tt_half *gate, float scale, tt_half *out) {
    int st = check_common(ctx, kv, layer, n_q_heads, q, out);
    if (st != TT_HIP_OK) return st;
    if (n_seq <= 0 || !slots || !seq_lens || !keep_mask) return TT_HIP_ERR_INVALID_ARGUMENT;
    IntTable starts(n_seq);
    for (int i = 0; i < n_seq; ++i) {
        if (slots[i] < 0 || slots[i] >= kv->n_slots || seq_lens[i] < 0) return TT_HIP_ERR_INVALID_ARGUMENT;
        if (n_seq > 1 && keep_stride < (size_t)seq_lens[i]) return TT_HIP_ERR_SHAPE;  // masks would overlap
        if (!kv->holds_keys(0, seq_lens[i])) return TT_HIP_ERR_CAPACITY;
        starts[i] = seq_lens[i] - 1;
    }
    BusyGuard guard(ctx);
    if (!guard.ok) return TT_HIP_ERR_BUSY;
    const long long row = (long long)n_q_heads * kv->head_dim;
    return run_attention(ctx, kv, 0, layer, n_seq, slots, starts.data(), seq_lens, 1, n_q_heads, q, row, row, gate, row,
                         row, scale, out, row, row, 1, 0, nullptr, 0, keep_mask, (long long)keep_stride);
}

int tt_hip_attn_decode_keep_indices(tt_hip_ctx *ctx, tt_hip_kv *kv, int layer, int n_seq, const int *slots, const int *seq_lens,
                                    const uint32_t *keep_indices, size_t keep_index_stride, const uint32_t *keep_counts,
                                    int n_q_heads, const tt_half *q, const tt_half *gate, float scale, tt_half *out) {
    int st = check_common(ctx, kv, layer, n_q_heads, q, out);
    if (st != TT_HIP_OK) return st;
    if (n_seq <= 0 || !slots || !seq_lens || !keep_indices || !keep_counts) return TT_HIP_ERR_INVALID_ARGUMENT;
    if (keep_index_stride == 0 || keep_index_stride > 0x7fffffffULL) return TT_HIP_ERR_SHAPE;
    IntTable starts(n_seq);
    int longest = 0;
    for (int i = 0; i < n_seq; ++i) {
        if (slots[i] < 0 || slots[i] >= kv->n_slots || seq_lens[i] < 0) return TT_HIP_ERR_INVALID_ARGUMENT;
        if (!kv->holds_keys(0, seq_lens[i])) return TT_HIP_ERR_CAPACITY;
        starts[i] = seq_lens[i] - 1;
        longest = std::max(longest, seq_lens[i]);
    }
    // One row of selection bytes per sequence in the context's store (a key at or past a sequence's length is
    // dropped by the kernel's own range test), then the mask form.
    const size_t row_stride = ((size_t)longest + 63) / 64 * 64 + 64;
    if ((unsigned long long)n_seq * row_stride > 0x7ff00000ULL) return TT_HIP_ERR_SHAPE;
    BusyGuard guard(ctx);
    if (!guard.ok) return TT_HIP_ERR_BUSY;
    if (hipSetDevice(ctx->device) != hipSuccess) return TT_HIP_ERR_HIP;
    st = ensure_keep_rows(ctx, (size_t)n_seq * row_stride);
    if (st != TT_HIP_OK) return st;
    hipLaunchKernelGGL(keep_rows_from_indices_kernel, dim3((unsigned)n_seq), dim3(256), 0, ctx->stream, ctx->keep_rows,
                       (unsigned)row_stride, keep_indices, (unsigned)keep_index_stride, keep_counts, 0x3fffffff, (int)row_stride);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(ctx, e, "keep_rows_from_indices_kernel");
    const long long row = (long long)n_q_heads * kv->head_dim;
    return run_attention(ctx, kv, 0, layer, n_seq, slots, starts.data(), seq_lens, 1, n_q_heads, q, row, row, gate, row,
                         row, scale, out, row, row, 1, 0, nullptr, 0, ctx->keep_rows, (long long)row_stride);
}

int tt_hip_attn_prefill_keep(tt_hip_ctx *ctx, tt_hip_kv *kv, int layer, int slot, int start_pos, int q_len, int kv_valid,
                             const uint8_t *keep_mask, size_t keep_stride, int n_q_heads, const tt_half *q, size_t q_stride,
                             const tt_half *gate, size_t gate_stride, float scale, tt_half *out, size_t o_stride) {
    int st = check_common(ctx, kv, layer, n_q_heads, q, out);
    if (st != TT_HIP_OK) return st;
    if (slot < 0 || slot >= kv->n_slots || start_pos < 0 || q_len <= 0 || !keep_mask) return TT_HIP_ERR_INVALID_ARGUMENT;
    const size_t packed = (size_t)n_q_heads * kv->head_dim;
    if (q_stride < packed || o_stride < packed || (gate && gate_stride < packed)) return TT_HIP_ERR_SHAPE;
    if ((long long)start_pos + q_len > kv_valid) return TT_HIP_ERR_INVALID_ARGUMENT;
    // a row's bytes cover every position the chunk can see; rows are read a word at a time
    if (keep_stride < (size_t)start_pos + (size_t)q_len || keep_stride % 4 != 0 || (uintptr_t)keep_mask % 4 != 0)
        return TT_HIP_ERR_SHAPE;
    if ((unsigned long long)q_len * keep_stride > 0x7ff00000ULL) return TT_HIP_ERR_SHAPE;  // 32-bit addressing of the rows
    if (!kv->holds_keys(0, kv_valid)) return TT_HIP_ERR_CAPACITY;
    BusyGuard guard(ctx);
    if (!guard.ok) return TT_HIP_ERR_BUSY;
    // The GQA-packed split-K tiles (the chunk kernel does not take a selection): every tile walks its rows' keys.
    return run_attention(ctx, kv, 0, layer, 1, &slot, &start_pos, &kv_valid, q_len, n_q_heads, q, 0, (long long)q_stride,
                         gate, 0, (long long)gate_stride, scale, out, 0, (long long)o_stride, 1, 0, nullptr, 0, keep_mask, 0,
                         (long long)keep_stride);
}

int tt_hip_attn_prefill_keep_indices(tt_hip_ctx *ctx, tt_hip_kv *kv, int layer, int slot, int start_pos, int q_len,
                                     int kv_valid, const uint32_t *keep_indices, size_t keep_index_stride,
                                     const uint32_t *keep_counts, int n_q_heads, const tt_half *q, size_t q_stride,
                                     const tt_half *gate, size_t gate_stride, float scale, tt_half *out, size_t o_stride) {
    int st = check_common(ctx, kv, layer, n_q_heads, q, out);
    if (st != TT_HIP_OK) return st;
    if (slot < 0 || slot >= kv->n_slots || start_pos < 0 || q_len <= 0 || !keep_indices || !keep_counts)
        return TT_HIP_ERR_INVALID_ARGUMENT;
    const size_t packed = (size_t)n_q_heads * kv->head_dim;
    if (q_stride < packed || o_stride < packed || (gate && gate_stride < packed)) return TT_HIP_ERR_SHAPE;
    if ((long long)start_pos + q_len > kv_valid) return TT_HIP_ERR_INVALID_ARGUMENT;
    if (keep_index_stride == 0 || keep_index_stride > 0x7fffffffULL) return TT_HIP_ERR_SHAPE;
    if (!kv->holds_keys(0, kv_valid)) return TT_HIP_ERR_CAPACITY;
    // (the plan kernel's bitmap of the context's blocks lives in LDS, 8 bytes per 1,024 keys, beside a run of the bits
    // it gathers: 64 KiB hold 8 million keys less that run, beyond what a page can address)
    if (((long long)kv_valid + 1023) / 1024 * 8 + (kPlanThreads + 1 + 32) * 4 > 65536) return TT_HIP_ERR_CAPACITY;
    BusyGuard guard(ctx);
    if (!guard.ok) return TT_HIP_ERR_BUSY;
    if (hipSetDevice(ctx->device) != hipSuccess) return TT_HIP_ERR_HIP;
    // The lists are served as they are: a launch turns them into each token tile's list of touched key blocks and
    // per-token key bits (keep_plan_kernel), which the attention kernel then walks -- work and memory of the order of
    // the selection.  Long chunks go in pieces of rows, so that the plan of one piece stays below 128 MiB.
    const int group = n_q_heads / kv->n_kv_heads, gh = packed_heads(group);
    const int tt = 32 / gh;  // tokens per tile of the 32-row tiles
    const long long ctx_blocks = ((long long)kv_valid + 31) / 32, entries = (long long)tt * (long long)keep_index_stride;
    const long long cap = entries < ctx_blocks ? entries : ctx_blocks;
    const long long group_cap = (entries < 8 * ctx_blocks ? entries : 8 * ctx_blocks) + 8;  // (a plan of groups, run_attention)
    const long long block_words = cap * (2 + tt), group_words = group_cap + group_cap / 8 * tt;
    const long long per_tile = ((block_words > group_words ? block_words : group_words) + 260) * 4;
    long long tiles_per_call = (128ll << 20) / per_tile;
    if (tiles_per_call < 1) tiles_per_call = 1;
    const long long rows_per_call = tiles_per_call * tt;
    PageSource staged{};
    const PageSource *pages = nullptr;
    // Quantised pages: a tile widens every block it walks, and blocks only, not groups of keys.  Where the tiles together walk
    // the context several times over and there are enough of them to matter, the visible blocks are dequantised once per
    // call instead, as for a dense chunk, and the fp16 kernels walk those.  us a sparse layer's step, pages as they are / dequantised, 8 bits
    // (over 4 bits, which take longer to widen, the second way gains more), rows with a selection of 2,051 keys each / all with one:
    //   heads of 256 from 32 tiles on: 16/2, 64 rows behind 12k keys 88 / 81, 86 / 75, 128 behind 60k 220 / 137, 148 / 121, 256 behind 150k
    //     479 / 325, 269 / 244; 24/2, 100 behind 60k 259 / 151, 198 / 131; walked 1.3 times, 128 behind 200k, 294 / 281, 226 / 240: left alone
    //   heads of 128, tiles of four tokens or fewer: 16/2, 128 rows behind 30k 129 / 96, 106 / 82; of more, whose selections touch most blocks
    //     anyway: 32/8, 100 rows behind 60k (walked 3.6 times) 251 / 270, 165 / 194, behind 12k (17 times) 132 / 124, 125 / 117
    //   heads of 64, whose tiles are the cheapest, over long contexts or many tiles: 16/4, 128 rows behind 12k 80 / 85, 79 / 85, behind
    //     60k 150 / 119, 106 / 95, 400 behind 100k 406 / 237, 219 / 168; 64/8, 80 rows behind 30k 162 / 111, 128 / 95.
    // Distance from 64 bits: the 2-norm falls by a sixth or more, the largest single difference grows by a tenth to two fifths (every value of V is rounded
    // to fp16 by itself, where a probability times a group's scale was, once for 64 dims).
    const long long tok_tiles = (q_len + tt - 1) / tt, tiles = tok_tiles * (group / gh) * kv->n_kv_heads;
    const long long walked = tok_tiles * (entries < kv_valid ? entries : kv_valid);
    const bool worth = kv->head_dim == 256 ? tiles >= 32 && walked >= 3ll * kv_valid
                       : kv->head_dim == 128 ? (tiles >= 128 && walked >= 5ll * kv_valid) || (tt <= 4 && tiles >= 64 && walked >= 3ll * kv_valid)
                                             : (tiles >= 256 && walked >= 5ll * kv_valid) || (tiles * kv_valid >= 64 * 40000ll && walked >= 3ll * kv_valid);
    if (kv->bits != 16 && !kv->ring && kv_valid >= 6144 && worth) {
        const int n_blocks = (kv_valid + 31) / 32;
        const size_t page = (size_t)n_blocks * 32 * kv->head_dim;
        if (ensure_stage(ctx, page * kv->n_kv_heads) == TT_HIP_OK) {  // (else, as inside a capture: the pages as they are)
            const int st = launch_kvq_dequant_blocks(kv, layer, slot, n_blocks, ctx->stage_k, ctx->stage_v, page);
            if (st != TT_HIP_OK) return st;
            staged = PageSource{ctx->stage_k, ctx->stage_v, (long long)page, 0};
            pages = &staged;
        }
    }
    for (long long r0 = 0; r0 < q_len; r0 += rows_per_call) {
        const int rows = (int)(q_len - r0 < rows_per_call ? q_len - r0 : rows_per_call);
        const int start = start_pos + (int)r0;
        const KeepLists lists{keep_indices + (size_t)r0 * keep_index_stride, keep_index_stride, keep_counts + r0};
        st = run_attention(ctx, kv, 0, layer, 1, &slot, &start, &kv_valid, rows, n_q_heads,
                           q + (size_t)r0 * q_stride, 0, (long long)q_stride, gate ? gate + (size_t)r0 * gate_stride : nullptr, 0,
                           (long long)gate_stride, scale, out + (size_t)r0 * o_stride, 0, (long long)o_stride, 1, 0, pages, 0, nullptr,
                           0, 0, false, &lists);
        if (st != TT_HIP_OK) return st;
    }
    return TT_HIP_OK;
}

int tt_hip_attn_verify(tt_hip_ctx *ctx, tt_hip_kv *kv, int layer, int n_seq, const int *slots,
                       const int *start_positions, int rows, int n_q_heads, const tt_half *q, const tt_half *gate,
                       float scale, tt_half *out) {
    return tt_hip_attn_verify_swa(ctx, kv, layer, n_seq, slots, start_positions, rows, 0, n_q_heads, q, gate, scale, out);
}

int tt_hip_attn_verify_swa(tt_hip_ctx *ctx, tt_hip_kv *kv, int layer, int n_seq, const int *slots,
                           const int *start_positions, int rows, int window, int n_q_heads, const tt_half *q,
                           const tt_half *gate, float scale, tt_half *out) {
    int st = check_common(ctx, kv, layer, n_q_heads, q, out);
    if (st != TT_HIP_OK) return st;
    if (n_seq <= 0 || rows <= 0 || !slots || !start_positions || window < 0) return TT_HIP_ERR_INVALID_ARGUMENT;
    IntTable totals(n_seq);
    for (int i = 0; i < n_seq; ++i) {
        if (slots[i] < 0 || slots[i] >= kv->n_slots || start_positions[i] < 0) return TT_HIP_ERR_INVALID_ARGUMENT;
        const long long first = window > 0 && start_positions[i] + 1 > window ? start_positions[i] + 1 - window : 0;
        if (!kv->holds_keys(first, (long long)start_positions[i] + rows)) return TT_HIP_ERR_CAPACITY;
        totals[i] = start_positions[i] + rows;
    }
    BusyGuard guard(ctx);
    if (!guard.ok) return TT_HIP_ERR_BUSY;
    const long long tok = (long long)n_q_heads * kv->head_dim;
    const long long seq = tok * rows;
    return run_attention(ctx, kv, 0, layer, n_seq, slots, start_positions, totals.data(), rows, n_q_heads, q, seq, tok,
                         gate, seq, tok, scale, out, seq, tok, 1, 0, nullptr, window);
}

int tt_hip_attn_prefill(tt_hip_ctx *ctx, tt_hip_kv *kv, int layer, int slot, int start_pos, int q_len, int kv_valid,
                        int n_q_heads, const tt_half *q, size_t q_stride, const tt_half *gate, size_t gate_stride,
                        float scale, tt_half *out, size_t o_stride) {
    return tt_hip_attn_prefill_swa(ctx, kv, layer, slot, start_pos, q_len, kv_valid, 0, n_q_heads, q, q_stride, gate,
                                   gate_stride, scale, out, o_stride);
}

int tt_hip_attn_prefill_swa(tt_hip_ctx *ctx, tt_hip_kv *kv, int layer, int slot, int start_pos, int q_len, int kv_valid,
                            int sliding_window, int n_q_heads, const tt_half *q, size_t q_stride, const tt_half *gate,
                            size_t gate_stride, float scale, tt_half *out, size_t o_stride) {
    int st = check_common(ctx, kv, layer, n_q_heads, q, out);
    if (st != TT_HIP_OK) return st;
    if (slot < 0 || slot >= kv->n_slots || start_pos < 0 || q_len <= 0 || sliding_window < 0) return TT_HIP_ERR_INVALID_ARGUMENT;
    const size_t packed = (size_t)n_q_heads * kv->head_dim;
    if (q_stride < packed || o_stride < packed || (gate && gate_stride < packed)) return TT_HIP_ERR_SHAPE;
    if ((long long)start_pos + q_len > kv_valid) return TT_HIP_ERR_INVALID_ARGUMENT;
    {
        const long long first = sliding_window > 0 && start_pos + 1 > sliding_window ? start_pos + 1 - sliding_window : 0;
        if (!kv->holds_keys(first, kv_valid)) return TT_HIP_ERR_CAPACITY;
    }
    BusyGuard guard(ctx);
    if (!guard.ok) return TT_HIP_ERR_BUSY;
    const bool aligned = aligned16(q) && aligned16(out) && (!gate || aligned16(gate)) && q_stride % 8 == 0 &&
                         o_stride % 8 == 0 && (!gate || gate_stride % 8 == 0);
    // A window that clips no row of the chunk is no window.
    const int window = sliding_window > 0 && (long long)start_pos + q_len > sliding_window ? sliding_window : 0;
    // (the chunk kernel takes a row's maximum over the raw scores: a scale that is not positive goes the split-K way)
    const bool serves = prefill_kernel_serves(n_q_heads, kv->n_kv_heads, kv->head_dim, aligned) && scale > 0.0f;
    const long long chunk_wgs = (long long)((q_len + 63) / 64) * (n_q_heads / 4);
    // The chunk kernel as it is -- a workgroup per pair of tiles and 4 heads, all their keys -- where its workgroups
    // fill half the chip, or a quarter of it with few key blocks each (a long first chunk of a prompt: 1024 rows from
    // position 0 take 39 us against 41 us through the split-K tiles, 1536 rows 51 against 66).  Fewer workgroups
    // walking more blocks lose to the other routes at any context: 128 rows behind 1920 keys took 100 us that way,
    // 25 us through the split-K tiles; behind a 1024-key window 62 us against 20 us.
    const long long pair_blocks = (2LL * start_pos + q_len) / 32 + 2;  // key blocks a workgroup's pair of tiles walks
    const bool filled = 2 * chunk_wgs >= ctx->n_cus || (window == 0 && 4 * chunk_wgs >= ctx->n_cus && pair_blocks <= 64);
    const int first_blocks = chunk_tile_blocks(start_pos, q_len, kv_valid, window, 0);
    const int last_blocks = chunk_tile_blocks(start_pos, q_len, kv_valid, window, (q_len + 31) / 32 - 1);
    const ChunkEstimate whole = estimate_chunk(ctx->n_cus, kv->head_dim, n_q_heads, kv->n_kv_heads, q_len, first_blocks, last_blocks);
    auto whole_tiles = [&](const PageSource *pages) {
        if (hipSetDevice(ctx->device) != hipSuccess) return (int)TT_HIP_ERR_HIP;
        return launch_prefill(ctx, kv, layer, slot, start_pos, q_len, kv_valid, n_q_heads, q, (long long)q_stride, gate,
                              (long long)gate_stride, scale, out, (long long)o_stride, 1, 0, nullptr, nullptr, pages, window,
                              whole.single_tiles);
    };
    const double splitk_us = estimate_splitk_chunk_us(ctx->n_cus, kv->head_dim, n_q_heads, kv->n_kv_heads, q_len, first_blocks, last_blocks);
    if (window > 0) {
        // The chunk kernel starts every tile at its window's first block.  It or the split-K kernel (GQA-packed tiles, each
        // walking only its rows' windows), whichever is estimated faster; quantised pages and head groups the chunk
        // kernel does not serve go through the latter.  32 / 8 heads of 128 behind a window of 4096 keys: 512 rows 65
        // against 78 us, 777 rows 105 against 80; 16 / 2 of 256 behind 1024 keys: 512 rows 24 against 34, 777 rows 43
        // against 34, 1024 rows 47 against 36.
        // Where the chunk does not fill the chip and the split-K tiles go in whole rounds with the last one part empty, the keys of a
        // window cut into ranges, as behind a long context (300 rows behind 4096 keys: 24 / 2 heads of 256 113.6 -> 55.3 us, 32 / 8 of
        // 128 56.7 -> 48.3; 16 / 2 of 256, 600 rows 115.7 -> 66.8, 270 behind 16,384 keys 188.6 -> 92.3), or the chunk kernel as it is.  16 us: the
        // combine pass and both kernels' starts.  Inside a capture the partial results' store does not grow.
        if (serves && kv->bits == 16 && !filled && q_len >= 256) {
            const int longest = longest_tile_blocks(start_pos, q_len, kv_valid, window);
            const double tiles_us = splitk_rounds_us(ctx->n_cus, n_q_heads, kv->n_kv_heads, q_len, longest, splitk_us);
            const KeyRanges r = plan_window_ranges(ctx->n_cus, kv->head_dim, n_q_heads, kv->n_kv_heads, start_pos, q_len, kv_valid, window);
            const size_t part_rows = (size_t)r.n_splits * n_q_heads * ((q_len + 31) / 32) * 32;
            if (r.n_splits >= 2 && r.us + 16.0 < 0.95 * std::min(whole.us, tiles_us) && (!ctx->capturing || part_rows <= ctx->part_rows))
                return run_attention(ctx, kv, 1, layer, 1, &slot, &start_pos, &kv_valid, q_len, n_q_heads, q, 0, (long long)q_stride, gate,
                                     0, (long long)gate_stride, scale, out, 0, (long long)o_stride, r.n_splits, r.split_blocks, nullptr, window);
            if (whole.us < 0.75 * tiles_us) return whole_tiles(nullptr);
        }
        // The estimates do not hold where the split-K tiles are all at work at once, as a few hundred rows of a short window are: 64 / 8
        // heads of 64, 226 rows behind 96 keys 7.0 us against 10.1, 32 / 8 of 128, 428 behind 128 12.9 / 14.6, 24 / 2 of 256, 247 behind
        // 33 12.6 / 19.1; one more round the other way (279 rows there 22.5 / 19.1, 560 of 32 / 8 19.1 / 13.8).
        const bool more_rounds = splitk_tiles(n_q_heads, kv->n_kv_heads, q_len) > splitk_tiles_at_once(ctx->n_cus, kv->head_dim);
        if (serves && kv->bits == 16 && (filled || (more_rounds && whole.us < splitk_us))) return whole_tiles(nullptr);
        return run_attention(ctx, kv, 0, layer, 1, &slot, &start_pos, &kv_valid, q_len, n_q_heads, q, 0, (long long)q_stride,
                             gate, 0, (long long)gate_stride, scale, out, 0, (long long)o_stride, 1, 0, nullptr, window);
    }
    // Quantised pages: the split-K kernel reads them as they are (dequantising in registers, once
    // per 32-row tile -- 269 TFLOP/s on a 4096-row chunk).  A chunk that the MFMA chunk kernel
    // would take is instead served from fp16 pages of the slot's visible blocks, dequantised once
    // per call into the context's staging store (4096 rows: one 9 us pass, then the fp16 kernel).
    PageSource staged{};
    const PageSource *pages = nullptr;
    // From this many keys on a chunk that does not fill the chip goes through the chunk kernel over key ranges (below:
    // through the split-K tiles): 786,432 / rows, i.e. 12k keys at 64 rows, 6k at 128, and at least 4096 (2560 over
    // quantised pages, whose visible blocks are dequantised once per call first).  The split-K tiles read the keys once
    // per tile of rows and leave small partial results; the ranges read them once per range and leave rows x heads x D
    // floats per range.  One box, fp16, split-K / ranges: 64 rows at 8k keys 31.6 / 33.4 us, at 12k 37.2 / 35.3; 96
    // rows at 4k 28.4 / 32.4, at 12k 47.7 / 42.8; 128 rows at 4k 32.0 / 35.0, at 8k 44.3 / 39.1; 192 rows at 4k 41.8 /
    // 38.6.  Over 8 bits: 64 rows at 4k 24.4 / 35.4, at 16k 50.1 / 49.2, at 32k 80.7 / 71.9; 128 rows at 4k 34.6 /
    // 40.2, at 8k 48.9 / 45.0.
    // Heads that leave rows of a split-K tile empty make more tiles of the same rows, and what that way takes goes by its tiles: there from 393,216 /
    // (tiles x D / 256) keys on where that is earlier, and from 2,048.  us a layer, split-K / ranges: 24 / 2 heads of 256, 96 rows behind 7,000 keys
    // 63.8 / 50.0, over 8 bits 81.0 / 55.7, 300 behind 3,000 109.2 / 74.9, 200 behind 1,600 53.0 / 56.0.  Not for other heads, though the ranges would often
    // be ahead (64 / 8 of 256, 130 rows behind 4,000 keys over 8 bits 173 / 119): not where the tiles share the chip out evenly (64 / 16 of 128, 64
    // rows behind 7,900 keys 48.1 / 51.3, over 8 bits 58.6 / 77.9, 96 rows behind 5,100 67.8 / 75.8; 32 / 4 of 256, 64 rows 56.9 / 60.7).
    const bool rows_left_empty = 32 % packed_heads(n_q_heads / kv->n_kv_heads) != 0;
    const long long by_rows = 786432 / (q_len > 0 ? q_len : 1), others_from = std::max<long long>(by_rows, kv->bits == 16 ? 4096 : 2560);
    long long ranges_from = others_from;
    if (rows_left_empty) {
        const long long tile_widths = splitk_tiles(n_q_heads, kv->n_kv_heads, q_len) * kv->head_dim;
        ranges_from = std::max<long long>(std::min(393216ll * 256 / (tile_widths > 0 ? tile_widths : 1), by_rows), 2048);
    }
    // ... and from this many rows on: 64; at fp16 32 rows deep in a context (32 rows at 32k keys 50 us against 54 us,
    // 48 rows 62 against 73).  Over quantised pages fewer rows stay with the split-K tiles, which widen a block once per
    // tile of 16 rows: dequantising the whole context for them costs more than that at any length measured (32 rows
    // at 64k keys over 8 bits 82 us against 107 us, 12 rows at 32k keys 30 us against 62 us).
    const int rows_from = kv->bits == 16 ? (kv_valid >= 32768 ? 32 : 64) : 64;
    if (serves && !filled && (kv->bits == 16 || !kv->ring) && q_len >= rows_from && kv_valid >= ranges_from && kv_valid < others_from) {
        // (no memory for the ranges' partial results or the dequantised pages, or a capture in which they would have to grow: the split-K way)
        const int blocks = (kv_valid + 31) / 32;
        const KeyRanges r = plan_key_ranges(ctx->n_cus, kv->head_dim, n_q_heads, kv->n_kv_heads, q_len, blocks);
        if (hipSetDevice(ctx->device) != hipSuccess) return TT_HIP_ERR_HIP;
        st = q_len >= 256 && whole.us < r.us ? TT_HIP_OK : ensure_partials(ctx, (size_t)r.n_splits * n_q_heads * ((q_len + 31) / 32) * 32, kv->head_dim);
        if (st == TT_HIP_OK && kv->bits != 16) st = ensure_stage(ctx, (size_t)blocks * 32 * kv->head_dim * kv->n_kv_heads);
        if (st == TT_HIP_ERR_BUSY || st == TT_HIP_ERR_OUT_OF_MEMORY) ranges_from = others_from;
        else if (st != TT_HIP_OK) return st;
    }
    if (kv->bits != 16 && !kv->ring && serves && q_len >= rows_from && (filled || kv_valid >= ranges_from)) {
        const int n_blocks = (kv_valid + 31) / 32;
        const size_t page = (size_t)n_blocks * 32 * kv->head_dim;
        if (hipSetDevice(ctx->device) != hipSuccess) return TT_HIP_ERR_HIP;
        st = ensure_stage(ctx, page * kv->n_kv_heads);
        if (st != TT_HIP_OK) return st;
        st = launch_kvq_dequant_blocks(kv, layer, slot, n_blocks, ctx->stage_k, ctx->stage_v, page);
        if (st != TT_HIP_OK) return st;
        staged = PageSource{ctx->stage_k, ctx->stage_v, (long long)page, 0};
        pages = &staged;
    }
    if (serves && (kv->bits == 16 || pages)) {
        // The chunk kernel gives a workgroup 64 query rows of 4 heads and ALL their keys: one
        // workgroup per CU at 4096 rows x 16 heads, but a 128-row chunk (the reference's default
        // prefillChunkTokens) deep into a long context would be 8 workgroups walking 32k keys
        // each (1318 us at 16q/2kv/256).  Three routes, chosen from timings at that shape:
        //  * at least half a chip of workgroups, or a quarter with few blocks each: the chunk kernel as it is;
        //  * 64 rows or more over 4096 keys or more (2560 over quantised pages): the chunk kernel with the keys cut into
        //    ranges, a workgroup per (tile, 4 heads, range), and the combine pass over the partial
        //    results (128 rows at 32k keys 98-106 us, 1024 rows 507-538 us; 256 rows at 4k keys 39 us
        //    against 46 us the split-K way);
        //  * anything else: the split-K kernel, which packs a KV head's q heads into its tiles
        //    like a verify pass (64 rows at 16k keys 62 us against 89 us; 512 rows at 2k keys
        //    59 us against 104 us, where the partial results outweigh the keys).
        int n_splits = 1, split_blocks = 0;
        double ranges_us = 0.0;
        if (!filled && q_len >= rows_from && kv_valid >= ranges_from) {
            const KeyRanges r = plan_key_ranges(ctx->n_cus, kv->head_dim, n_q_heads, kv->n_kv_heads, q_len, (kv_valid + 31) / 32);
            n_splits = r.n_splits;
            split_blocks = r.split_blocks;
            ranges_us = r.us;
        }
        // Unfilled chunks, too, where a workgroup per tile is estimated faster than the ranges (1536 rows behind 8000 keys
        // 281 -> 237 us) or the split-K tiles (1024 rows behind 2000 keys 84 -> 77 us, 1536 rows 130 -> 92).
        const bool whole_ahead = q_len >= 256 && whole.us < (n_splits >= 2 ? ranges_us : splitk_us);
        if (filled || whole_ahead || (pages && n_splits < 2)) return whole_tiles(pages);
        if (n_splits >= 2)
            return run_attention(ctx, kv, 1, layer, 1, &slot, &start_pos, &kv_valid, q_len, n_q_heads, q, 0,
                                 (long long)q_stride, gate, 0, (long long)gate_stride, scale, out, 0, (long long)o_stride,
                                 n_splits, split_blocks, pages);
        return run_attention(ctx, kv, 0, layer, 1, &slot, &start_pos, &kv_valid, q_len, n_q_heads, q, 0,
                             (long long)q_stride, gate, 0, (long long)gate_stride, scale, out, 0, (long long)o_stride);
    }
    // What the chunk kernel does not serve (head groups that are no multiple of 4, unaligned rows, quantised pages
    // that are not staged, a non-positive scale): the split-K kernel over GQA-packed tiles, like a verify pass -- or, where heads that do
    // not divide a tile's 32 rows leave some of them empty, tiles of 32 rows of ONE head, each walking all its keys, as long as they are
    // plentiful and the context is short or they are very plentiful (one row at 32k keys over 8 bits took 460 us as 16 one-head tiles
    // walking 32k keys each).  us a layer over 8 bits, one-head tiles / packed ones, of groups of 4 (32/8 heads of 128): 100 rows behind
    // 7,000 keys 86.1 / 58.8, 700 behind 2,000 91.8 / 80.1; of 8 (16/2 of 256): 256 rows behind 2,000 64.2 / 52.1, 700 of a prompt 76.6 / 67.5;
    // of 9 (36/4 of 128): 1,500 rows behind 3,000 256 / 297; of 5 (40/8 of 128): 700 behind 7,000 253 / 262.
    const long long head_tiles = (long long)((q_len + 31) / 32) * n_q_heads;
    const bool plentiful = 2 * head_tiles >= ctx->n_cus && (kv_valid <= 8192 || head_tiles >= 2LL * ctx->n_cus);
    auto in_tiles = [&](int kind) {
        return run_attention(ctx, kv, kind, layer, 1, &slot, &start_pos, &kv_valid, q_len, n_q_heads, q, 0, (long long)q_stride,
                             gate, 0, (long long)gate_stride, scale, out, 0, (long long)o_stride);
    };
    // (over fp16 pages the two ways mostly take the same -- 116 of 120 chunks of groups of one and two within 5 %, 16/8 heads of 128, 300 rows behind 2,000 keys 37.5 /
    // 38.6, 1,500 102.4 / 100.4, but 32/16 of 64, 100 rows behind 7,000, 52.9 / 37.8 --: one-head tiles, which need no partial results)
    if ((rows_left_empty || kv->bits == 16) && plentiful) return in_tiles(1);
    st = in_tiles(0);
    // (without memory for the splits' partial results, as inside a capture that would have to grow it: tiles of one head, which have none)
    if (plentiful && (st == TT_HIP_ERR_BUSY || st == TT_HIP_ERR_OUT_OF_MEMORY)) st = in_tiles(1);
    return st;
}

}  // extern "C"
