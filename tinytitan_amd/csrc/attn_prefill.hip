// Causal chunk (prefill) flash attention on gfx950 MFMA, K/V tiles staged in LDS,
// score and value wavefronts specialised.
//
// Same transposed formulation as the split-K kernel (a lane owns a query row):
//   S^T[key][row] = K . Q^T      A = K fragment from LDS,   B = Q^T fragment in registers
//   O^T[d][row]  += V^T . P^T    A = V^T fragment from LDS, B = P^T as it left S^T's registers
// with v_mfma_f32_32x32x16_f16.
//
// Work decomposition.  A workgroup serves 4 q heads of one KV head over 64 query rows, as two
// 32-row tiles processed one after the other: token tile n_tiles-1-i ("long"), then tile i
// ("short").  Tile i needs i+1 key blocks, its partner n_tiles-i, so every workgroup does the
// same number of MFMAs whatever i is -- the causal triangle is balanced by construction.
//
// Each (head, tile) is served by TWO wavefronts on the same SIMD:
//   * the score wave holds Q (64 registers at D = 256), computes S^T for key block j, runs the
//     online softmax (reference max, row sum) and leaves P^T -- already in MFMA B-operand
//     order -- plus the per-row rescale factors in LDS;
//   * the value wave holds O^T (128 accumulation registers at D = 256) and, one step behind,
//     accumulates P^T(j-1) against V(j-1).
// Neither needs more than half of the register file, so two waves fit per SIMD, and the
// hardware overlaps one wave's MFMAs with the other's softmax VALU work and LDS reads; eight
// waves per CU also issue LDS reads about 1.6x faster than four can (the per-wave issue rate
// is what limits a 4-wave design).  One workgroup barrier separates the steps, of one key block.
//
// Heads of 128 have half the matrix instructions for the same softmax, and a score wave is then most of a step: their two wavefronts a
// SIMD share the KEYS instead (attn_prefill_halves_kernel).
//
// K/V blocks stream L2 -> LDS with direct-to-LDS 128-bit loads (no registers), four stages
// deep, issued one or two steps ahead of their first use; the K fragment layout in HBM is the MFMA
// operand layout, V is permuted into it by the copy.
//
// The online softmax rescales lazily: a row's reference max only moves when its block max
// exceeds it by more than 8 (log2 units), so probabilities stay below 2^8 (well inside fp16's
// range) and the value wave rescales its accumulators a handful of times per row.
//
// Replaces attention_prefill_causal_q8 / attention_prefill_causal_tiled
// (sources/TinyTitanCore/Metal/Prefill/prefill.metal:1056-1313) dispatched by
// PrefillAttention.encodeCausal (sources/TinyTitan/Kernels/Attention/PrefillAttention.swift:165-258).
#include "chunk_plan.h"
#include "internal.h"
#include "wave_ops.h"

namespace tt {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));

struct PrefillArgs {
    const _Float16 *k_slot;  // page of kv head 0 of this slot
    const _Float16 *v_slot;
    const _Float16 *q;
    const _Float16 *gate;
    _Float16 *out;
    long long page_elems;
    long long q_stride, g_stride, o_stride;
    int group;     // q heads per kv head
    int hsubs;     // group / 4
    int n_tiles;   // ceil(q_len / 32)
    int n_pairs;   // ceil(n_tiles / 2); with single_tiles: n_tiles
    int single_tiles;  // 1: a workgroup takes ONE tile instead of a long and a short one
    int per_kvh;   // hsubs * n_pairs
    int xs;        // XCDs per kv head (8 / n_kv_heads), 0: plain mapping
    int n_kv_heads;
    int start, q_len, kv_valid;
    int window;  // sliding window (0: none): the row at position p sees keys [max(0, p + 1 - window), p + 1)
    int ring_blocks;  // ring cache: key block b lives in block b % ring_blocks of the page; 0 = where it is
    float scale_log2e;
    // Key splits (n_splits > 1): workgroup (base, split) walks key blocks [split * split_blocks,
    // (split + 1) * split_blocks) of each of its tiles and leaves unnormalised partials
    // (reference max, sum, O) in the split-K kernel's layout for its combine pass.
    int n_splits, split_blocks, base_grid;
    int xcd_chunk;  // key ranges with xs > 0: (range, tile, head set) items one XCD takes, ceil(per_kvh * n_splits / xs)
    float *part_o;   // [split][head * n_tiles + tile][32 rows][D]
    float *part_ml;  // [split][head * n_tiles + tile][32 rows][2]
};

namespace {

constexpr float kNegBig = -1.0e30f;
constexpr float kRescaleThreshold = 8.0f;
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

typedef __attribute__((address_space(3))) void *lds_ptr_t;
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

// 16 bytes per lane, global -> LDS without passing through registers: lane l's 16 bytes land at
// lds_addr + 16 l.  Issued as inline assembly on purpose: the compiler, when it sees an LDS DMA,
// guards every later LDS read with a full vmcnt(0) wait (it cannot tell the stages apart),
// which would turn a multi-stage prefetch into none.  Completion is tracked by hand instead:
// TT_WAIT_VMCNT before the barrier that publishes a stage.
__device__ __forceinline__ void copy16_global_to_lds(const void *base, unsigned lane_offset, unsigned lds_addr) {
    // base and lds_addr are wave-uniform by construction; say so, in case the compiler lost track
    const unsigned long long b = (unsigned long long)base;
    const unsigned b_hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(b >> 32));
    const unsigned b_lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)b);  // (the builtin returns a signed int)
    base = (const void *)(((unsigned long long)b_hi << 32) | (unsigned long long)b_lo);
    lds_addr = (unsigned)__builtin_amdgcn_readfirstlane((int)lds_addr);
    // m0 carries the LDS address of the copy.  The compiler owns m0 (it is a reserved register: naming it as a clobber is not honoured), but has
    // no use for it in the kernels that copy by this (tests/test_wait_states.py looks), so it is not put back.  Between a scalar write of m0 and a
    // copy into LDS belongs one wait state, which is nobody's to add but the block's own.
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %0" : : "s"(base), "v"(lane_offset), "s"(lds_addr) : "memory");
}

// N pieces of 1 KiB that lie one behind the other in both places (an instruction's offset counts for both).
template <int N>
__device__ __forceinline__ void copies_global_to_lds(const void *base, unsigned first, unsigned second, unsigned lds_addr) {
    static_assert(N == 2, "two copies");
    const unsigned long long b = (unsigned long long)base;
    const unsigned b_hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(b >> 32));
    const unsigned b_lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)b);
    base = (const void *)(((unsigned long long)b_hi << 32) | (unsigned long long)b_lo);
    lds_addr = (unsigned)__builtin_amdgcn_readfirstlane((int)lds_addr);
    unsigned saved_m0;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %1\n\tglobal_load_lds_dwordx4 %4, %1 offset:1024\n\ts_mov_b32 m0, %0"
                 : "=&s"(saved_m0)
                 : "s"(base), "v"(first), "s"(lds_addr), "v"(second)
                 : "memory");
}

// o *= alpha in place (written out the compiler moves all of o around in every step for the few that rescale).  Ahead of it the block's
// softmax, behind it two wait states before a matrix instruction reads.
__device__ __forceinline__ void rescale_tile(f16v &o, float alpha) {
#pragma unroll
    for (int j = 0; j < 16; j += 4) {
        float a0 = o[j], a1 = o[j + 1], a2 = o[j + 2], a3 = o[j + 3];
        asm volatile("v_mul_f32 %0, %4, %0\n\tv_mul_f32 %1, %4, %1\n\tv_mul_f32 %2, %4, %2\n\tv_mul_f32 %3, %4, %3\n\ts_nop 4"
                     : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3)
                     : "v"(alpha));
        o[j] = a0;
        o[j + 1] = a1;
        o[j + 2] = a2;
        o[j + 3] = a3;
    }
}

// vmcnt(n) only: leaves the LDS/scalar and export counters alone.
#define TT_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | (0x7 << 4) | (0xF << 8))

// One online-softmax step of the score wave on a block's scores: mask, move the row's reference
// max where the block max exceeds it by more than the threshold, and produce the
// probabilities (B operand of the two P.V k-steps) against the reference.  The row sum is taken
// over the ROUNDED probabilities, i.e. over exactly the weights the P.V MFMAs see, by v_fma_mix_f32: a half of either side
// joins an fp32 sum in one instruction that runs beside a matrix instruction of the SIMD's other wavefront.  (v_dot2_f32_f16, half as many,
// waits until the matrix pipe is free: 64 of them beside another wavefront's MFMAs take as long as those do, 64 of any other instruction
// here 1.25 times their own time.  64/8 heads of 64, 2,048 rows behind 4,000 keys 252.0 -> 235.3 us; 32/8 of 128, 4,096 behind 8,000
// 729 -> 719; heads of 256, whose softmax is a smaller part, the same.)  Returns the factor the row's accumulators must be scaled by before this block is added.
__device__ __forceinline__ float softmax_step(const f16v &s_raw, bool mask, int kbase, int lo, int lim, int g, float scale_log2e, float &m,
                                              float &l, h8 (&pf)[2]) {
    // The maximum is taken over the raw scores and scaled once (the host sends only chunks with scale > 0 here), and a
    // probability is one fused multiply-add and one exp2 off its raw score.
    float t[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) t[v] = s_raw[v];
    if (mask) {  // wave-uniform: only the blocks on or past the tile's diagonal, or at its window's lower edge
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int key = kbase + 8 * (v >> 2) + 4 * g + (v & 3);
            if (key >= lim || key < lo) t[v] = -INFINITY;
        }
    }
    float mx = fmaxf(t[0], t[1]);
#pragma unroll
    for (int v = 2; v < 16; v += 2) mx = fmaxf(fmaxf(t[v], t[v + 1]), mx);
    mx = max_across_halves(mx) * scale_log2e;
    const bool move = mx > m + kRescaleThreshold;  // a row's first visible block always moves
    const float m_new = move ? mx : m;
    const float alpha = move ? fast_exp2(m - m_new) : 1.0f;
    l *= alpha;
    m = m_new;
    float l_odd = 0.0f;  // (two sums: neither waits for the other's last addition)
#pragma unroll
    for (int v = 0; v < 16; v += 2) {
        const h2 p = {(_Float16)fast_exp2(__builtin_fmaf(t[v], scale_log2e, -m)), (_Float16)fast_exp2(__builtin_fmaf(t[v + 1], scale_log2e, -m))};
        asm("v_fma_mix_f32 %0, %1, 1.0, %0 op_sel_hi:[1,0,0]" : "+v"(l) : "v"(p));
        asm("v_fma_mix_f32 %0, %1, 1.0, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(l_odd) : "v"(p));
        pf[v >> 3][v & 7] = p[0];
        pf[v >> 3][(v & 7) + 1] = p[1];
    }
    l += l_odd;
    return alpha;
}

// Workgroup -> (kv head, head sub-group, tile pair); kv heads are spread over XCDs so
// that each XCD's L2 holds one kv head's K/V.
struct ChunkItem {
    int kvh, hsub, pair, split;
    bool longest_first;
};
__device__ __forceinline__ bool chunk_item(const PrefillArgs &a, ChunkItem &item) {
    int split = blockIdx.x / a.base_grid;
    const int wg = blockIdx.x - split * a.base_grid;  // base_grid is a multiple of 8: wg & 7 is still the XCD
    int kvh, r;
    if (a.xcd_chunk > 0) {
        // Key ranges: the (range, tile, head set) items of a kv head, range-major, are cut into as many runs as the kv
        // head has XCDs (workgroup b runs on XCD b % 8).  Every XCD gets the same number of workgroups whatever the
        // number of tiles -- dealt out tile by tile, 3 or 5 tiles per head set leave some XCDs with twice the work of
        // others -- and a range's K/V blocks are fetched into one L2, or two, instead of all of the kv head's.
        const int x = blockIdx.x & 7, j = blockIdx.x >> 3;
        kvh = x / a.xs;
        const int w = (x - kvh * a.xs) * a.xcd_chunk + j;
        if (w >= a.per_kvh * a.n_splits) return false;
        split = w / a.per_kvh;
        r = w - split * a.per_kvh;
    } else if (a.xs > 0) {
        const int x = wg & 7, y = wg >> 3;
        kvh = x / a.xs;
        r = y * a.xs + (x - kvh * a.xs);
    } else {
        kvh = wg / a.per_kvh;
        r = wg - kvh * a.per_kvh;
    }
    if (r >= a.per_kvh || kvh >= a.n_kv_heads) return false;
    // (whole tiles one by one: the head sets' longest tiles first, and so on down)
    item.longest_first = a.single_tiles && a.n_splits == 1;
    // (one division: each is a chain in front of the first load)
    const int per = item.longest_first ? a.hsubs : a.n_pairs, quotient = r / per, rest = r - quotient * per;
    item.kvh = kvh;
    item.hsub = item.longest_first ? rest : quotient;
    item.pair = item.longest_first ? quotient : rest;
    item.split = split;
    return true;
}

}  // namespace

template <int D>
__global__ __launch_bounds__(512, D == 64 ? 4 : 1) void attn_prefill_kernel(const PrefillArgs a) {
    constexpr int KS = D / 16;  // k-steps of S^T
    constexpr int MT = D / 32;  // 32-dim tiles of O^T
    constexpr int BLOCK_BYTES = 32 * D * 2;
    constexpr int RING = kChunkRing;
    constexpr int SLOT_BYTES = BLOCK_BYTES;
    constexpr int CHUNKS = BLOCK_BYTES / 1024;    // 1 KiB chunks per block (= KS = 2 MT)
    constexpr int CPW = CHUNKS / 4;               // copies one wave issues per step (K and V of a block over 8 waves)
    constexpr int V_OFF = RING * SLOT_BYTES;           // K ring, then V ring
    constexpr int P_OFF = 2 * RING * SLOT_BYTES;       // P^T: [2 steps][4 heads][2 k-steps][64 lanes][16 B]
    constexpr int P_STEP = 4 * 2048;
    constexpr int ALPHA_OFF = P_OFF + 2 * P_STEP;      // rescale factors: [2 steps][4 heads][32 rows] floats
    constexpr int LSUM_OFF = ALPHA_OFF + 2 * 4 * 128;  // row sums: [4 heads][32 rows] floats
    constexpr int STAGE_OFF = LSUM_OFF + 4 * 128;      // output rows on their way out: [4 heads][32 rows][32 dims + 16 B]
    constexpr int STAGE_PITCH = 64 + 16;
    extern __shared__ __attribute__((aligned(16))) char smem[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool value_wave = wave >= 4;
    const int w4 = wave & 3;
    const int li = lane & 31, g = lane >> 5;

    ChunkItem item;
    if (!chunk_item(a, item)) return;
    const int kvh = item.kvh, hsub = item.hsub, pair = item.pair, split = item.split;
    const bool longest_first = item.longest_first;
    const int head = kvh * a.group + hsub * 4 + w4;
    const _Float16 *kp = a.k_slot + (size_t)kvh * a.page_elems;
    const _Float16 *vp = a.v_slot + (size_t)kvh * a.page_elems;

    // Copies of step i: K of step i + RING and V of step i + RING - 2 (copies_ahead), of which this wave issues CPW one-KiB chunks.
    // Step j's blocks live in slot j % RING of their ring.  Past the end of the tile the
    // last block is copied again (into a slot nobody reads any more), so that every step puts
    // the same number of copies in flight and one constant vmcnt tracks them.
    const unsigned smem_base = (unsigned)(size_t)(lds_ptr_t)smem;
    const unsigned k_lane_offset = (unsigned)lane * 16u;
    const unsigned v_lane_offset = (unsigned)v_piece(D, li, g) * 2u;  // this lane's 16 bytes inside a V chunk gather
    int jb = 0;  // first key block of this workgroup's range in the current tile
    // Step j of the tile in hand lives in slot (j + slot_off) % ring.  When a second tile follows (carry_nb > 0:
    // it has that many blocks, from block 0), the copies past the end of the first fetch ITS first blocks -- a ring of K
    // and one of V are in LDS when the first tile's last step ends, in the slots that follow on, and the second tile starts
    // without waiting for memory.  (A wave copies and reads K or V, so the offset is that of its own ring.)
    int slot_off = 0, carry_nb = 0;
    auto page_block = [&](int block) { return a.ring_blocks ? block % a.ring_blocks : block; };
    const int my_chunk = w4 * CPW;
    // A step's copies: this wave's CPW one-KiB chunks of ONE block -- of K for the score waves (the LDS layout is the HBM
    // layout, fragment s is chunk s), of V for the value waves (gathered so that LDS holds fragment (mt, t) as [lane][8 halves]).  Where the block lies in the page and in the
    // ring is worked out ONCE per step (step_copies); a copy then costs two scalar adds on top of its load -- worked
    // out per copy it was 30 scalar instructions each, 120 to 145 a step in the instruction stream of a wave whose
    // matrix instructions wait behind them.
    struct StepCopies {
        const char *src;
        unsigned dst;
    };
    unsigned v_src_off[CPW];  // source offsets of this value wave's chunks inside a V block
#pragma unroll
    for (int c = 0; c < CPW; ++c) {
        const int chunk = my_chunk + c, mt = chunk >> 1, t = chunk & 1;
        v_src_off[c] = (unsigned)v_piece(D, 32 * mt, 2 * t) * 2u;
    }
    auto step_copies = [&](int i, int nb) {  // of step i; nb blocks in the range
        StepCopies sc;
        const int j = i + (value_wave ? copies_ahead(true) : copies_ahead(false));
        const _Float16 *page = value_wave ? vp : kp;
        sc.src = reinterpret_cast<const char *>(page + (size_t)page_block(copied_block(j, jb, nb, carry_nb)) * (32 * D)) + (value_wave ? 0 : my_chunk * 1024);
        sc.dst = smem_base + (unsigned)((value_wave ? V_OFF : 0) + in_ring(j + slot_off) * SLOT_BYTES + w4 * CPW * 1024);
        return sc;
    };
    auto issue_copy = [&](const StepCopies &sc, int c) {  // copy c (0 .. CPW-1)
        if (!value_wave) copy16_global_to_lds(sc.src + c * 1024, k_lane_offset, sc.dst + c * 1024);
        else copy16_global_to_lds(sc.src + v_src_off[c], v_lane_offset, sc.dst + c * 1024);
    };
    auto issue_step = [&](int i, int nb) {
        const StepCopies sc = step_copies(i, nb);
#pragma unroll
        for (int c = 0; c < CPW; ++c) issue_copy(sc, c);
    };

    char *const p_mine = smem + P_OFF + w4 * 2048 + lane * 16;  // + step parity * P_STEP, + k-step * 1024
    float *const alpha_mine = reinterpret_cast<float *>(smem + ALPHA_OFF) + w4 * 32 + li;  // + step parity * 128
    float *const lsum_mine = reinterpret_cast<float *>(smem + LSUM_OFF) + w4 * 32 + li;

    // Tiles in pairs (tile i with tile n - 1 - i: every workgroup the same number of key blocks under a causal
    // mask from position 0) -- or one tile each: where the keys are cut into ranges (deep in a context the tiles are equally
    // long anyway, and a workgroup with one tile leaves half the partial results of one with two), and where pairs would
    // leave CUs idle (estimate_chunk in chunk_plan.h), the longest tile first.
    const int n_passes = (a.single_tiles || pair == a.n_tiles - 1 - pair) ? 1 : 2;
    for (int pass = 0; pass < n_passes; ++pass) {
        // The long tile goes first: the short one then fills in behind it.
        const int tile = longest_first ? a.n_tiles - 1 - pair : a.single_tiles ? pair : (pass == 0 ? a.n_tiles - 1 - pair : pair);
        const int tok = tile * 32 + li;
        const bool valid = tok < a.q_len;
        const int lim = valid ? min(a.kv_valid, a.start + tok + 1) : 0;  // keys [lo, lim) are visible
        const int lo = (a.window > 0 && a.start + tok + 1 > a.window) ? a.start + tok + 1 - a.window : 0;
        // With a window the tile starts at the block of the first key its first row sees; the rows'
        // lower bounds differ, so the blocks up to the one of its last row's bound are masked too.
        const int tile_lo = (a.window > 0 && a.start + tile * 32 + 1 > a.window) ? a.start + tile * 32 + 1 - a.window : 0;
        const int window_block = tile_lo >> 5;
        const int last_lo_block = a.window > 0 ? (tile_lo + 31) >> 5 : -1;
        const int end = min(a.kv_valid, a.start + min(a.q_len, tile * 32 + 32));
        const int nb_tile = (end + 31) >> 5;                   // key blocks this tile needs
        const int mask_from = (a.start + tile * 32 + 1) >> 5;  // first block in which some row is masked by causality
        // This workgroup's share of them (all, without key splits); local step i is block jb + i
        jb = window_block + (a.n_splits > 1 ? split * a.split_blocks : 0);
        const int nb = (a.n_splits > 1 ? min(nb_tile, jb + a.split_blocks) : nb_tile) - jb;
        if (nb <= 0) continue;  // nothing of this tile in the range (the same for every wave)
        const int first_masked = min(mask_from, end >> 5);  // ... or cut by the valid length

        if (pass > 0) __syncthreads();  // every wave is done with the previous pass's LDS
        const bool carried = carry_nb > 0;  // this tile's first blocks came in behind the previous tile's last
        carry_nb = 0;
        if (pass == 0 && n_passes == 2 && a.n_splits == 1 && a.window == 0) {
            // the second tile's blocks: keys [0, its last row's position], from block 0
            const int end2 = min(a.kv_valid, a.start + min(a.q_len, pair * 32 + 32));
            carry_nb = max((end2 + 31) >> 5, 0);
        }
        if (!carried) {
            // K of steps 0 .. RING - 1, V of steps 0 .. RING - 3, each to a place of its own: nothing orders two copies in flight.
#pragma unroll
            for (int i = -copies_ahead(false); i < 0; ++i)
                if (!value_wave || i >= -copies_ahead(true)) issue_step(i, nb);
        }

        // End of step i.  What the next step reads from LDS, K(i+2) and V(i), was copied in step i + 2 - RING
        // and must have landed; the copies of the RING - 2 steps since may still fly.  Then the
        // barrier that publishes them and this step's P^T.
        auto end_step = [&]() {
            TT_WAIT_VMCNT((RING - 2) * CPW);
            __syncthreads();
        };

        // Step i (0 .. steps + 1): the score waves run the MFMAs of step i's blocks, the value waves those of
        // step i - 2's; both fetch the NEXT step's fragments from LDS into the registers the
        // MFMAs have just read, so that after the barrier the matrix pipe starts at once.
        // The two roles run separate loops (their register sets are disjoint that way) that
        // meet at the same barriers.
        if (!value_wave) {
            // Query fragments (B operand); rows of padding tokens are zero.
            h8 qf[KS];
            const _Float16 *qp = a.q + (long long)(valid ? tok : 0) * a.q_stride + (long long)head * D + 8 * g;
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const h8 x = *reinterpret_cast<const h8 *>(qp + 16 * s);
                qf[s] = valid ? x : (h8)(_Float16)0;
            }
            float m = kNegBig, l = 0.0f;
            TT_WAIT_VMCNT(0);  // the first stages and the query rows
            __syncthreads();
            h8 kf[KS];
#pragma unroll
            for (int t = 0; t < KS; ++t)
                kf[t] = *reinterpret_cast<const h8 *>(smem + slot_off * SLOT_BYTES + lane * 16 + t * 1024);
            __syncthreads();  // every score wave holds K of step 0: step 0 may refill its slot
#pragma nounroll
            for (int i = 0; i < nb; ++i) {
                const char *next = smem + in_ring(i + 1 + slot_off) * SLOT_BYTES + lane * 16;
                const StepCopies sc = step_copies(i, nb);
                f16v s = (f16v)0.0f;
#pragma unroll
                for (int t = 0; t < KS; ++t) {
                    s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[t], qf[t], s, 0, 0, 0);
                    kf[t] = *reinterpret_cast<const h8 *>(next + t * 1024);
                    // this step's copies, one at a time between MFMAs: a burst would stall the wave
                    // on the CU's vector memory path (64 B/clk for all eight waves)
                    if (t % (KS / CPW) == 0) issue_copy(sc, t / (KS / CPW));
                    __builtin_amdgcn_sched_barrier(0);
                }
                h8 pf[2];
                const int block = jb + i;
                const float alpha = softmax_step(s, block >= first_masked || block <= last_lo_block, block << 5, lo, lim, g, a.scale_log2e, m, l, pf);
                char *pdst = p_mine + (i & 1) * P_STEP;
#pragma unroll
                for (int t = 0; t < 2; ++t) *reinterpret_cast<h8 *>(pdst + t * 1024) = pf[t];
                if (g == 0) alpha_mine[(i & 1) * 128] = alpha;
                end_step();
            }
            issue_step(nb, nb);
            end_step();  // the value waves' last two steps
            issue_step(nb + 1, nb);
            end_step();
            const float lt = sum_across_halves(l);
            if (g == 0) {
                if (a.n_splits > 1) {  // partial: the row's reference max (log2 domain) and sum over this key range
                    float *ml = a.part_ml + ((((size_t)split * a.group * a.n_kv_heads + head) * a.n_tiles + tile) * 32 + li) * 2;
                    ml[0] = m;
                    ml[1] = lt;
                } else {
                    *lsum_mine = lt;
                }
            }
            TT_WAIT_VMCNT(0);
            __syncthreads();
        } else {
            f16v o[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) o[mt] = (f16v)0.0f;
            TT_WAIT_VMCNT(0);
            __syncthreads();
            __syncthreads();  // (the score waves fetch K of step 0 between these two)
            // Two steps behind the score wave: step j's P^T (written in step j) and V fragments are
            // fetched from LDS into registers during step j + 1 and consumed in step j + 2, so
            // that the MFMAs of a step start right after its barrier.
            issue_step(0, nb);
            end_step();  // step 0: the score waves' first
            issue_step(1, nb);
            h8 vf[2 * MT], pf[2];
#pragma unroll
            for (int c = 0; c < 2 * MT; ++c)
                vf[c] = *reinterpret_cast<const h8 *>(smem + V_OFF + slot_off * SLOT_BYTES + lane * 16 + c * 1024);
#pragma unroll
            for (int t = 0; t < 2; ++t) pf[t] = *reinterpret_cast<const h8 *>(p_mine + t * 1024);
            float alpha = alpha_mine[0];
            end_step();  // step 1
#pragma nounroll
            for (int i = 2; i <= nb + 1; ++i) {
                const int jn = i - 1;  // the step fetched in this one (past the last one: stale but harmless data)
                const char *next = smem + V_OFF + in_ring(jn + slot_off) * SLOT_BYTES + lane * 16;
                const char *psrc = p_mine + (jn & 1) * P_STEP;
                const StepCopies sc = step_copies(i, nb);
                if (__any(alpha != 1.0f)) {
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) o[mt] *= alpha;
                }
                alpha = alpha_mine[(jn & 1) * 128];
                auto multiply = [&](int u, int mt, int t) {  // the u-th: k-step t of 32-dim tile mt
                    const int c = 2 * mt + t;  // the fragment's place in the slot
                    o[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[c], pf[t], o[mt], 0, 0, 0);
                    vf[c] = *reinterpret_cast<const h8 *>(next + c * 1024);
                    if (u % (KS / CPW) == 0) issue_copy(sc, u / (KS / CPW));
                    __builtin_amdgcn_sched_barrier(0);
                };
                if constexpr (D == 256) {
                    // All k-steps of a 32-dim tile back to back: consecutive MFMAs on one accumulator
                    // forward it inside the matrix pipe instead of going through the register file.
                    h8 pn[2];
#pragma unroll
                    for (int t = 0; t < 2; ++t) pn[t] = *reinterpret_cast<const h8 *>(psrc + t * 1024);
#pragma unroll
                    for (int u = 0; u < 2 * MT; ++u) multiply(u, u / 2, u % 2);
#pragma unroll
                    for (int t = 0; t < 2; ++t) pf[t] = pn[t];
                } else {
                    // One k-step after the other: its P^T is read into the registers that its MFMAs are done with.
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
#pragma unroll
                        for (int mt = 0; mt < MT; ++mt) multiply(t * MT + mt, mt, t);
                        pf[t] = *reinterpret_cast<const h8 *>(psrc + t * 1024);
                    }
                }
                end_step();
            }
            TT_WAIT_VMCNT(0);
            __syncthreads();  // the row sums are in LDS
            // Lane (li, g), register v of tile mt holds dim 32 mt + 8 (v / 4) + 4 g + v % 4 of row li.
            // (The lane's addresses are worked out here, not in front of the tiles: no register is left to keep them in.)
            int row_here = li;
            asm volatile("" : "+v"(row_here));
            if (a.n_splits > 1) {
                // Partial: the unnormalised accumulators, for the combine pass.
                float *po = a.part_o + ((((size_t)split * a.group * a.n_kv_heads + head) * a.n_tiles + tile) * 32 + row_here) * D + 4 * g;
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int vq = 0; vq < 4; ++vq) {
                        const f4 x = {o[mt][4 * vq], o[mt][4 * vq + 1], o[mt][4 * vq + 2], o[mt][4 * vq + 3]};
                        *reinterpret_cast<f4 *>(po + 32 * mt + 8 * vq) = x;
                    }
            } else {
                // Epilogue: normalise, gate in fp32, one fp16 round, store.  The rounded values go through LDS, one
                // 32-dim tile of the wave's 32 rows at a time (a region of their own: the rings may already hold the
                // next tile's blocks), so that a store instruction writes 64 contiguous bytes of 16 rows -- 8-byte
                // pieces straight from the accumulator layout took the value waves ~5 us per tile.
                char *const stage = smem + STAGE_OFF + w4 * (32 * STAGE_PITCH);
                const float lt = *lsum_mine;
                const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
                // A tile's gate values are asked for one tile ahead, by every lane (a row past the chunk's end reads row 0's): under a
                // condition of its own each load was waited for where it stood.  (Together with a cheaper division: 16/2 heads of 256, position 0,
                // 4,096 rows 155 -> 149 us, 2,048 69 -> 64.5, 1,024 40 -> 36.5; 32/8 of 128, 4,096 rows 179 -> 172.)
                const bool gated = a.gate != nullptr;
                const _Float16 *const gate_row = a.gate + (long long)(valid ? tile * 32 + row_here : 0) * a.g_stride + (long long)head * D + 4 * g;
                h4 gate[2][4];
                auto load_gate = [&](int mt) {
#pragma unroll
                    for (int vq = 0; vq < 4; ++vq) gate[mt & 1][vq] = *reinterpret_cast<const h4 *>(gate_row + 32 * mt + 8 * vq);
                };
                if (gated) load_gate(0);
                const int out_row = lane >> 2, out_piece = lane & 3;  // a store: lane l writes piece l % 4 of row l / 4 (+ 16)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    if (gated && mt + 1 < MT) load_gate(mt + 1);
#pragma unroll
                    for (int vq = 0; vq < 4; ++vq) {
                        float r4[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) r4[i] = o[mt][4 * vq + i] * inv;
                        if (gated) {
#pragma unroll
                            for (int i = 0; i < 4; ++i) r4[i] *= sigmoid((float)gate[mt & 1][vq][i]);
                        }
                        const h4 hv = {(_Float16)r4[0], (_Float16)r4[1], (_Float16)r4[2], (_Float16)r4[3]};
                        *reinterpret_cast<h4 *>(stage + li * STAGE_PITCH + (8 * vq + 4 * g) * 2) = hv;
                    }
#pragma unroll
                    for (int half = 0; half < 2; ++half) {
                        const int row = 16 * half + out_row;
                        const h8 x = *reinterpret_cast<const h8 *>(stage + row * STAGE_PITCH + out_piece * 16);
                        const int t = tile * 32 + row;
                        if (t < a.q_len)
                            *reinterpret_cast<h8 *>(a.out + (long long)t * a.o_stride + (long long)head * D + 32 * mt + out_piece * 8) = x;
                    }
                }
            }
        }
        if (carry_nb > 0) slot_off = in_ring(slot_off + nb);  // where the next tile's first step sits
    }
}


// Heads of 128: the two wavefronts of a SIMD share a (head, tile) by KEYS -- of a step's two blocks wavefront w4 takes the first,
// w4 + 4 the second -- and each does all of its block's work: scores, softmax, values.  P^T stays in its registers, and a block's 16 matrix instructions
// stand against one softmax in either wavefront, where a score wave had 16 and two softmaxes a step and its value wave 16 and none.
//
// What bounds a step is what two instruction streams issue on one SIMD (16 matrix instructions of 33 cycles and about 130 others each,
// and the issue goes to the older wavefront first), so they are kept half a step apart: between two barriers the first half goes softmax,
// values, next scores and the second values, scores, softmax, a softmax beside the other's matrix instructions, which also have the
// higher priority.  The loop keeps its places as running sums (`look` works one out anew where a page's ring or the range ends): 75 scalar
// instructions a step, with each place from the step's number, were 7 %.  The halves meet at the tile's end, each writing out half of the dims.
// 32/8 heads, 777 rows behind a window of 4,096 keys 79.5 -> 70 us (a step of 0.96 -> 0.86 us; its matrix instructions and barrier alone 0.64),
// 4,096 rows behind 8,000 keys 729 -> 659 (0.93 -> 1.02 PFLOP/s), from position 0 179 -> 161, 128 rows behind 32,000
// 97.6 -> 88.  Measured and dropped: both halves in step (2,144 instead of 1,640 cycles by the issue model; 84 us), copies five steps ahead (the same),
// all of a step's copies in one run or in other places (the same to 1 %), the higher priority for the softmax or for the younger half (0 to -4 %).
template <int D>
__global__ __launch_bounds__(512, 2) void attn_prefill_halves_kernel(const PrefillArgs a) {
    constexpr int KS = D / 16, MT = D / 32;
    constexpr int BLOCK_BYTES = 32 * D * 2, CHUNKS = BLOCK_BYTES / 1024;
    constexpr int CPW = CHUNKS / 4;  // copies of K, and of V, that one wave issues per step: a quarter of its own block
    constexpr int RING = kHalvesRing, SLOT_BYTES = 2 * BLOCK_BYTES, RING_BYTES = RING * SLOT_BYTES;
    static_assert((RING_BYTES & (RING_BYTES - 1)) == 0, "places go round by a mask");
    constexpr int V_OFF = RING_BYTES, X_OFF = 2 * RING_BYTES;  // X: what the halves hand each other, then rows on their way out
    constexpr int STAGE_PITCH = 64 + 16;
    extern __shared__ __attribute__((aligned(16))) char smem[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = wave >> 2, w4 = wave & 3;
    const int li = lane & 31, g = lane >> 5;

    ChunkItem item;
    if (!chunk_item(a, item)) return;
    const int pair = item.pair, split = item.split;
    const int head = item.kvh * a.group + item.hsub * 4 + w4;
    const _Float16 *kp = a.k_slot + (size_t)item.kvh * a.page_elems;
    const _Float16 *vp = a.v_slot + (size_t)item.kvh * a.page_elems;

    // Copies of a step: this wavefront's quarter of its half's block, of K and of V.  K lies in HBM as in LDS; of V a
    // 16-byte piece per lane, gathered so that LDS holds fragment (mt, t) as [lane][8 halves].
    const unsigned smem_base = (unsigned)(size_t)(lds_ptr_t)smem;
    const unsigned k_lane_offset = (unsigned)(w4 * CPW * 1024 + lane * 16);
    unsigned v_lane_offset[CPW];  // (the second copy's offset of 1024 counts for both places, and none may be below zero)
#pragma unroll
    for (int c = 0; c < CPW; ++c) {
        const int chunk = w4 * CPW + c;
        v_lane_offset[c] = (unsigned)(v_piece(D, li, g) + v_piece(D, 32 * (chunk >> 1), 2 * (chunk & 1))) * 2u + 1024u * (CPW - 1 - c);
    }
    const unsigned copy_base = smem_base + (unsigned)(half * BLOCK_BYTES + w4 * CPW * 1024);
    const int wrap = a.ring_blocks ? a.ring_blocks : 0x40000000;
    unsigned slot_off = 0;  // where the tile's step 0 sits in the rings, in bytes
    bool carried = false;   // the tile's first blocks came in behind the last of the one before
    // What step i + 1 reads was copied in step i - 1 or before.
    auto end_step = [&]() {
        TT_WAIT_VMCNT(2 * CPW);
        __syncthreads();
    };

    const int n_passes = (a.single_tiles || pair == a.n_tiles - 1 - pair) ? 1 : 2;
    for (int pass = 0; pass < n_passes; ++pass) {
        const int tile = item.longest_first ? a.n_tiles - 1 - pair : a.single_tiles ? pair : (pass == 0 ? a.n_tiles - 1 - pair : pair);
        const int tok = tile * 32 + li;
        const bool valid = tok < a.q_len;
        const int lim = valid ? min(a.kv_valid, a.start + tok + 1) : 0;  // keys [lo, lim) are visible
        const int lo = (a.window > 0 && a.start + tok + 1 > a.window) ? a.start + tok + 1 - a.window : 0;
        const int tile_lo = (a.window > 0 && a.start + tile * 32 + 1 > a.window) ? a.start + tile * 32 + 1 - a.window : 0;
        const int window_block = tile_lo >> 5;
        const int last_lo_block = a.window > 0 ? (tile_lo + 31) >> 5 : -1;
        const int end = min(a.kv_valid, a.start + min(a.q_len, tile * 32 + 32));
        const int nb_tile = (end + 31) >> 5;                   // key blocks this tile needs
        const int mask_from = (a.start + tile * 32 + 1) >> 5;  // first block in which some row is masked by causality
        const int jb = window_block + (a.n_splits > 1 ? split * a.split_blocks : 0);
        const int nb = (a.n_splits > 1 ? min(nb_tile, jb + a.split_blocks) : nb_tile) - jb;
        if (nb <= 0) continue;  // nothing of this tile in the range (the same for every wave)
        const int steps = (nb + 1) / 2, mine = (nb + 1 - half) / 2;  // blocks jb + 2 i + half, i < mine
        const int first_masked = min(mask_from, end >> 5);

        if (pass > 0) __syncthreads();  // every wave is done with the other tile's LDS
        // The tile that follows takes its first blocks from the copies behind this one's last: from the block of the first key its first row sees.
        int next_first = 0, next_nb = 0;
        if (pass == 0 && n_passes == 2 && a.n_splits == 1) {
            if (a.window > 0) next_first = max(a.start + pair * 32 + 1 - a.window, 0) >> 5;
            next_nb = ((min(a.kv_valid, a.start + min(a.q_len, pair * 32 + 32)) + 31) >> 5) - next_first;
        }
        // Where the copies stand: sources of the next step's, its place, and how many steps run on in the page before that takes
        // another look (a ring's end, the range's last block, and behind that each one).
        const char *k_src, *v_src;
        unsigned copy_off = slot_off;
        int copy_step = carried ? kHalvesAhead : 0, run = 0, left = 0;
        if (carried) copy_off = (copy_off + kHalvesAhead * SLOT_BYTES) & (RING_BYTES - 1);
        auto look = [&]() {
            copy_step += run;
            const int phys = halves_block(copy_step, half, jb, nb, next_first, next_nb) % wrap;
            run = copy_step < mine ? min(mine - copy_step, (wrap - phys + 1) / 2) : 1;
            left = run;
            const size_t at = (size_t)(unsigned)phys * BLOCK_BYTES;
            k_src = reinterpret_cast<const char *>(kp) + at;
            v_src = reinterpret_cast<const char *>(vp) + at - 1024 * (CPW - 1);
        };
        look();
        auto copy_k = [&]() { copies_global_to_lds<CPW>(k_src, k_lane_offset, k_lane_offset, copy_base + copy_off); };
        auto copy_v = [&]() {  // behind copy_k
            copies_global_to_lds<CPW>(v_src, v_lane_offset[0], v_lane_offset[CPW - 1], copy_base + V_OFF + copy_off);
            k_src += SLOT_BYTES;
            v_src += SLOT_BYTES;
            copy_off = (copy_off + SLOT_BYTES) & (RING_BYTES - 1);
            if (--left == 0) look();
        };
        if (!carried) {
#pragma unroll
            for (int i = 0; i < kHalvesAhead - 1; ++i) {
                copy_k();
                copy_v();
            }
        }
        unsigned k_read = slot_off, v_read = slot_off;  // where the step lies whose K, V are read next
        // Blocks jb + 2 i + half with plain_from <= i < plain_from + plain need no mask.
        const int plain_from = last_lo_block < jb + half ? 0 : (last_lo_block - jb - half) / 2 + 1;
        const unsigned plain = (unsigned)max((first_masked - jb - half + 1) / 2 - plain_from, 0);
        h8 qf[KS];
        const _Float16 *qp = a.q + (long long)(valid ? tok : 0) * a.q_stride + (long long)head * D + 8 * g;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const h8 x = *reinterpret_cast<const h8 *>(qp + 16 * s);
            qf[s] = valid ? x : (h8)(_Float16)0;
        }
        float m = kNegBig, l = 0.0f;
        f16v o[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) o[mt] = (f16v)0.0f;
        TT_WAIT_VMCNT(0);  // the first steps' blocks and the query rows
        if (!carried) { copy_k(); copy_v(); }
        __syncthreads();
        h8 kf[KS], vf[2 * MT], pf[2];
        f16v s1;
        const char *const my_lds = smem + half * BLOCK_BYTES + lane * 16;
#pragma unroll
        for (int t = 0; t < KS; ++t) kf[t] = *reinterpret_cast<const h8 *>(my_lds + slot_off + t * 1024);

        // Scores of the block whose K is in registers.
        auto scores = [&]() {
            s1 = (f16v)0.0f;
#pragma unroll
            for (int t = 0; t < KS; ++t) s1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[t], qf[t], s1, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        // Its probabilities; its V is read meanwhile.
        auto weigh = [&](int i) {
            __builtin_amdgcn_s_setprio(0);
            const char *v_now = my_lds + V_OFF + v_read;
            v_read = (v_read + SLOT_BYTES) & (RING_BYTES - 1);
#pragma unroll
            for (int t = 0; t < 2 * MT; ++t) vf[t] = *reinterpret_cast<const h8 *>(v_now + t * 1024);
            __builtin_amdgcn_sched_barrier(0);
            const float alpha = softmax_step(s1, (unsigned)(i - plain_from) >= plain, (jb + 2 * i + half) << 5, lo, lim, g, a.scale_log2e, m, l, pf);
            if (__any(alpha != 1.0f)) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) rescale_tile(o[mt], alpha);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        // ... and its values; the next block's K is read meanwhile, and the step's copies go out.
        auto values = [&]() {
            __builtin_amdgcn_s_setprio(1);
            k_read = (k_read + SLOT_BYTES) & (RING_BYTES - 1);
            const char *k_next = my_lds + k_read;
#pragma unroll
            for (int u = 0; u < 2 * MT; ++u) {
                const int mt = u % MT, t = u / MT;
                o[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[2 * mt + t], pf[t], o[mt], 0, 0, 0);
                kf[u] = *reinterpret_cast<const h8 *>(k_next + u * 1024);
                if (u == 1) copy_k();
                if (u == MT + 1) copy_v();
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        static_assert(KS == 2 * MT, "a K fragment per value MFMA");
        auto values_of_last = [&]() {
#pragma unroll
            for (int u = 0; u < 2 * MT; ++u) o[u % MT] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[2 * (u % MT) + u / MT], pf[u / MT], o[u % MT], 0, 0, 0);
        };
        if (half == 0) {
            scores();
#pragma nounroll
            for (int i = 0; i < steps; ++i) {
                weigh(i);
                values();
                scores();
                end_step();
            }
        } else {
            copy_k();
            copy_v();
            scores();
            if (mine > 0) weigh(0);
            end_step();
#pragma nounroll
            for (int i = 1; i < mine; ++i) {
                values();
                scores();
                weigh(i);
                end_step();
            }
            if (mine > 0) {
                if (mine < steps) {  // (an odd number of blocks: the last step is the other half's)
                    copy_k();
                    copy_v();
                    end_step();
                }
                values_of_last();
            }
        }
        TT_WAIT_VMCNT(0);  // no copy of this tile is on its way when the next one's begin
        // The halves' results.  Every wave has 8 KiB: X, and the places in the rings that the last step's copies would have taken (the
        // next tile's first three steps are in the others).  What it hands over -- (reference max, sum), then the dims that the
        // other wave writes out -- goes through its own 8 KiB, but the pair first through the OTHER's: whoever reads a place is the one who writes it next, so
        // one barrier behind each is all the order there is.
        const int mt0 = half * (MT / 2);  // the 32-dim tiles that this wave writes out: mt0 .. mt0 + MT / 2 - 1
        const unsigned last_slot = (slot_off + (unsigned)(steps + RING - 1) * SLOT_BYTES) & (RING_BYTES - 1);
        auto place_of = [&](int w) { return smem + lane * 16 + (w < 4 ? X_OFF + w * 8192 : (w < 6 ? (int)last_slot : V_OFF + (int)last_slot) + (w & 1) * 8192); };
        char *const x_mine = place_of(wave), *const x_other = place_of(wave ^ 4);
        l = sum_across_halves(l);
        *reinterpret_cast<float2 *>(x_other) = float2{m, l};
        __syncthreads();
        // The rows' gate values are asked for now, by every lane (a row past the chunk's end reads row 0's): behind the exchange they
        // would be a trip to memory of their own.
        const bool gated = a.gate != nullptr && a.n_splits == 1;
        h4 gate[MT / 2][4];
        if (gated) {
            const _Float16 *const gate_row = a.gate + (long long)(valid ? tok : 0) * a.g_stride + (long long)head * D + 32 * mt0 + 4 * g;
#pragma unroll
            for (int r = 0; r < MT / 2; ++r)
#pragma unroll
                for (int vq = 0; vq < 4; ++vq) gate[r][vq] = *reinterpret_cast<const h4 *>(gate_row + 32 * r + 8 * vq);
        }
        const float2 other = *reinterpret_cast<const float2 *>(x_mine);
        const float top = fmaxf(m, other.x), scale_mine = fast_exp2(m - top), scale_other = fast_exp2(other.x - top);
        l = l * scale_mine + other.y * scale_other;
        m = top;
        f16v result[MT / 2];
#pragma unroll
        for (int r = 0; r < MT / 2; ++r)
#pragma unroll
            for (int vq = 0; vq < 4; ++vq) {
                f4 give;
#pragma unroll
                for (int v = 0; v < 4; ++v) {  // (half is uniform over the wave: selected register by register)
                    give[v] = half == 0 ? o[MT / 2 + r][4 * vq + v] : o[r][4 * vq + v];
                    result[r][4 * vq + v] = (half == 0 ? o[r][4 * vq + v] : o[MT / 2 + r][4 * vq + v]) * scale_mine;
                }
                *reinterpret_cast<f4 *>(x_mine + (4 * r + vq) * 1024) = give;
            }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < MT / 2; ++r)
#pragma unroll
            for (int vq = 0; vq < 4; ++vq) {
                const f4 x = *reinterpret_cast<const f4 *>(x_other + (4 * r + vq) * 1024);
#pragma unroll
                for (int v = 0; v < 4; ++v) result[r][4 * vq + v] += x[v] * scale_other;
            }
        if (a.n_splits > 1) {
            const size_t row = (((size_t)split * a.group * a.n_kv_heads + head) * a.n_tiles + tile) * 32 + li;
            if (half == 0 && g == 0) {
                a.part_ml[row * 2] = m;
                a.part_ml[row * 2 + 1] = l;
            }
            float *po = a.part_o + row * D + 4 * g;
#pragma unroll
            for (int r = 0; r < MT / 2; ++r)
#pragma unroll
                for (int vq = 0; vq < 4; ++vq) {
                    const f4 x = {result[r][4 * vq], result[r][4 * vq + 1], result[r][4 * vq + 2], result[r][4 * vq + 3]};
                    *reinterpret_cast<f4 *>(po + 32 * (mt0 + r) + 8 * vq) = x;
                }
        } else {
            char *const stage = x_other - lane * 16;  // (which this wave alone has read)
            const float inv = l > 0.0f ? 1.0f / l : 0.0f;
            const int out_row = lane >> 2, out_piece = lane & 3;
#pragma unroll
            for (int r = 0; r < MT / 2; ++r) {
#pragma unroll
                for (int vq = 0; vq < 4; ++vq) {
                    float r4[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) r4[i] = result[r][4 * vq + i] * inv;
                    if (gated) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) r4[i] *= sigmoid((float)gate[r][vq][i]);
                    }
                    const h4 hv = {(_Float16)r4[0], (_Float16)r4[1], (_Float16)r4[2], (_Float16)r4[3]};
                    *reinterpret_cast<h4 *>(stage + li * STAGE_PITCH + (8 * vq + 4 * g) * 2) = hv;
                }
#pragma unroll
                for (int part = 0; part < 2; ++part) {
                    const int row = 16 * part + out_row;
                    const h8 x = *reinterpret_cast<const h8 *>(stage + row * STAGE_PITCH + out_piece * 16);
                    const int t = tile * 32 + row;
                    if (t < a.q_len)
                        *reinterpret_cast<h8 *>(a.out + (long long)t * a.o_stride + (long long)head * D + 32 * (mt0 + r) + out_piece * 8) = x;
                }
            }
        }
        carried = next_nb > 0;
        if (carried) slot_off = (slot_off + (unsigned)steps * SLOT_BYTES) & (RING_BYTES - 1);  // where its first step sits
    }
}


// The kernel wants 4 q heads per KV head in a workgroup and 16-byte aligned rows; anything
// else is served by the split-K kernel.
bool prefill_kernel_serves(int n_q_heads, int n_kv_heads, int head_dim, bool aligned) {
    const int group = n_q_heads / n_kv_heads;
    return aligned && group % 4 == 0 && (head_dim == 256 || head_dim == 128 || head_dim == 64);
}

// the rings of K and V (128, 64 and 32 KiB at D = 256, 128 and 64) + P^T hand-over (16 KiB) + rescale factors and row sums + the output rows' staging (10 KiB)
static constexpr int prefill_lds_bytes(int D) { return 2 * kChunkRing * 32 * D * 2 + 2 * 4 * 2048 + 2 * 4 * 128 + 4 * 128 + 4 * 32 * 80; }

// ... the rings of the kernel over halves of the keys (128 KiB at D = 128) + the places that its wavefronts hand their results over in
static constexpr int prefill_halves_lds_bytes(int D) { return 2 * kHalvesRing * 2 * 32 * D * 2 + 8 * 4096; }
static_assert(prefill_lds_bytes(256) <= 160 * 1024 && prefill_halves_lds_bytes(128) <= 160 * 1024, "a CU's LDS");

int configure_prefill_kernels(tt_hip_ctx *ctx) {
    auto configure = [](const void *kernel, int lds) { return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds); };
    hipError_t e = configure(reinterpret_cast<const void *>(attn_prefill_kernel<256>), prefill_lds_bytes(256));
    if (e == hipSuccess) e = configure(reinterpret_cast<const void *>(attn_prefill_kernel<128>), prefill_lds_bytes(128));
    if (e == hipSuccess) e = configure(reinterpret_cast<const void *>(attn_prefill_kernel<64>), prefill_lds_bytes(64));
    if (e == hipSuccess) e = configure(reinterpret_cast<const void *>(attn_prefill_halves_kernel<128>), prefill_halves_lds_bytes(128));
    return e == hipSuccess ? TT_HIP_OK : hip_fail(ctx, e, "hipFuncSetAttribute(chunk kernel max dynamic LDS)");
}

// (the kernels' LDS limits were raised when the first context on this device was created)
template <typename F>
static int launch_chunk(tt_hip_ctx *ctx, F kernel, const PrefillArgs &args, unsigned grid, int lds) {
    launch_profiled(ctx, kernel, dim3(grid), dim3(512), (unsigned)lds, args);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? TT_HIP_OK : hip_fail(ctx, e, "attn_prefill_kernel launch");
}

int launch_prefill(tt_hip_ctx *ctx, tt_hip_kv *kv, int layer, int slot, int start, int q_len, int kv_valid,
                   int n_q_heads, const tt_half *q, long long q_stride, const tt_half *gate, long long g_stride,
                   float scale, tt_half *out, long long o_stride, int n_splits, int split_blocks, float *part_o,
                   float *part_ml, const PageSource *pages, int window, bool single_tiles) {
    PrefillArgs a{};
    a.window = window;
    if (!pages && kv->bits != 16) return TT_HIP_ERR_INVALID_ARGUMENT;  // this kernel reads fp16 pages only
    const size_t slot_off = (size_t)slot * kv->n_kv_heads * kv->page_elems();
    a.k_slot = pages ? pages->k : kv->k[layer] + slot_off;
    a.v_slot = pages ? pages->v : kv->v[layer] + slot_off;
    a.q = reinterpret_cast<const _Float16 *>(q);
    a.gate = reinterpret_cast<const _Float16 *>(gate);
    a.out = reinterpret_cast<_Float16 *>(out);
    a.page_elems = pages ? pages->page_elems : (long long)kv->page_elems();
    a.ring_blocks = pages ? pages->ring_blocks : kv->ring_blocks();
    a.q_stride = q_stride;
    a.g_stride = g_stride;
    a.o_stride = o_stride;
    a.group = n_q_heads / kv->n_kv_heads;
    a.hsubs = a.group / 4;
    a.n_tiles = (q_len + 31) / 32;
    a.single_tiles = n_splits > 1 || single_tiles ? 1 : 0;
    a.n_pairs = a.single_tiles ? a.n_tiles : (a.n_tiles + 1) / 2;
    a.per_kvh = a.hsubs * a.n_pairs;
    a.n_kv_heads = kv->n_kv_heads;
    a.xs = (kv->n_kv_heads <= 8 && 8 % kv->n_kv_heads == 0) ? 8 / kv->n_kv_heads : 0;
    a.start = start;
    a.q_len = q_len;
    a.kv_valid = kv_valid;
    a.scale_log2e = scale * 1.4426950408889634f;
    unsigned grid;
    if (a.xs > 0) grid = 8u * (unsigned)((a.per_kvh + a.xs - 1) / a.xs);
    else grid = (unsigned)(a.per_kvh * kv->n_kv_heads);
    a.base_grid = (int)grid;
    a.n_splits = n_splits > 1 ? n_splits : 1;
    a.split_blocks = split_blocks;
    a.part_o = part_o;
    a.part_ml = part_ml;
    if (a.n_splits > 1 && (!part_o || !part_ml || split_blocks <= 0)) return TT_HIP_ERR_INVALID_ARGUMENT;
    grid *= (unsigned)a.n_splits;
    a.xcd_chunk = 0;
    if (a.n_splits > 1 && a.xs > 0) {
        a.xcd_chunk = (a.per_kvh * a.n_splits + a.xs - 1) / a.xs;
        grid = 8u * (unsigned)a.xcd_chunk;
    }
    const int walk = a.n_splits > 1 ? std::min(split_blocks, most_tile_blocks(start, q_len, kv_valid, window))
                                    : most_tile_blocks(start, q_len, kv_valid, window);
    switch (kv->head_dim) {
        case 256: return launch_chunk(ctx, attn_prefill_kernel<256>, a, grid, prefill_lds_bytes(256));
        case 128:
            if (halves_of_keys(walk, (long long)grid, ctx->n_cus)) return launch_chunk(ctx, attn_prefill_halves_kernel<128>, a, grid, prefill_halves_lds_bytes(128));
            return launch_chunk(ctx, attn_prefill_kernel<128>, a, grid, prefill_lds_bytes(128));
        case 64: return launch_chunk(ctx, attn_prefill_kernel<64>, a, grid, prefill_lds_bytes(64));
        default: return TT_HIP_ERR_SHAPE;
    }
}

}  // namespace tt
