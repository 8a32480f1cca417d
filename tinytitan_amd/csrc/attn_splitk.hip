// Split-K flash attention over the swizzled KV pages (fp16 values, or 8 / 4-bit levels
// dequantised in registers; linear pages or a ring): GQA decode, multi-row verify and causal
// prefill for the shapes the chunk kernel does not take, each with an optional sliding
// window, on gfx950 MFMA.
//
// Formulation (everything transposed so that per-query-row state is per-lane):
//   S^T[key][row]  = K[key][:] . Q[row][:]        A = K fragment,  B = Q^T fragment
//   O^T[d][row]   += V^T[d][key] * P^T[key][row]  A = V^T fragment, B = P^T fragment
// A lane owns one query row (column of S^T / O^T): the running max, the running
// sum and the rescale factor are plain per-lane scalars, the key reduction is
// in-register plus one or two cross-lane steps, and P goes from the first
// contraction's result registers straight into the second one's B operand
// because the V page stores keys in exactly that order.
//
// Replaces attention_decode_partial / attention_decode_combine
// (sources/TinyTitanCore/Metal/Attention/attention.metal:162-269, :395-437) and,
// for multi-row tiles, attention_prefill_causal_q8
// (sources/TinyTitanCore/Metal/Prefill/prefill.metal:1172-1313).
#include <type_traits>

#include "chunk_plan.h"
#include "internal.h"
#include "wave_ops.h"

namespace tt {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));

constexpr float kNegBig = -1.0e30f;  // finite stand-in for "no key seen yet"
// A row's reference maximum only moves when a block's maximum exceeds it by more than this (log2
// units): probabilities stay below 2^4, and the accumulators -- 144 registers that the 32-row
// variant keeps in AGPRs, so a rescale is three instructions each -- are rescaled a handful of
// times per row instead of in almost every block (with 32 rows per wave SOME row sees a new
// maximum in nearly every block).  Any reference works for the merges: m, l and O move together.
// Over fp16 pages the threshold is 8 (probabilities below 2^8, well inside fp16): a wavefront that walks only a few
// dozen blocks, as in a sparse chunk, spends a visible share of them rescaling.  Over quantised pages it stays 4: there
// a probability is multiplied by a group's scale (up to 514) and a boost of 4 before it becomes an fp16 operand.
constexpr float kLazyRescale = 4.0f, kLazyRescaleHalfPages = 8.0f;
constexpr int kLdsPad = 4;           // floats of padding per staged O row

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Eight halves from a row that is only guaranteed 2-byte alignment, as ONE load and without a
// branch (global loads take any alignment here; a branch on the alignment would make the
// compiler wait for every outstanding load where the two paths join).
typedef h8 h8_unaligned __attribute__((aligned(2)));
// (A pointer rebuilt from scalar registers has lost its address space; the query pointer is device memory, and
// saying so keeps its loads global ones, counted apart from LDS traffic.)
typedef const __attribute__((address_space(1))) _Float16 *global_halves;
__device__ __forceinline__ h8 load_h8(global_halves p) {
    return *reinterpret_cast<const __attribute__((address_space(1))) h8_unaligned *>(p);
}

// Tile decoding shared by both kernels.
struct TileInfo {
    int kvh, hsub, tok_tile, t0, tile_rows, tile_end, start, total;
    int k0;  // first key of split 0: 0, or the block that holds the first key the tile's first row sees through its window
};

__device__ __forceinline__ TileInfo tile_info(const SplitKHot &a, const SplitKSeq &sq, int tile) {
    TileInfo t;
    if (a.tok_tiles == 1 && a.hsubs == 1) {  // a decode step, a verify pass of a few rows: a tile is a KV head
        t.tok_tile = 0;
        t.hsub = 0;
        t.kvh = tile;
    } else {
        t.tok_tile = tile % a.tok_tiles;
        t.hsub = (tile / a.tok_tiles) % a.hsubs;
        t.kvh = tile / (a.tok_tiles * a.hsubs);
    }
    t.start = sq.start;
    t.total = sq.total;
    t.t0 = t.tok_tile * a.tt;
    t.tile_rows = min(a.tt, a.rows - t.t0);
    t.tile_end = max(0, min(t.total, t.start + t.t0 + t.tile_rows));  // keys visible to the tile's last row
    const int first_lim = min(t.total, t.start + t.t0 + 1);
    t.k0 = (a.window > 0 && first_lim > a.window) ? ((first_lim - a.window) & ~31) : 0;
    return t;
}

// The gate's four values of one output item, asked for ahead of the arithmetic they end up multiplying (a combine pass
// that fetches them only when its sums are done waits for memory once more with nothing else to do), and kept as they come:
// converted in the branch that loads them, they were waited for there, in front of the partial results' loads.  One load
// whatever the row's alignment (see load_h8: of two branches, one for each, the compiler waits for a load in the first).
typedef h4 h4_unaligned __attribute__((aligned(2)));
template <typename Args>
__device__ __forceinline__ h4 load_gate4(const Args &a, int seq, int tok, int head, int d, int D) {
    h4 g = (h4)(_Float16)0.0f;
    if (a.gate) g = *(const __attribute__((address_space(1))) h4_unaligned *)(global_halves)(a.gate + seq * a.g_seq_stride + tok * a.g_tok_stride + (long long)head * D + d);
    return g;
}
// Final value of one output element with the gate's values in hand: normalise, gate in fp32, round once.
template <typename Args>
__device__ __forceinline__ void store_out4_gated(const Args &a, int seq, int tok, int head, int d, int D, f4 o, float inv_l,
                                                 bool aligned, h4 g) {
    f4 r = o * inv_l;
    if (a.gate) {
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] *= sigmoid((float)g[i]);
    }
    typedef __attribute__((address_space(1))) _Float16 *global_out;
    const global_out op = (global_out)(a.out + seq * a.o_seq_stride + tok * a.o_tok_stride + (long long)head * D + d);
    if (aligned) {
        *(__attribute__((address_space(1))) h4 *)op = h4{(_Float16)r[0], (_Float16)r[1], (_Float16)r[2], (_Float16)r[3]};
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) op[i] = (_Float16)r[i];
    }
}

// ---------------------------------------------------------------------------
// Register tiles of one 32-key block and the per-row online-softmax state.
// NT = 32 uses v_mfma_f32_32x32x16_f16 (32 query rows per wave), NT = 16 uses
// v_mfma_f32_16x16x32_f16 (16 query rows, half the accumulator registers).
// ---------------------------------------------------------------------------
template <int D, int NT>
struct KTile;
template <int D, int NT>
struct VTile;
template <int D>
struct KTile<D, 32> {
    h8 f[D / 16];
};
template <int D>
struct VTile<D, 32> {
    h8 f[D / 32][2];
};
template <int D>
struct KTile<D, 16> {
    h8 a[D / 32], b[D / 32];  // S^T tile a: keys {0-7, 16-23}; tile b: keys {8-15, 24-31}
};
template <int D>
struct VTile<D, 16> {
    h8 f[D / 16];
};

// The dims of a 32-row tile's V operands over fp16 pages of heads of 256, where they are paired.  A 128-byte line there holds eight dims of
// a chunk; two operand tiles in a row then share the lines of the same 64 dims, the first one's rows the lower four dims of
// each line, the second one's the upper four, so that the first of their loads asks for all of those lines and the second
// finds them on their way.  Row 4 q + i of operand tile mt is dim v_tile_dim(mt) + v_row_dim(4 q + i).
__device__ __forceinline__ constexpr int v_tile_dim(int mt, bool paired) { return paired ? 64 * (mt >> 1) + 4 * (mt & 1) : 32 * mt; }
__device__ __forceinline__ constexpr int v_row_dim(int row, bool paired) { return paired ? 8 * (row >> 2) + (row & 3) : row; }

template <int D, int NT>
struct Lane {
    static constexpr int LN = NT;
    int li, g;       // position inside the lane group, lane group
    int koff, voff;  // this lane's element offset inside a K / V block
    __device__ __forceinline__ explicit Lane(int lane, bool paired = false) {
        li = lane & (LN - 1);
        g = lane / LN;
        if constexpr (NT == 32) {
            koff = (g * 32 + li) * 8;
            voff = v_piece(D, v_row_dim(li, paired), g);
        } else {
            const int ka = li < 8 ? li : li + 8;
            koff = (g * 32 + ka) * 8;
            voff = v_piece(D, li, g);
        }
    }
};

// K/V pages are read through buffer resources: the lane's byte offset inside a
// block is one VGPR for the whole kernel, the block/step offset rides in an SGPR
// and the immediate, so the loads need no per-load address registers, and reads
// past the page would return zeros instead of faulting.
typedef int i4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *base, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, bytes, 0x00020000);
}

// AUX is the load's cache policy: 0, or kStreamed for pages that a launch reads exactly once (a decode step, a
// verify pass of a few rows).  Those loads are marked non-temporal: the data is not kept in L2 or in the
// memory-side cache ahead of lines that will be used again (the split partials, the next layer's weights), and
// a pass over 64 MiB of pages runs 7 % faster for it (13.5 -> 12.5 us), the step behind it 10 %.
// With kPaired its V operands are paired (v_tile_dim).
constexpr int kStreamed = 2;  // the nt bit of a gfx950 buffer load
constexpr int kPaired = 256;
template <int AUX>
__device__ __forceinline__ h8 buf_load_h8(__amdgpu_buffer_rsrc_t rsrc, unsigned lane_bytes, unsigned wave_bytes) {
    i4 r = __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane_bytes, wave_bytes, AUX & ~kPaired);
    return __builtin_bit_cast(h8, r);
}

// `block_bytes` is the block's byte offset inside the page (wave-uniform, always that of a block
// the page holds).  `void_bytes` is added to every lane's offset: 0 for a real load; kVoidLoad
// makes every lane's offset exceed the resource's size, so the load returns zeros without going
// to memory -- the lane offset is what the hardware's range check is defined on.
constexpr unsigned kVoidLoad = 0x7ff00000u;

// What is added to a lane's offsets for the loads of one block: by the keys the lane's load holds, where a selection
// names them.  A touched block of a sparse selection often holds one kept group of four keys: the lanes of K then
// fetch those keys' 16-byte pieces instead of all 32, and a step of V whose sixteen keys are all dropped is not
// fetched; a dropped key's elements read as zeros, under a score that the selection masks and a probability of 0.
// (128 rows with a selection each behind 131k keys 189 -> 162 us, a decode step's row there 18.1 -> 16.4; loads of V lines
// that hold one kept group remain.  Where a chunk's lists fetch whole blocks: lists_fetch_by_key.)
template <int D, int NT>
struct Voids {
    unsigned all;   // the block as a whole (parameters of quantised pages)
    unsigned k[2];  // 32 rows: [0]; 16 rows: tile a, tile b
    unsigned v[2];  // 32 rows: key step t; 16 rows: [0]
    __device__ __forceinline__ explicit Voids(unsigned void_bytes) : all(void_bytes), k{void_bytes, void_bytes}, v{void_bytes, void_bytes} {}
    // `keys`: bit i set = key i of the block is kept by some row of the tile.
    __device__ __forceinline__ Voids(unsigned void_bytes, unsigned keys, const Lane<D, NT> &ln) : all(void_bytes) {
        auto unless = [&](unsigned mask) { return (keys & mask) ? void_bytes : kVoidLoad; };
        if constexpr (NT == 32) {
            k[0] = k[1] = unless(1u << ln.li);
            v[0] = unless(0x0f0fu << (4 * ln.g));
            v[1] = unless(0x0f0f0000u << (4 * ln.g));
        } else {
            const int ka = ln.li < 8 ? ln.li : ln.li + 8;
            k[0] = unless(1u << ka);
            k[1] = unless(256u << ka);
            v[0] = v[1] = unless(0x0f0fu << (16 * (ln.g >> 1) + 4 * (ln.g & 1)));
        }
    }
};

template <int AUX, int D, int NT>
__device__ __forceinline__ void load_k(KTile<D, NT> &t, __amdgpu_buffer_rsrc_t rk, unsigned block_bytes,
                                       const Lane<D, NT> &ln, const Voids<D, NT> &vo) {
    const unsigned lane_bytes = (unsigned)ln.koff * 2u;
    if constexpr (NT == 32) {
#pragma unroll
        for (int s = 0; s < D / 16; ++s) t.f[s] = buf_load_h8<AUX>(rk, lane_bytes + vo.k[0], block_bytes + s * (2 * 32 * 16));
    } else {
#pragma unroll
        for (int s = 0; s < D / 32; ++s) {
            t.a[s] = buf_load_h8<AUX>(rk, lane_bytes + vo.k[0], block_bytes + s * (4 * 32 * 16));
            t.b[s] = buf_load_h8<AUX>(rk, lane_bytes + vo.k[1], block_bytes + s * (4 * 32 * 16) + 128);
        }
    }
}

template <int AUX, int D, int NT>
__device__ __forceinline__ void load_v(VTile<D, NT> &t, __amdgpu_buffer_rsrc_t rv, unsigned block_bytes,
                                       const Lane<D, NT> &ln, const Voids<D, NT> &vo) {
    const unsigned lane_bytes = (unsigned)ln.voff * 2u;
    if constexpr (NT == 32) {
#pragma unroll
        for (int mt = 0; mt < D / 32; ++mt)
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
                t.f[mt][tt] = buf_load_h8<AUX>(rv, lane_bytes + vo.v[tt], block_bytes + 2 * v_piece(D, v_tile_dim(mt, AUX & kPaired), 2 * tt));
    } else {
#pragma unroll
        for (int mt = 0; mt < D / 16; ++mt) t.f[mt] = buf_load_h8<AUX>(rv, lane_bytes + vo.v[0], block_bytes + 2 * v_piece(D, 16 * mt, 0));
    }
}

template <int D, int NT>
struct RowState {
    static constexpr int MT = (NT == 32) ? D / 32 : D / 16;
    typedef typename std::conditional<NT == 32, f16v, f4>::type acc_t;
    float m, l;
    acc_t o[MT];
    __device__ __forceinline__ void init() {
        m = kNegBig;
        l = 0.0f;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) o[mt] = (acc_t)0.0f;
    }
};

// One 32-key block, phase 1: S^T = K Q^T (log2 domain, scaled).  For NT = 16 the
// query fragments come from LDS (`qlds`, one h8 per lane per step) so that the
// wave stays within 256 registers; for NT = 32 they live in registers (`qf`).
template <int D, int NT>
struct Scores;
template <int D>
struct Scores<D, 32> {
    f16v s;
};
template <int D>
struct Scores<D, 16> {
    f4 sa, sb;
};

template <int D, int NT>
__device__ __forceinline__ void block_scores(Scores<D, NT> &sc, const KTile<D, NT> &kt, const h8 *qf, const h8 *qlds,
                                             int lane) {
    if constexpr (NT == 32) {
        (void)qlds;
        (void)lane;
        sc.s = (f16v)0.0f;
#pragma unroll
        for (int t = 0; t < D / 16; ++t) sc.s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kt.f[t], qf[t], sc.s, 0, 0, 0);
    } else {
        (void)qf;
        sc.sa = (f4)0.0f;
        sc.sb = (f4)0.0f;
#pragma unroll
        for (int t = 0; t < D / 32; ++t) {
            const h8 q = qlds[t * 64 + lane];
            sc.sa = __builtin_amdgcn_mfma_f32_16x16x32_f16(kt.a[t], q, sc.sa, 0, 0, 0);
            sc.sb = __builtin_amdgcn_mfma_f32_16x16x32_f16(kt.b[t], q, sc.sb, 0, 0, 0);
        }
    }
}

// Rescaling the 32-row variant's accumulators.  They live in AGPRs, which only the matrix instructions, loads and the
// accvgpr moves can name.  Written as `o *= alpha` the compiler copies all of them to VGPRs at the top of EVERY block
// -- 128 to 144 instructions -- whether the block's rows move their reference or not, and only the multiplies and the
// copies back sit behind the branch.  Here four accumulator registers at a time are operands of an assembly block
// that wants them in AGPRs and multiplies them where they are, so a block that moves no row touches no accumulator.
// Wait states the hardware leaves to software: a vector instruction must not read or overwrite a matrix instruction's
// result for up to 18 cycles after that issued (`rescale_settle` waits 19 ahead of the first block: in the loop sixteen
// score MFMAs and the softmax separate them from the last P.V MFMA anyway), and a matrix instruction must not read a
// register within 2 cycles of a vector instruction writing it (every block ends on a wait of 5).
__device__ __forceinline__ void rescale_settle() { asm volatile("s_nop 15\n\ts_nop 2"); }
__device__ __forceinline__ void rescale4(float &a0, float &a1, float &a2, float &a3, float alpha) {
    float t0, t1, t2, t3;
    asm volatile(
        "v_accvgpr_read_b32 %4, %0\n\tv_accvgpr_read_b32 %5, %1\n\tv_accvgpr_read_b32 %6, %2\n\tv_accvgpr_read_b32 %7, %3\n\t"
        "v_mul_f32 %4, %8, %4\n\tv_mul_f32 %5, %8, %5\n\tv_mul_f32 %6, %8, %6\n\tv_mul_f32 %7, %8, %7\n\t"
        "v_accvgpr_write_b32 %0, %4\n\tv_accvgpr_write_b32 %1, %5\n\tv_accvgpr_write_b32 %2, %6\n\tv_accvgpr_write_b32 %3, %7\n\t"
        "s_nop 4"
        : "+a"(a0), "+a"(a1), "+a"(a2), "+a"(a3), "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3)
        : "v"(alpha));
}
__device__ __forceinline__ void rescale_tile(f16v &o, float alpha) {
#pragma unroll
    for (int j = 0; j < 16; j += 4) {
        float a0 = o[j], a1 = o[j + 1], a2 = o[j + 2], a3 = o[j + 3];
        rescale4(a0, a1, a2, a3, alpha);
        o[j] = a0;
        o[j + 1] = a1;
        o[j + 2] = a2;
        o[j + 3] = a3;
    }
}

// Phase 2a: mask and online softmax of one block.  This lane's row sees keys [lo, lim); kbase is
// the block's first key.  Leaves the block's probabilities in `pf` as fp16 B
// operands of the P.V MFMAs and rescales the row's accumulators (`extra` is a further one that
// follows the same running max, or null).
template <int D, int NT>
struct Probs;
template <int D>
struct Probs<D, 32> {
    h8 pf[2];
};
template <int D>
struct Probs<D, 16> {
    h8 pf;
};

template <int D, int NT>
__device__ __forceinline__ void block_softmax(RowState<D, NT> &st, Scores<D, NT> &sc, Probs<D, NT> &pr,
                                              const Lane<D, NT> &ln, int kbase, int lo, int lim, float scale_log2e,
                                              typename RowState<D, NT>::acc_t *extra = nullptr, unsigned kept = ~0u,
                                              const unsigned *row_keep = nullptr, unsigned row_bits = ~0u) {
    // kept: bit i set = key kbase + i takes part (a sparse selection shared by the tile's rows; all ones without one).
    // row_keep: this lane's own row's 32 selection bytes of the block, as 8 words (a per-query selection).
    // row_bits: the same as one bit per key (a per-query selection that came as index lists); all ones without one.
    const bool any_row_bits = __any(row_bits != ~0u);
    const bool need_mask = __any(kbase + 32 > lim || kbase < lo) || kept != ~0u || row_keep != nullptr || any_row_bits;
    unsigned rk[4] = {~0u, ~0u, ~0u, ~0u};  // the words that hold this lane's keys, picked by the lane's place in the tile
    if (row_keep) {
        if constexpr (NT == 32) {  // key offsets 8 a + 4 g + (v & 3): word 2 a + g
#pragma unroll
            for (int i = 0; i < 4; ++i) rk[i] = ln.g ? row_keep[2 * i + 1] : row_keep[2 * i];
        } else {  // tile a: offsets 4 (g & 1) + 16 (g >> 1) + v, tile b: 8 more
            const unsigned lo_a = (ln.g & 1) ? row_keep[1] : row_keep[0], hi_a = (ln.g & 1) ? row_keep[5] : row_keep[4];
            const unsigned lo_b = (ln.g & 1) ? row_keep[3] : row_keep[2], hi_b = (ln.g & 1) ? row_keep[7] : row_keep[6];
            rk[0] = (ln.g >> 1) ? hi_a : lo_a;
            rk[1] = (ln.g >> 1) ? hi_b : lo_b;
        }
    }
    if constexpr (NT == 32) {
        f16v &s = sc.s;
        // The three reasons to drop a key, each behind its own wave-uniform test and over all 16 values at once: a
        // selected block far behind the chunk's rows needs no range test, a dense block at the diagonal no selection.
        const bool need_range = __any(kbase + 32 > lim || kbase < lo);
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] *= scale_log2e;
        if (need_range) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int key = kbase + 8 * (v >> 2) + 4 * ln.g + (v & 3);
                if (key >= lim || key < lo) s[v] = -INFINITY;
            }
        }
        if (kept != ~0u) {
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (!((kept >> (8 * (v >> 2) + 4 * ln.g + (v & 3))) & 1u)) s[v] = -INFINITY;
        }
        if (row_keep) {
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (!((rk[v >> 2] >> (8 * (v & 3))) & 0xffu)) s[v] = -INFINITY;
        }
        if (any_row_bits) {
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (!((row_bits >> (8 * (v >> 2) + 4 * ln.g + (v & 3))) & 1u)) s[v] = -INFINITY;
        }
        float mx = kNegBig;
#pragma unroll
        for (int v = 0; v < 16; ++v) mx = fmaxf(mx, s[v]);
        mx = max_across_halves(mx);
        const float m_new = mx > st.m + (extra ? kLazyRescale : kLazyRescaleHalfPages) ? mx : st.m;
        const float alpha = fast_exp2(st.m - m_new);
        float psum = 0.0f;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const float p = fast_exp2(s[v] - m_new);
            psum += p;
            pr.pf[v >> 3][v & 7] = (_Float16)p;
        }
        st.l = st.l * alpha + psum;
        st.m = m_new;
        if (!__all(alpha == 1.0f)) {
            rescale_settle();
#pragma unroll
            for (int mt = 0; mt < D / 32; ++mt) rescale_tile(st.o[mt], alpha);
            if (extra) rescale_tile(*extra, alpha);
        }
    } else {
        f4 &sa = sc.sa, &sb = sc.sb;
        const int key0 = kbase + (ln.g & 1) * 4 + (ln.g >> 1) * 16;  // first key of this lane's tile-a results
        float mx = kNegBig;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            float xa = sa[v] * scale_log2e, xb = sb[v] * scale_log2e;
            if (need_mask) {
                if (key0 + v >= lim || key0 + v < lo || !((kept & row_bits) >> (key0 + v - kbase) & 1u) || !((rk[0] >> (8 * v)) & 0xffu))
                    xa = -INFINITY;
                if (key0 + 8 + v >= lim || key0 + 8 + v < lo || !((kept & row_bits) >> (key0 + 8 + v - kbase) & 1u) ||
                    !((rk[1] >> (8 * v)) & 0xffu))
                    xb = -INFINITY;
            }
            sa[v] = xa;
            sb[v] = xb;
            mx = fmaxf(mx, fmaxf(xa, xb));
        }
        mx = max_across_quarters(mx);
        const float m_new = mx > st.m + (extra ? kLazyRescale : kLazyRescaleHalfPages) ? mx : st.m;
        const float alpha = fast_exp2(st.m - m_new);
        float psum = 0.0f;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float pa = fast_exp2(sa[v] - m_new), pb = fast_exp2(sb[v] - m_new);
            psum += pa + pb;
            pr.pf[v] = (_Float16)pa;
            pr.pf[4 + v] = (_Float16)pb;
        }
        st.l = st.l * alpha + psum;
        st.m = m_new;
        if (!__all(alpha == 1.0f)) {
#pragma unroll
            for (int mt = 0; mt < D / 16; ++mt) st.o[mt] *= alpha;
            if (extra) *extra *= alpha;
        }
    }
}

// Phase 2b: O^T += V^T P^T.
template <int D, int NT>
__device__ __forceinline__ void block_softmax_pv(RowState<D, NT> &st, Scores<D, NT> &sc, const VTile<D, NT> &vt,
                                                 const Lane<D, NT> &ln, int kbase, int lo, int lim, float scale_log2e,
                                                 unsigned kept = ~0u, const unsigned *row_keep = nullptr, unsigned row_bits = ~0u) {
    Probs<D, NT> pr;
    block_softmax<D, NT>(st, sc, pr, ln, kbase, lo, lim, scale_log2e, nullptr, kept, row_keep, row_bits);
    if constexpr (NT == 32) {
#pragma unroll
        for (int mt = 0; mt < D / 32; ++mt)
#pragma unroll
            for (int t = 0; t < 2; ++t)
                st.o[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vt.f[mt][t], pr.pf[t], st.o[mt], 0, 0, 0);
    } else {
#pragma unroll
        for (int mt = 0; mt < D / 16; ++mt) st.o[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vt.f[mt], pr.pf, st.o[mt], 0, 0, 0);
    }
}

// The two phases of a 32-row fp16 tile with the NEXT block's loads between their MFMAs: a fragment's load follows the
// MFMA that read it, into the same registers, one scheduling region per pair.  Where the block's loads stand apart
// from the MFMAs in the source, the compiler is free to move them ahead of the MFMAs -- into 64 other registers,
// which the per-query selection's variant does not have: it then parks the tile in AGPRs at the end of the block,
// behind a wait for every load, and nothing of the next block is in flight under the arithmetic of this one.
template <int AUX, int D>
__device__ __forceinline__ void block_scores_refill(Scores<D, 32> &sc, KTile<D, 32> &kt, const h8 *qf, __amdgpu_buffer_rsrc_t rk,
                                                    unsigned next_bytes, const Lane<D, 32> &ln, const Voids<D, 32> &vo) {
    const unsigned lane_bytes = (unsigned)ln.koff * 2u + vo.k[0];
    sc.s = (f16v)0.0f;
#pragma unroll
    for (int t = 0; t < D / 16; ++t) {
        sc.s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kt.f[t], qf[t], sc.s, 0, 0, 0);
        asm volatile("" : "+a"(sc.s));  // (an MFMA is no memory operation: only its result's use here keeps it ahead of the load)
        kt.f[t] = buf_load_h8<AUX>(rk, lane_bytes, next_bytes + t * (2 * 32 * 16));
        __builtin_amdgcn_sched_barrier(0);
    }
}
template <int AUX, int D>
__device__ __forceinline__ void block_softmax_pv_refill(RowState<D, 32> &st, Scores<D, 32> &sc, VTile<D, 32> &vt,
                                                        const Lane<D, 32> &ln, int kbase, int lo, int lim, float scale_log2e,
                                                        __amdgpu_buffer_rsrc_t rv, unsigned next_bytes, const Voids<D, 32> &vo,
                                                        unsigned kept, const unsigned *row_keep, unsigned row_bits) {
    Probs<D, 32> pr;
    block_softmax<D, 32>(st, sc, pr, ln, kbase, lo, lim, scale_log2e, nullptr, kept, row_keep, row_bits);
    const unsigned lane_bytes[2] = {(unsigned)ln.voff * 2u + vo.v[0], (unsigned)ln.voff * 2u + vo.v[1]};
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mt = 0; mt < D / 32; ++mt) {
#pragma unroll
        for (int t = 0; t < 2; ++t) st.o[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vt.f[mt][t], pr.pf[t], st.o[mt], 0, 0, 0);
        asm volatile("" : "+a"(st.o[mt]));
#pragma unroll
        for (int t = 0; t < 2; ++t) vt.f[mt][t] = buf_load_h8<AUX>(rv, lane_bytes[t], next_bytes + 2 * v_piece(D, v_tile_dim(mt, AUX & kPaired), 2 * t));
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Eight listed groups of four keys taken as one block (KEEP = 4): every lane has offsets of its own.  K: a lane's key is one
// of its group's four, 64 contiguous bytes per 8 dims.  V: the eight keys of a lane's operand are two groups, half a
// chunk (8 bytes) of each, over heads of 256 in 256 contiguous bytes per 16 dims.  (While those lay in all of the block's lines their
// passage through the vector cache was the kernel: 128 rows of 16/2 heads with a selection each behind 131k keys, 64 requests
// a load instead of 16, 114 -> 74.8 us.)  A group that is not there has kVoidLoad for an offset.
struct GroupOffsets {
    unsigned k;
    unsigned v[2][2];  // [key step][half of the operand]
};
template <int D>
__device__ __forceinline__ GroupOffsets group_offsets(const int (&ids)[5], const Lane<D, 32> &ln) {
    constexpr unsigned BLOCK = 32 * D * 2;
    GroupOffsets o;
    auto block_at = [&](int id) { return (unsigned)(id >> 3) * BLOCK; };
    o.k = ids[0] < 0 ? kVoidLoad : block_at(ids[0]) + (unsigned)(ln.g * 32 + 4 * (ids[0] & 7) + (ln.li & 3)) * 16u;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int id = ids[1 + 2 * t + h], j = id & 7;  // keys 4 j .. 4 j + 3 of the block: half (j / 2) % 2 of chunk 2 (j / 4) + j % 2
            o.v[t][h] = id < 0 ? kVoidLoad : block_at(id) + 2u * (unsigned)(v_piece(D, ln.li, 2 * (j >> 2) + (j & 1)) + ((j >> 1) & 1) * 4);
        }
    return o;
}
typedef unsigned group_words __attribute__((ext_vector_type(2)));
__device__ __forceinline__ h8 load_group_pair(__amdgpu_buffer_rsrc_t rv, const unsigned (&at)[2], unsigned wave_bytes) {
    const group_words lo = __builtin_bit_cast(group_words, __builtin_amdgcn_raw_buffer_load_b64(rv, at[0], wave_bytes, 0));
    const group_words hi = __builtin_bit_cast(group_words, __builtin_amdgcn_raw_buffer_load_b64(rv, at[1], wave_bytes, 0));
    const i4 both = {(int)lo[0], (int)lo[1], (int)hi[0], (int)hi[1]};
    return __builtin_bit_cast(h8, both);
}
template <int D>
__device__ __forceinline__ void load_k_groups(KTile<D, 32> &kt, __amdgpu_buffer_rsrc_t rk, const GroupOffsets &o) {
#pragma unroll
    for (int t = 0; t < D / 16; ++t) kt.f[t] = buf_load_h8<0>(rk, o.k, t * (2 * 32 * 16));
}
template <int D>
__device__ __forceinline__ void load_v_groups(VTile<D, 32> &vt, __amdgpu_buffer_rsrc_t rv, const GroupOffsets &o) {
#pragma unroll
    for (int mt = 0; mt < D / 32; ++mt)
#pragma unroll
        for (int t = 0; t < 2; ++t) vt.f[mt][t] = load_group_pair(rv, o.v[t], 2 * v_piece(D, 32 * mt, 0));
}
// The two phases with the next groups' loads between their MFMAs, as in block_scores_refill / block_softmax_pv_refill.
template <int D>
__device__ __forceinline__ void group_scores_refill(Scores<D, 32> &sc, KTile<D, 32> &kt, const h8 *qf, __amdgpu_buffer_rsrc_t rk, const GroupOffsets &next) {
    sc.s = (f16v)0.0f;
#pragma unroll
    for (int t = 0; t < D / 16; ++t) {
        sc.s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kt.f[t], qf[t], sc.s, 0, 0, 0);
        asm volatile("" : "+a"(sc.s));
        kt.f[t] = buf_load_h8<0>(rk, next.k, t * (2 * 32 * 16));
        __builtin_amdgcn_sched_barrier(0);
    }
}
template <int D>
__device__ __forceinline__ void group_softmax_pv_refill(RowState<D, 32> &st, Scores<D, 32> &sc, VTile<D, 32> &vt, const Lane<D, 32> &ln,
                                                        float scale_log2e, __amdgpu_buffer_rsrc_t rv, const GroupOffsets &next, unsigned row_bits) {
    Probs<D, 32> pr;
    // (the bits say all: a listed key that the row cannot see is not among them)
    block_softmax<D, 32>(st, sc, pr, ln, 0, 0, 32, scale_log2e, nullptr, ~0u, nullptr, row_bits);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mt = 0; mt < D / 32; ++mt) {
#pragma unroll
        for (int t = 0; t < 2; ++t) st.o[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vt.f[mt][t], pr.pf[t], st.o[mt], 0, 0, 0);
        asm volatile("" : "+a"(st.o[mt]));
#pragma unroll
        for (int t = 0; t < 2; ++t) vt.f[mt][t] = load_group_pair(rv, next.v[t], 2 * v_piece(D, 32 * mt, 0));
        __builtin_amdgcn_sched_barrier(0);
    }
}

// ---------------------------------------------------------------------------
// Quantised pages (8 or 4 bits per value; layout in kv_layout.h).  A block's tiles hold the
// levels as loaded plus this lane's scales and biases; levels become fp16 MFMA operands in
// registers, right before the instruction that uses them:
//   K  operand = level * scale + bias per (key, group of 64 dims), one packed fp16 FMA per two
//      elements -- the loader of sources/TinyTitanCore/Metal/Attention/attention.metal:89-117
//      with one fp16 rounding of the product-sum instead of none.
//   V  O^T[d][row] = sum_key (level * scale + bias) P = sum_key level * (scale * P)
//                                                     + sum_key bias * P:
//      the scale goes into P (one B operand per group), the levels are the A operand as they
//      are, and the bias term is ONE more MFMA per key step whose A rows are the groups' biases;
//      its accumulator (row = group) is added to the group's dims once, at the end.  scale * P
//      carries a factor 4 (the level accumulators are divided by 4 at the end), which keeps
//      small probabilities times small scales out of fp16's subnormal range; fp16 values bound
//      scale to 514 and P stays below 16, so 4 * scale * P stays below 32896.
// Levels are widened with v_perm_b32: byte b under exponent byte 0x64 is the fp16 number
// 1024 + b, and subtracting 1024 is exact.
// ---------------------------------------------------------------------------
typedef unsigned u2v __attribute__((ext_vector_type(2)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
constexpr float kProbBoost = 4.0f;

template <int AUX, int N>
__device__ __forceinline__ void buf_load_words(unsigned (&dst)[N], __amdgpu_buffer_rsrc_t rsrc, unsigned lane_bytes,
                                               unsigned wave_bytes) {
    static_assert(N == 1 || N == 2 || N == 4, "one load instruction");
    if constexpr (N == 1) {
        dst[0] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, lane_bytes, wave_bytes, AUX);
    } else if constexpr (N == 2) {
        const u2v r = __builtin_amdgcn_raw_buffer_load_b64(rsrc, lane_bytes, wave_bytes, AUX);
        dst[0] = r[0];
        dst[1] = r[1];
    } else {
        const u4v r = __builtin_bit_cast(u4v, __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane_bytes, wave_bytes, AUX));
        dst[0] = r[0];
        dst[1] = r[1];
        dst[2] = r[2];
        dst[3] = r[3];
    }
}

// Eight bytes -> eight halves holding 0..255 exactly.
__device__ __forceinline__ h8 widen_bytes(unsigned w0, unsigned w1) {
    const unsigned e = 0x64646464u;
    const u4v x = {__builtin_amdgcn_perm(e, w0, 0x04010400u), __builtin_amdgcn_perm(e, w0, 0x04030402u),
                   __builtin_amdgcn_perm(e, w1, 0x04010400u), __builtin_amdgcn_perm(e, w1, 0x04030402u)};
    return __builtin_bit_cast(h8, x) - (h8)(_Float16)1024;
}
// Eight nibbles of one dword, element 2 i in the low nibble of byte i, in element order.
__device__ __forceinline__ h8 widen_nibbles(unsigned w) {
    const unsigned lo = w & 0x0f0f0f0fu, hi = (w >> 4) & 0x0f0f0f0fu, e = 0x64006400u;
    const u4v x = {__builtin_amdgcn_perm(hi, lo, 0x0c040c00u) | e, __builtin_amdgcn_perm(hi, lo, 0x0c050c01u) | e,
                   __builtin_amdgcn_perm(hi, lo, 0x0c060c02u) | e, __builtin_amdgcn_perm(hi, lo, 0x0c070c03u) | e};
    return __builtin_bit_cast(h8, x) - (h8)(_Float16)1024;
}

template <int BITS>
__device__ __forceinline__ h8 k_operand(const unsigned (&w)[BITS / 4], unsigned scale_bias) {
    const h2 sb = __builtin_bit_cast(h2, scale_bias);
    h8 levels;
    if constexpr (BITS == 8) levels = widen_bytes(w[0], w[1]);
    else levels = widen_nibbles(w[0]);
    return levels * (h8)sb[0] + (h8)sb[1];
}

template <int D, int NT, int BITS>
struct KTileQ;
template <int D, int NT, int BITS>
struct VTileQ;
// K levels: one load per lane holds the 16 dims of a key's unit -- 16 bytes at 8 bits, 8 at 4 --
// and feeds two contraction steps (dims 0-7, then 8-15).  The lane's unit of step pair p is
// 2 p + g (32-row tiles: dims 32 p + 16 g ..) or 4 p + g (16-row tiles: dims 64 p + 16 g ..); the
// query fragments in LDS are laid out in the same order (q_dim_of_step).
template <int D, int BITS>
struct KTileQ<D, 32, BITS> {
    unsigned f[D / 32][BITS / 2];
    unsigned sb[D / 64];  // {scale, bias} of this lane's key, per group
};
template <int D, int BITS>
struct KTileQ<D, 16, BITS> {
    unsigned a[D / 64][BITS / 2], b[D / 64][BITS / 2];
    unsigned sba[D / 64], sbb[D / 64];
};
// V levels: one load per lane holds its chunk's eight keys for the dims d and d + 32 -- two runs
// of 8 bytes at 8 bits, the low and high nibbles of one run at 4 bits.
template <int D, int BITS>
struct VTileQ<D, 32, BITS> {
    unsigned f[D / 64][2][BITS / 2];  // [pair of dim tiles 2 j, 2 j + 1][key step][dword]
    unsigned sc[D / 64][2][4];        // 8 scales per group and key step
    unsigned bias[2][4];              // rows = groups: this lane's group's 8 biases per key step, or zeros
};
template <int D, int BITS>
struct VTileQ<D, 16, BITS> {
    unsigned f[D / 32][BITS / 2];  // load i = 2 j + rr: dim tiles 4 j + rr and 4 j + 2 + rr
    unsigned sc[D / 64][4];
    unsigned bias[4];
};

// First dim of the 8 that lane group g contracts in step t of a quantised tile.
template <int NT>
__device__ __forceinline__ int q_dim_of_step(int t, int g) {
    return (NT == 32 ? 32 : 64) * (t >> 1) + 16 * g + 8 * (t & 1);
}

// The operand of contraction step `half` (0 / 1) of a loaded K unit.
template <int BITS>
__device__ __forceinline__ h8 k_unit_operand(const unsigned (&w)[BITS / 2], int half, unsigned scale_bias) {
    if constexpr (BITS == 8) {
        const unsigned pair[2] = {w[2 * half], w[2 * half + 1]};
        return k_operand<8>(pair, scale_bias);
    } else {
        const unsigned one[1] = {w[half]};
        return k_operand<4>(one, scale_bias);
    }
}
// The two V operands of a loaded run: dims d (lo) and d + 32 (hi).
template <int BITS>
__device__ __forceinline__ void v_run_operands(const unsigned (&w)[BITS / 2], h8 &lo, h8 &hi) {
    if constexpr (BITS == 8) {
        lo = widen_bytes(w[0], w[1]);
        hi = widen_bytes(w[2], w[3]);
    } else {
        lo = widen_bytes(w[0] & 0x0f0f0f0fu, w[1] & 0x0f0f0f0fu);
        hi = widen_bytes((w[0] >> 4) & 0x0f0f0f0fu, (w[1] >> 4) & 0x0f0f0f0fu);
    }
}

// Byte offsets of this lane inside a block's K / V levels, and of the tile's loads.
template <int D, int NT, int BITS>
struct QuantOffsets {
    static constexpr unsigned LEVELS = 32u * D * BITS / 8, GPH = D / 64;
    static constexpr unsigned K_UNIT = 16u * BITS / 8;                 // bytes of one key's unit
    static constexpr unsigned K_PAIR = (NT == 32 ? 2u : 4u) * 32u * K_UNIT;  // bytes between step pairs
    static constexpr unsigned V_RUN = 8u * BITS / 4;                   // bytes of one (dim pair, chunk) run
    __device__ __forceinline__ static unsigned k_lane(const Lane<D, NT> &ln) { return (unsigned)ln.koff / 8u * K_UNIT; }
    __device__ __forceinline__ static unsigned v_lane(const Lane<D, NT> &ln) { return (unsigned)(ln.li * 4 + ln.g) * V_RUN; }
};

template <int AUX, int D, int NT, int BITS>
__device__ __forceinline__ void load_k(KTileQ<D, NT, BITS> &t, __amdgpu_buffer_rsrc_t rk, unsigned block_bytes,
                                       const Lane<D, NT> &ln, const Voids<D, NT> &vo) {
    typedef QuantOffsets<D, NT, BITS> O;
    const unsigned lane_bytes = O::k_lane(ln);
    if constexpr (NT == 32) {
#pragma unroll
        for (int p = 0; p < D / 32; ++p) buf_load_words<AUX>(t.f[p], rk, lane_bytes + vo.k[0], block_bytes + p * O::K_PAIR);
        buf_load_words<AUX>(t.sb, rk, (unsigned)ln.li * O::GPH * 4 + vo.k[0], block_bytes + O::LEVELS);
    } else {
#pragma unroll
        for (int p = 0; p < D / 64; ++p) {
            buf_load_words<AUX>(t.a[p], rk, lane_bytes + vo.k[0], block_bytes + p * O::K_PAIR);
            buf_load_words<AUX>(t.b[p], rk, lane_bytes + vo.k[1], block_bytes + p * O::K_PAIR + 8 * O::K_UNIT);
        }
        const unsigned ka = ln.li < 8 ? ln.li : ln.li + 8;
        buf_load_words<AUX>(t.sba, rk, ka * O::GPH * 4 + vo.k[0], block_bytes + O::LEVELS);
        buf_load_words<AUX>(t.sbb, rk, ka * O::GPH * 4 + vo.k[1], block_bytes + O::LEVELS + 8 * O::GPH * 4);
    }
}

template <int AUX, int D, int NT, int BITS>
__device__ __forceinline__ void load_v(VTileQ<D, NT, BITS> &t, __amdgpu_buffer_rsrc_t rv, unsigned block_bytes,
                                       const Lane<D, NT> &ln, const Voids<D, NT> &vo) {
    typedef QuantOffsets<D, NT, BITS> O;
    const unsigned lane_bytes = O::v_lane(ln);  // (row * 4 + chunk) runs
    const unsigned param_lane = (unsigned)ln.g * 16 + vo.all;
    // Bias rows: lane rows 0 .. GPH-1 carry a group's biases, the others read zeros (void load).
    const unsigned bias_lane = (unsigned)ln.li * 64 + (unsigned)ln.g * 16 + ((unsigned)ln.li < O::GPH ? vo.all : kVoidLoad);
    if constexpr (NT == 32) {
#pragma unroll
        for (int j = 0; j < D / 64; ++j)
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) buf_load_words<AUX>(t.f[j][tt], rv, lane_bytes + vo.v[tt], block_bytes + (j * 32 * 4 + tt * 2) * O::V_RUN);
#pragma unroll
        for (int grp = 0; grp < (int)O::GPH; ++grp)
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) buf_load_words<AUX>(t.sc[grp][tt], rv, param_lane, block_bytes + O::LEVELS + grp * 64 + tt * 32);
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) buf_load_words<AUX>(t.bias[tt], rv, bias_lane, block_bytes + O::LEVELS + O::GPH * 64 + tt * 32);
    } else {
#pragma unroll
        for (int i = 0; i < D / 32; ++i) buf_load_words<AUX>(t.f[i], rv, lane_bytes + vo.v[0], block_bytes + i * 16 * 4 * O::V_RUN);
#pragma unroll
        for (int grp = 0; grp < (int)O::GPH; ++grp) buf_load_words<AUX>(t.sc[grp], rv, param_lane, block_bytes + O::LEVELS + grp * 64);
        buf_load_words<AUX>(t.bias, rv, bias_lane, block_bytes + O::LEVELS + O::GPH * 64);
    }
}

// The two phases over quantised tiles also REFILL the tiles for the wave's next block: a
// load's registers are free as soon as its levels have been widened, so the load for the next
// block is issued right there, before the MFMAs that use the widened copies.  Every load thus
// has a whole block of work between issue and use -- a tile that was refilled in one piece
// after the phase had only the other phase (levels are half the bytes of fp16 values, so half
// as much was in flight), and the wave stood waiting for memory twice per block.  `next_bytes` /
// `vo` address the next block as in load_k; the scale/bias words of K are fetched into
// spare registers first and swapped in at the end.
template <int AUX, int D, int NT, int BITS>
__device__ __forceinline__ void block_scores(Scores<D, NT> &sc, KTileQ<D, NT, BITS> &kt, const h8 *qf, const h8 *qlds, int lane,
                                             __amdgpu_buffer_rsrc_t rk, unsigned next_bytes, const Lane<D, NT> &ln,
                                             const Voids<D, NT> &vo) {
    typedef QuantOffsets<D, NT, BITS> O;
    constexpr int GPH = D / 64;
    const unsigned lane_bytes = O::k_lane(ln);
    (void)qf;
    if constexpr (NT == 32) {
        unsigned sb_next[GPH];
        buf_load_words<AUX>(sb_next, rk, (unsigned)ln.li * GPH * 4 + vo.k[0], next_bytes + O::LEVELS);
        sc.s = (f16v)0.0f;
        h8 q = qlds[lane];
#pragma unroll
        for (int p = 0; p < D / 32; ++p) {
            const h8 q1 = qlds[(2 * p + 1) * 64 + lane];
            const h8 q_next = qlds[(p + 1 < D / 32 ? 2 * p + 2 : 2 * p) * 64 + lane];  // read ahead of their use
            // widening the second half fills the time the first MFMA runs (they chain on one accumulator)
            const h8 k0 = k_unit_operand<BITS>(kt.f[p], 0, kt.sb[p / 2]);
            sc.s = __builtin_amdgcn_mfma_f32_32x32x16_f16(k0, q, sc.s, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            const h8 k1 = k_unit_operand<BITS>(kt.f[p], 1, kt.sb[p / 2]);
            buf_load_words<AUX>(kt.f[p], rk, lane_bytes + vo.k[0], next_bytes + p * O::K_PAIR);
            sc.s = __builtin_amdgcn_mfma_f32_32x32x16_f16(k1, q1, sc.s, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            q = q_next;
        }
#pragma unroll
        for (int grp = 0; grp < GPH; ++grp) kt.sb[grp] = sb_next[grp];
    } else {
        unsigned sba_next[GPH], sbb_next[GPH];
        const unsigned ka = ln.li < 8 ? ln.li : ln.li + 8;
        buf_load_words<AUX>(sba_next, rk, ka * GPH * 4 + vo.k[0], next_bytes + O::LEVELS);
        buf_load_words<AUX>(sbb_next, rk, ka * GPH * 4 + vo.k[1], next_bytes + O::LEVELS + 8 * GPH * 4);
        sc.sa = (f4)0.0f;
        sc.sb = (f4)0.0f;
        h8 q = qlds[lane];
#pragma unroll
        for (int p = 0; p < D / 64; ++p) {
            const h8 q1 = qlds[(2 * p + 1) * 64 + lane];
            const h8 q_next = qlds[(p + 1 < D / 64 ? 2 * p + 2 : 2 * p) * 64 + lane];
            const h8 a0 = k_unit_operand<BITS>(kt.a[p], 0, kt.sba[p]);
            sc.sa = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, q, sc.sa, 0, 0, 0);
            const h8 b0 = k_unit_operand<BITS>(kt.b[p], 0, kt.sbb[p]);
            sc.sb = __builtin_amdgcn_mfma_f32_16x16x32_f16(b0, q, sc.sb, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            const h8 a1 = k_unit_operand<BITS>(kt.a[p], 1, kt.sba[p]);
            buf_load_words<AUX>(kt.a[p], rk, lane_bytes + vo.k[0], next_bytes + p * O::K_PAIR);
            sc.sa = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, q1, sc.sa, 0, 0, 0);
            const h8 b1 = k_unit_operand<BITS>(kt.b[p], 1, kt.sbb[p]);
            buf_load_words<AUX>(kt.b[p], rk, lane_bytes + vo.k[1], next_bytes + p * O::K_PAIR + 8 * O::K_UNIT);
            sc.sb = __builtin_amdgcn_mfma_f32_16x16x32_f16(b1, q1, sc.sb, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            q = q_next;
        }
#pragma unroll
        for (int grp = 0; grp < GPH; ++grp) {
            kt.sba[grp] = sba_next[grp];
            kt.sbb[grp] = sbb_next[grp];
        }
    }
}

__device__ __forceinline__ h8 words_as_h8(const unsigned (&w)[4]) {
    const u4v x = {w[0], w[1], w[2], w[3]};
    return __builtin_bit_cast(h8, x);
}

// `bias_acc` accumulates sum_key bias[group][key] * P[key][row] in its row `group`.
template <int AUX, int D, int NT, int BITS>
__device__ __forceinline__ void block_softmax_pv(RowState<D, NT> &st, Scores<D, NT> &sc, VTileQ<D, NT, BITS> &vt,
                                                 const Lane<D, NT> &ln, int kbase, int lo, int lim, float scale_log2e,
                                                 typename RowState<D, NT>::acc_t &bias_acc, __amdgpu_buffer_rsrc_t rv,
                                                 unsigned next_bytes, const Voids<D, NT> &vo, unsigned kept = ~0u,
                                                 const unsigned *row_keep = nullptr, unsigned row_bits = ~0u) {
    typedef QuantOffsets<D, NT, BITS> O;
    constexpr int GPH = D / 64;
    const unsigned lane_bytes = O::v_lane(ln);
    const unsigned param_lane = (unsigned)ln.g * 16 + vo.all;
    const unsigned bias_lane = (unsigned)ln.li * 64 + (unsigned)ln.g * 16 + ((unsigned)ln.li < (unsigned)GPH ? vo.all : kVoidLoad);
    Probs<D, NT> pr;
    block_softmax<D, NT>(st, sc, pr, ln, kbase, lo, lim, scale_log2e, &bias_acc, kept, row_keep, row_bits);
    if constexpr (NT == 32) {
        h8 ps[GPH][2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const h8 boosted = pr.pf[t] * (h8)(_Float16)kProbBoost;
#pragma unroll
            for (int grp = 0; grp < GPH; ++grp) {
                ps[grp][t] = boosted * words_as_h8(vt.sc[grp][t]);
                buf_load_words<AUX>(vt.sc[grp][t], rv, param_lane, next_bytes + O::LEVELS + grp * 64 + t * 32);
            }
            bias_acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(words_as_h8(vt.bias[t]), pr.pf[t], bias_acc, 0, 0, 0);
            buf_load_words<AUX>(vt.bias[t], rv, bias_lane, next_bytes + O::LEVELS + GPH * 64 + t * 32);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int j = 0; j < D / 64; ++j) {  // dim tiles 2 j (dims 64 j + row) and 2 j + 1 (32 above), both of group j
                h8 lo_op, hi_op;
                v_run_operands<BITS>(vt.f[j][t], lo_op, hi_op);
                buf_load_words<AUX>(vt.f[j][t], rv, lane_bytes + vo.v[t], next_bytes + (j * 32 * 4 + t * 2) * O::V_RUN);
                st.o[2 * j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo_op, ps[j][t], st.o[2 * j], 0, 0, 0);
                st.o[2 * j + 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi_op, ps[j][t], st.o[2 * j + 1], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
    } else {
        h8 ps[GPH];
        const h8 boosted = pr.pf * (h8)(_Float16)kProbBoost;
#pragma unroll
        for (int grp = 0; grp < GPH; ++grp) {
            ps[grp] = boosted * words_as_h8(vt.sc[grp]);
            buf_load_words<AUX>(vt.sc[grp], rv, param_lane, next_bytes + O::LEVELS + grp * 64);
        }
        bias_acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(words_as_h8(vt.bias), pr.pf, bias_acc, 0, 0, 0);
        buf_load_words<AUX>(vt.bias, rv, bias_lane, next_bytes + O::LEVELS + GPH * 64);
        __builtin_amdgcn_sched_barrier(0);
        // load i = 2 j + rr covers rows 16 rr + lane row of 64-dim group j: dims 64 j + 16 rr + row
        // (tile 4 j + rr) and 32 above (tile 4 j + 2 + rr)
#pragma unroll
        for (int i = 0; i < D / 32; ++i) {
            const int j = i >> 1, rr = i & 1;
            h8 lo_op, hi_op;
            v_run_operands<BITS>(vt.f[i], lo_op, hi_op);
            buf_load_words<AUX>(vt.f[i], rv, lane_bytes + vo.v[0], next_bytes + i * 16 * 4 * O::V_RUN);
            st.o[4 * j + rr] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo_op, ps[j], st.o[4 * j + rr], 0, 0, 0);
            st.o[4 * j + 2 + rr] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi_op, ps[j], st.o[4 * j + 2 + rr], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// ---------------------------------------------------------------------------
// Pass 1.  grid = (split, tile, sequence); WAVES wavefronts per workgroup, wave
// w takes key blocks w, w + WAVES, ... of the split (split 0 starts at key 0, or
// at the block of the first key the tile's window reaches).  A block's K and V
// tiles live in registers; the next block's K loads are issued as soon as the
// score MFMAs have consumed the current ones and its V loads right after the P.V
// MFMAs, so a wave always has 16-32 KiB in flight (BITS = 16; the quantised tiles
// are refilled fragment by fragment inside the phases).  The NT = 16 variant fits
// 256 registers, so two workgroups share a CU and their phases overlap.  The
// workgroup merges its waves through LDS and writes one partial, or the final
// rows when the launch has a single split.  BITS: 16, 8 or 4 per cached value.
// ---------------------------------------------------------------------------
// KEEP = 1: a sparse key selection, one byte per key position (0 drops the key), as the reference's decode kernels take it
// (keep[p], sources/TinyTitanCore/Metal/Attention/attention.metal:182-188, :229): a dropped key is as if it were absent.
// KEEP = 2: one such row of bytes per query row, keep[t * stride + key], as its chunk kernels take it
// (sources/TinyTitanCore/Metal/Prefill/prefill.metal:1063-1068, :1129).
// KEEP = 3: the same selection as per-query index lists (keepIdx / keepCount, prefill.metal:1069-1117), served from the
// plan keep_plan_kernel makes of them: per token tile the ascending list of key blocks its tokens keep a key of, and per
// entry and token the kept keys as 32 bits -- the walk costs the selection, never the context.
// KEEP = 4: the same, where few of a touched block's keys are listed (fp16 pages, tiles of 32): the plan lists groups of
// four keys, and eight listed groups, wherever they lie, make a turn of the loop.
// KEEP = 5: KEEP = 3 whose blocks' loads cover the listed keys only (lists_fetch_by_key).
// The hot arguments, this workgroup's sequence entry and where the rows go and their gate beside them, by five scalar loads issued
// together (the compiler would fetch each field where it is first used: five or six dependent trips to the kernarg segment before
// the first K/V load can go out, about 0.15 us each, and another ahead of the gate's loads).
typedef int i16v __attribute__((ext_vector_type(16)));
struct HotWords {
    i16v lo, hi;
};
struct SplitKOut {
    const _Float16 *gate;
    _Float16 *out;
    long long g_seq_stride, g_tok_stride, o_seq_stride, o_tok_stride;
};
static_assert(offsetof(SplitKArgs, gate) == 0x480 && offsetof(SplitKArgs, o_tok_stride) == 0x480 + offsetof(SplitKOut, o_tok_stride) &&
                  offsetof(SplitKArgs, out) == 0x480 + offsetof(SplitKOut, out) && sizeof(SplitKOut) == 48,
              "load_args' offsets");
__device__ __forceinline__ void load_args(SplitKHot &hot, SplitKSeq &sq, SplitKOut &out, int seq) {
    typedef int i8v __attribute__((ext_vector_type(8)));
    struct OutWords {
        i8v lo;
        i4 hi;
    };
    const unsigned long long base = (unsigned long long)__builtin_amdgcn_kernarg_segment_ptr();
    const unsigned long long entry = base + (unsigned)seq * (unsigned)sizeof(SplitKSeq);
    HotWords w;
    i4 e, t_hi;
    i8v t_lo;
    asm volatile("s_load_dwordx16 %0, %5, 0x0\n\ts_load_dwordx16 %1, %5, 0x40\n\ts_load_dwordx4 %2, %6, 0x80\n\t"
                 "s_load_dwordx8 %3, %5, 0x480\n\ts_load_dwordx4 %4, %5, 0x4a0\n\ts_waitcnt lgkmcnt(0)"
                 : "=&s"(w.lo), "=&s"(w.hi), "=&s"(e), "=&s"(t_lo), "=&s"(t_hi)
                 : "s"(base), "s"(entry)
                 : "memory");
    hot = __builtin_bit_cast(SplitKHot, w);
    sq = __builtin_bit_cast(SplitKSeq, e);
    const OutWords t = {t_lo, t_hi};
    __builtin_memcpy(&out, &t, sizeof(out));
}
typedef __attribute__((address_space(4))) const i4 *seq_entries;  // SplitKSeq: [3] is first_split
__device__ __forceinline__ seq_entries seq_table() {
    return (seq_entries)((__attribute__((address_space(4))) const char *)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(SplitKArgs, seq));
}
static_assert(kMaxSeqPerLaunch == 64 && offsetof(SplitKSeq, first_split) == 12, "a lane per sequence");
static_assert(offsetof(SplitKArgs, hot) == 0 && offsetof(SplitKArgs, seq) == 0x80, "load_args' offsets");

// STREAM: the launch reads every K/V byte once (see kStreamed); 2: and its V operands are paired (see v_tile_dim).
// A row's 32 selection bytes of one key block, as 8 words in two loads (the row stride is a multiple of 4 bytes, which is
// all a buffer load of four dwords asks for; dwords past the buffer's range read as zero one by one).
__device__ __forceinline__ void load_row_words(unsigned (&dst)[8], __amdgpu_buffer_rsrc_t rsrc, unsigned bytes) {
    const u4v lo = __builtin_bit_cast(u4v, __builtin_amdgcn_raw_buffer_load_b128(rsrc, bytes, 0, 0));
    const u4v hi = __builtin_bit_cast(u4v, __builtin_amdgcn_raw_buffer_load_b128(rsrc, bytes + 16u, 0, 0));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        dst[i] = lo[i];
        dst[4 + i] = hi[i];
    }
}

template <int D, int NT, int WAVES, int BITS, int KEEP = 0, int STREAM = 0>
__global__ __launch_bounds__(WAVES * 64, (NT == 16 && KEEP < 2 ? 2 : 1)) void attn_splitk_kernel(const SplitKArgs args) {
    constexpr bool PAIRED = STREAM == 2;
    static_assert(!PAIRED || (D == 256 && NT == 32 && BITS == 16 && KEEP == 0));
    constexpr int AUX = (STREAM ? kStreamed : 0) | (PAIRED ? kPaired : 0);
    extern __shared__ float lds[];
    constexpr int ROW = D + kLdsPad;  // staged O row stride in floats
    constexpr int REGION = NT * ROW + NT * 2;
    constexpr int KS = (NT == 32) ? D / 16 : D / 32;
    constexpr unsigned BLK_BYTES = BITS == 16 ? 32 * D * 2 : 32 * D * BITS / 8 + 32 * (D / 64) * 4;  // bytes per block
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // scalar: block pointers stay in SGPRs
    const Lane<D, NT> ln(lane, PAIRED);
    const int li = ln.li, g = ln.g;
    int seq = blockIdx.z;
    SplitKHot a;
    SplitKSeq sq;
    SplitKOut out;
    load_args(a, sq, out, seq);
    int split = blockIdx.x, tile = blockIdx.y;
    if (a.flags & kHotPackedSplits) {
        // Sequences of unlike lengths, their splits one behind the other in x: the entries of all of them in one load (those
        // past the last start beyond every split), and this split's sequence is the last that starts no later.
        const int first = seq_table()[lane][3];
        seq = (int)__popcll(__ballot(first <= split)) - 1;
        sq = __builtin_bit_cast(SplitKSeq, seq_table()[seq]);
        split -= sq.first_split;
    }
    if (a.flags & kHotXcdGrid) {  // many token tiles: the (split, tile) pairs are dealt out XCD by XCD, tile fastest
        const unsigned pairs = (unsigned)a.n_tiles * (unsigned)a.n_splits_max, per_xcd = (pairs + 7u) >> 3;
        const unsigned pair = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
        if (pair >= pairs) return;  // the grid is rounded up to a multiple of eight
        split = (int)(pair / (unsigned)a.n_tiles);
        tile = (int)(pair - (unsigned)split * (unsigned)a.n_tiles);
    }
    const TileInfo ti = tile_info(a, sq, tile);
    const int k_begin = ti.k0 + split * a.split_len;
    if (k_begin >= ti.tile_end && split != 0) return;  // split 0 always runs so that an empty range yields zeros
    const int k_end = min(k_begin + a.split_len, ti.tile_end);
    const int b_end = (k_end + 31) >> 5;

    const size_t page = ((size_t)sq.slot * a.n_kv_heads + ti.kvh) * (size_t)a.page_elems;
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(a.k_layer + page, (unsigned)(a.page_elems * 2));
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(a.v_layer + page, (unsigned)(a.page_elems * 2));

    // This lane's query row.
    const int t_local = (li * a.gh_inv) >> 16;  // li / gh
    const int hg = li - t_local * a.gh;
    const bool valid = t_local < ti.tile_rows;
    const int tok = ti.t0 + (valid ? t_local : 0);  // clamped so that the address is always in range
    const int head = ti.kvh * a.group + ti.hsub * a.gh + hg;
    const int lim = valid ? min(ti.total, ti.start + tok + 1) : 0;  // keys [lo, lim) are visible
    const int lo = (a.window > 0 && lim > a.window) ? lim - a.window : 0;  // sliding window: the last `window` keys
    const global_halves qp = (global_halves)(a.q + seq * a.q_seq_stride + tok * a.q_tok_stride + (long long)head * D);

    // Order of the first requests.  A wave's vector loads are issued in program order and an issue stalls while
    // the CU's memory pipeline is full, which it is as soon as every wave of the chip has asked for its first
    // block: a load behind 32 KiB of K/V requests only goes out when most of that data has arrived, microseconds
    // later.  So the query is requested first, then K of the first block; the wave then takes the query (short
    // wait: it was first in line), and V of the first block follows while the first scores are worked out.
    // The NT = 16 variant and every quantised variant keep the query fragments in LDS (the quantised 32-row
    // variant would otherwise need more than 512 registers), each wave its OWN copy, in the region it stages its
    // accumulators in at the end: no wave waits for another before its first block.  The fp16 32-row variant
    // keeps them in registers.
    constexpr bool Q_IN_LDS = NT == 16 || BITS != 16;
    constexpr int QSTEP = NT == 32 ? 16 : 32;  // dims per contraction step
    h8 qf[KS];
    h8 *qlds = reinterpret_cast<h8 *>(lds + wave * REGION);  // [step][lane] h8: KS KiB of the wave's REGION
    static_assert(!Q_IN_LDS || KS * 1024 <= REGION * 4, "the wave's query copy fits its merge region");
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        // quantised tiles contract the dims in their own order (two steps per loaded unit)
        const h8 x = load_h8(qp + (BITS == 16 ? QSTEP * s + 8 * g : q_dim_of_step<NT>(s, g)));
        qf[s] = x;
    }
    // Unconditional (straight-line code keeps the compiler's count of outstanding loads exact): a
    // wave whose first block lies past the split's end issues void loads.
    int b = (k_begin >> 5) + wave;
    typename std::conditional<BITS == 16, KTile<D, NT>, KTileQ<D, NT, BITS>>::type kt;
    typename std::conditional<BITS == 16, VTile<D, NT>, VTileQ<D, NT, BITS>>::type vt;
    // Selection bytes: lane i (and i + 32) holds the byte of key 32 b + i of the block in hand; the next block's
    // are loaded a block ahead.  Past the sequence's end the buffer load returns 0 (those keys are not visible anyway).
    // A block without a kept key is not read: its loads are void (no memory traffic), its turn works on zeros that
    // the selection masks anyway, so the HBM bytes of a selection are the blocks it touches, not the context.
    // (Skipping the turn's arithmetic too, with a branch around it, made the kernel slower: the compiler then
    // waits for every load in flight at the join.)  Where the mask is tested block by block, the first block of a
    // wavefront is read before its bytes are known -- waiting for them would put a round trip in front of it.
    // Where the mask starts on a word boundary the wavefront learns up front which of its blocks hold a kept
    // key at all -- lane j reads the 32 bytes of its j-th block, one ballot makes a 64-bit word of them (the host
    // keeps a split to 64 blocks per wavefront) -- and then walks only those, from the first: their arithmetic goes as
    // well, and with a selection of one group in eight blocks most wavefronts read none or one (read before its bytes were
    // known, every wavefront's first block was 33 MB a launch: 131k keys 20.7 -> 15.7 us with the step behind it).
    __amdgpu_buffer_rsrc_t rkeep;
    unsigned keep_cur = 1, keep_next = 1, keep_after = 1;
    const int b_first = b;
    unsigned long long todo = 0;  // bit j: block b_first + j * WAVES is still to be worked on
    unsigned first_keys = ~0u;  // the first block's keys that some row keeps
    if constexpr (KEEP == 1) {
        rkeep = make_rsrc(args.keep + seq * args.keep_seq_stride, (unsigned)ti.total);
        const int mine = b_first < b_end ? (b_end - b_first + WAVES - 1) / WAVES : 0;  // this wavefront's blocks, at most 64
        todo = mine >= 64 ? ~0ull : ((1ull << mine) - 1ull);
        if (a.keep_words) {
            unsigned words[8], block_keys = 0;  // bit i: key i of the lane's block is kept
#pragma unroll
            for (int i = 0; i < 8; ++i) words[i] = __builtin_amdgcn_raw_buffer_load_b32(rkeep, (unsigned)(b_first + lane * WAVES) * 32u + 4u * i, 0, 0);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const unsigned set = (((words[i] & 0x7f7f7f7fu) + 0x7f7f7f7fu) | words[i]) & 0x80808080u;  // a byte's top bit: the byte is not zero
                block_keys |= ((set >> 7) * 0x10204080u >> 28) << (4 * i);
            }
            unsigned long long touched = __ballot(block_keys != 0);
            // A mask is exactly `total` bytes: when that is not a multiple of 4 its last word straddles the end of
            // the buffer's range and may read as zero whatever its bytes hold.  The block of the last key is
            // therefore always walked and fetched whole; its keys are still tested byte by byte.
            int tail_j = -1;
            if (ti.total & 3) {
                const int last_block = (ti.total - 1) >> 5, j = (last_block - b_first) / WAVES;
                if (last_block >= b_first && (last_block - b_first) % WAVES == 0 && j < 64) {
                    touched |= 1ull << j;
                    tail_j = j;
                }
            }
            todo &= touched;
            const int j0 = todo ? __ffsll((long long)todo) - 1 : 0;
            b = todo ? b_first + j0 * WAVES : b_end;
            first_keys = j0 == tail_j ? ~0u : (unsigned)__builtin_amdgcn_readlane((int)block_keys, j0);
            todo &= todo - 1;
            keep_cur = __builtin_amdgcn_raw_buffer_load_b8(rkeep, (unsigned)b * 32u + (unsigned)(lane & 31), 0, 0);
            const int nb0 = todo ? b_first + (__ffsll((long long)todo) - 1) * WAVES : b_end;
            keep_next = __builtin_amdgcn_raw_buffer_load_b8(rkeep, (unsigned)nb0 * 32u + (unsigned)(lane & 31), 0, 0);
        } else {
            todo &= ~1ull;  // the first block is in hand
            keep_cur = __builtin_amdgcn_raw_buffer_load_b8(rkeep, (unsigned)b * 32u + (unsigned)(lane & 31), 0, 0);
            // block by block: the next block is the wavefront's second, and its bytes are asked for ahead of the
            // first block's data
            keep_next = __builtin_amdgcn_raw_buffer_load_b8(rkeep, (unsigned)(b + WAVES) * 32u + (unsigned)(lane & 31), 0, 0);
        }
    }
    // Per-query selections: the lane's own row of bytes, 32 per block as 8 words, a block ahead.  The range of the
    // buffer is the rows' extent, so a read past it (void blocks, rows of padding lanes) returns 0.
    // Here too a block that no row of the tile keeps a key of is not read: the words of the next two blocks are in hand.
    unsigned row_cur[8], row_next[8], row_after[8];
    unsigned row_bytes0 = 0;
    unsigned window_words[kKeepWindows] = {};
    int *const listed = reinterpret_cast<int *>(lds + WAVES * REGION);  // the workgroup's touched blocks, then [wave][window] counts
    int n_listed = 0, list_at = 0, nxt = 0, aft = 0;
    auto listed_block = [&](int i) { return i < n_listed ? __builtin_amdgcn_readfirstlane(listed[i]) : b_end; };
    if constexpr (KEEP == 2) {
        rkeep = make_rsrc(args.keep + seq * args.keep_seq_stride, (unsigned)((long long)a.rows * args.keep_row_stride));
        row_bytes0 = (unsigned)((long long)tok * args.keep_row_stride);
        load_row_words(row_cur, rkeep, row_bytes0 + (unsigned)b * 32u);
        if (a.keep_words) {
            // Long splits: which of the split's blocks does ANY row of the tile keep a key of?  Wavefront w looks at
            // the split's blocks [512 w, 512 w + 512) -- lane j at blocks j, j + 64, ... of them, consecutive lanes
            // at consecutive 32 bytes, so that a load instruction reads a contiguous 2 KiB -- in every token's row of
            // bytes (a tile's rows are its tokens times the heads that share them); the touched blocks go into a
            // list in LDS and the loop walks only those, arithmetic included, so a sparse chunk costs its selection
            // and not its context -- and a split can be as long as kKeepWindows * 64 blocks a wavefront: few
            // workgroups, each with one prologue, one merge and one partial.
            // Two rows at a time, straight-line: their 4 kKeepWindows loads are all in flight together (a loop over
            // single rows waits for each row's loads before it asks for the next: ~3 us a row); a tile's odd last
            // row is paired with void loads.
            for (int r = 0; r < ti.tile_rows; r += 2) {
                u4v got[2][kKeepWindows][2];
#pragma unroll
                for (int rr = 0; rr < 2; ++rr) {
                    const unsigned row = r + rr < ti.tile_rows ? (unsigned)((long long)(ti.t0 + r + rr) * args.keep_row_stride) : kVoidLoad;
#pragma unroll
                    for (int w = 0; w < kKeepWindows; ++w) {
                        const unsigned at = row + (unsigned)((k_begin >> 5) + (wave * kKeepWindows + w) * 64 + lane) * 32u;
                        got[rr][w][0] = __builtin_bit_cast(u4v, __builtin_amdgcn_raw_buffer_load_b128(rkeep, at, 0, 0));
                        got[rr][w][1] = __builtin_bit_cast(u4v, __builtin_amdgcn_raw_buffer_load_b128(rkeep, at + 16u, 0, 0));
                    }
                }
#pragma unroll
                for (int w = 0; w < kKeepWindows; ++w) {
                    const u4v any = got[0][w][0] | got[0][w][1] | got[1][w][0] | got[1][w][1];
                    window_words[w] |= any[0] | any[1] | any[2] | any[3];
                }
            }
        } else {
            load_row_words(row_next, rkeep, row_bytes0 + (unsigned)(b + WAVES) * 32u);
        }
    }
    // Index lists: this wavefront takes entries e_at, e_at + WAVES, ... of the tile's list up to the split's end.  The block
    // of the entry after next and the row's bits of the next two entries are always on their way.
    const int *plan_blocks_tile = nullptr;
    const unsigned *plan_bits_tile = nullptr;
    int e_at = 0, e_hi = 0, walked = 0;
    constexpr bool LISTS = KEEP == 3 || KEEP == 5;
    constexpr bool BY_KEY = KEEP == 1 || KEEP == 5;  // see Voids
    typedef int i2 __attribute__((ext_vector_type(2)));
    i2 after_entry = {0, 0};  // block, keys of it that any token keeps
    unsigned nxt_keys = ~0u;
    unsigned bits_cur = ~0u, bits_next = ~0u, bits_after = ~0u;
    const int bits_col = valid ? t_local : 0;
    // A place in the tile's list as the plan gives it, inside the list's room whatever the words hold (nothing else bounds the reads below).
    auto plan_place = [&](int word) { return (int)min((unsigned)__builtin_amdgcn_readfirstlane(word), (unsigned)args.plan_cap); };
    auto plan_entry = [&](int k) {  // the wavefront's k-th entry (a load; every lane the same words)
        const int e = e_at + k * WAVES;
        const int *at = plan_blocks_tile + 2 * (size_t)(e < e_hi ? e : 0);
        i2 got = {0, 0};
        if constexpr (BY_KEY) got = *reinterpret_cast<const i2 *>(at);
        else got[0] = at[0];  // (the register of a second word that nothing uses is given to something else, which then waits for the load)
        const i2 none = {b_end, 0};
        return e < e_hi ? got : none;
    };
    auto plan_row_bits = [&](int k) {
        const int e = e_at + k * WAVES;
        const unsigned got = plan_bits_tile[(size_t)(e < e_hi ? e : 0) * a.tt + bits_col];
        return e < e_hi ? got : 0u;
    };
    if constexpr (LISTS) {
        const int *ranges = args.plan_ranges + (size_t)ti.tok_tile * (a.n_splits_max + 1) + split;
        e_at = plan_place(ranges[0]) + wave;
        e_hi = plan_place(ranges[1]);
        plan_blocks_tile = args.plan_blocks + (size_t)ti.tok_tile * args.plan_cap * 2;
        plan_bits_tile = args.plan_bits + (size_t)ti.tok_tile * args.plan_cap * a.tt;
        const i2 e0 = plan_entry(0), e1 = plan_entry(1);
        after_entry = plan_entry(2);
        bits_cur = plan_row_bits(0);
        bits_next = plan_row_bits(1);
        b = __builtin_amdgcn_readfirstlane(e0[0]);
        first_keys = (unsigned)__builtin_amdgcn_readfirstlane(e0[1]);
        nxt = __builtin_amdgcn_readfirstlane(e1[0]);
        nxt_keys = (unsigned)__builtin_amdgcn_readfirstlane(e1[1]);
    }
    // Groups: this wavefront takes runs of eight list positions v, v + WAVES, ... (aligned: a run may reach over the ends of the
    // split's stretch [g_lo, g_hi), whose outside is void and masked).  A run's ids are asked for two turns ahead, its
    // row bits one.
    int run = 0, run_end = 0, g_lo = 0, g_hi = 0;
    int ids_next[5];
    GroupOffsets at_next;
    auto group_ids = [&](int (&ids)[5], int v) {
        const int place[5] = {li >> 2, g, g + 2, 4 + g, 6 + g};
        const int base = 8 * min(v, run_end - 1);
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            const int p = base + place[i], got = plan_blocks_tile[p];
            ids[i] = v < run_end && p >= g_lo && p < g_hi ? got : -1;
        }
    };
    auto run_bits = [&](int v) {
        const unsigned got = plan_bits_tile[(size_t)min(v, run_end - 1) * a.tt + bits_col];
        const int lo_cut = max(g_lo - 8 * v, 0), hi_cut = g_hi - 8 * v;  // positions of the run inside the stretch: [lo_cut, hi_cut)
        const unsigned inside = (~0u << (4 * min(lo_cut, 7))) & (hi_cut >= 8 ? ~0u : (1u << (4 * max(hi_cut, 0))) - 1u);
        return v < run_end && valid ? got & inside : 0u;
    };
    if constexpr (KEEP == 4) {
        const int *ranges = args.plan_ranges + (size_t)ti.tok_tile * (a.n_splits_max + 1) + split;
        g_lo = plan_place(ranges[0]);
        g_hi = plan_place(ranges[1]);
        run_end = g_hi > g_lo ? (g_hi + 7) >> 3 : 0;
        run = (g_lo >> 3) + wave;
        plan_blocks_tile = args.plan_blocks + (size_t)ti.tok_tile * args.plan_cap;
        plan_bits_tile = args.plan_bits + (size_t)ti.tok_tile * (args.plan_cap >> 3) * a.tt;
        b = b_end;  // (the walk over blocks finds nothing)
    }
    const bool first_real = b < b_end;
    const unsigned first_bytes = first_real ? (unsigned)(a.ring_blocks ? b % a.ring_blocks : b) * BLK_BYTES : 0u;
    Voids<D, NT> first_void(first_real ? 0u : kVoidLoad);
    if constexpr (BY_KEY) first_void = Voids<D, NT>(first_real ? 0u : kVoidLoad, first_keys, ln);
    if constexpr (KEEP == 4) {
        if (run_end > 0) {
            int ids_first[5];
            group_ids(ids_first, run);
            group_ids(ids_next, run + WAVES);
            bits_cur = run_bits(run);
            at_next = group_offsets<D>(ids_first, ln);
            load_k_groups<D>(kt, rk, at_next);
        }
    } else {
        load_k<AUX>(kt, rk, first_bytes, ln, first_void);
    }
    __builtin_amdgcn_sched_barrier(0);  // the first block's K loads are issued HERE, before the query is waited for
    if constexpr (KEEP == 2) {
        if (a.keep_words) {
            // One list for the workgroup, its entries dealt out to the wavefronts in turn: every wavefront then walks
            // a quarter of the split's touched blocks, however they fall among the blocks each one looked at.
            // (the split has at most WAVES * kKeepWindows * 64 blocks: the host sees to it)
            int *const counts = listed + WAVES * kKeepWindows * 64;  // [wave][window]
            unsigned long long words[kKeepWindows];
#pragma unroll
            for (int w = 0; w < kKeepWindows; ++w) {
                const int j = (wave * kKeepWindows + w) * 64 + lane;  // the block's place in the split
                // (the wavefronts' first blocks -- the split's first WAVES -- are in hand)
                words[w] = __ballot(window_words[w] != 0 && (k_begin >> 5) + j < b_end && j >= WAVES);
                if (lane == 0) counts[wave * kKeepWindows + w] = __popcll(words[w]);
            }
            __syncthreads();
            int at = 0;
#pragma unroll
            for (int v = 0; v < WAVES; ++v)  // entries in (wave, window, lane) order: ascending blocks
#pragma unroll
                for (int w = 0; w < kKeepWindows; ++w) {
                    if (v == wave && w == 0) at = n_listed;
                    n_listed += counts[v * kKeepWindows + w];
                }
#pragma unroll
            for (int w = 0; w < kKeepWindows; ++w) {
                if ((words[w] >> lane) & 1ull)
                    listed[at + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(words[w] >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)words[w], 0u))] =
                        (k_begin >> 5) + (wave * kKeepWindows + w) * 64 + lane;
                at += __popcll(words[w]);
            }
            __syncthreads();
            nxt = listed_block(wave);
            aft = listed_block(wave + WAVES);
            load_row_words(row_next, rkeep, row_bytes0 + (unsigned)nxt * 32u);
        }
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        qf[s] = valid ? qf[s] : (h8)(_Float16)0;
        if constexpr (Q_IN_LDS) qlds[s * 64 + lane] = qf[s];  // read back by this wave only: no barrier
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (KEEP == 4) {
        if (run_end > 0) load_v_groups<D>(vt, rv, at_next);
    } else {
        load_v<AUX>(vt, rv, first_bytes, ln, first_void);
    }
    __builtin_amdgcn_sched_barrier(0);

    RowState<D, NT> st;
    st.init();
    typename RowState<D, NT>::acc_t bias_acc = (typename RowState<D, NT>::acc_t)0.0f;  // quantised pages only
    if constexpr (KEEP == 4) {
        for (; run < run_end; run += WAVES) {
            Scores<D, NT> sc;
            at_next = group_offsets<D>(ids_next, ln);
            group_ids(ids_next, run + 2 * WAVES);
            bits_next = run_bits(run + WAVES);
            group_scores_refill<D>(sc, kt, qf, rk, at_next);
            group_softmax_pv_refill<D>(st, sc, vt, ln, a.scale_log2e, rv, at_next, bits_cur);
            bits_cur = bits_next;
        }
    }
    // The next block's loads are issued UNCONDITIONALLY (void loads past the split's end).  A branch
    // around them would leave the compiler unable to count the loads in flight, and it would then
    // make the P.V step wait for the next block's K tile as well as for its own V tile.
    while (KEEP != 4 && b < b_end) {
        Scores<D, NT> sc;
        int nb = b + WAVES;
        unsigned kept = ~0u;
        bool next_kept = true;
        unsigned next_keys = ~0u;  // the next block's keys that some row keeps
        const unsigned *row_keep = nullptr;
        if constexpr (KEEP == 1) {
            // the next block and the one after it, off the word of blocks still to do
            nb = todo ? b_first + (__ffsll((long long)todo) - 1) * WAVES : b_end;
            todo &= todo - 1;
            const int after = todo ? b_first + (__ffsll((long long)todo) - 1) * WAVES : b_end;
            keep_after = __builtin_amdgcn_raw_buffer_load_b8(rkeep, (unsigned)after * 32u + (unsigned)(lane & 31), 0, 0);
            kept = (unsigned)__ballot(keep_cur != 0);  // lanes 32..63 repeat lanes 0..31
            next_keys = (unsigned)__ballot(keep_next != 0);
            next_kept = next_keys != 0u;
        }
        if constexpr (KEEP == 2) {
            if (a.keep_words) {
                // the next touched block and the one after it, off the list (the one after that is read here, a turn ahead)
                nb = nxt;
                nxt = aft;
                aft = listed_block(wave + (list_at + 2) * WAVES);
                ++list_at;
                load_row_words(row_after, rkeep, row_bytes0 + (unsigned)nxt * 32u);
            } else {
                unsigned any = 0;
                load_row_words(row_after, rkeep, row_bytes0 + (unsigned)(nb + WAVES) * 32u);
#pragma unroll
                for (int i = 0; i < 8; ++i) any |= row_next[i];
                next_kept = __ballot(any != 0) != 0ull;
            }
            row_keep = row_cur;
        }
        unsigned row_bits = ~0u;
        if constexpr (LISTS) {
            nb = nxt;
            next_keys = nxt_keys;
            nxt = __builtin_amdgcn_readfirstlane(after_entry[0]);
            nxt_keys = (unsigned)__builtin_amdgcn_readfirstlane(after_entry[1]);
            after_entry = plan_entry(walked + 3);
            bits_after = plan_row_bits(walked + 2);
            ++walked;
            row_bits = bits_cur;
        }
        const bool real = nb < b_end && next_kept;
        const unsigned next = real ? (unsigned)(a.ring_blocks ? nb % a.ring_blocks : nb) * BLK_BYTES : 0u;
        Voids<D, NT> vo(real ? 0u : kVoidLoad);
        if constexpr (BY_KEY) vo = Voids<D, NT>(real ? 0u : kVoidLoad, next_keys, ln);
        if constexpr (BITS == 16 && NT == 32) {
            block_scores_refill<AUX, D>(sc, kt, qf, rk, next, ln, vo);
            block_softmax_pv_refill<AUX, D>(st, sc, vt, ln, b << 5, lo, lim, a.scale_log2e, rv, next, vo, kept, row_keep, row_bits);
        } else if constexpr (BITS == 16) {
            block_scores(sc, kt, qf, qlds, lane);
            load_k<AUX>(kt, rk, next, ln, vo);
            block_softmax_pv<D, NT>(st, sc, vt, ln, b << 5, lo, lim, a.scale_log2e, kept, row_keep, row_bits);
            load_v<AUX>(vt, rv, next, ln, vo);
        } else {  // the phases refill their tiles as they go
            block_scores<AUX, D, NT, BITS>(sc, kt, qf, qlds, lane, rk, next, ln, vo);
            block_softmax_pv<AUX, D, NT, BITS>(st, sc, vt, ln, b << 5, lo, lim, a.scale_log2e, bias_acc, rv, next, vo, kept,
                                          row_keep, row_bits);
        }
        if constexpr (KEEP == 1) {
            keep_cur = keep_next;
            keep_next = keep_after;
        }
        if constexpr (KEEP == 2) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                row_cur[i] = row_next[i];
                row_next[i] = row_after[i];
            }
        }
        if constexpr (LISTS) {
            bits_cur = bits_next;
            bits_next = bits_after;
        }
        b = nb;
    }
    if constexpr (BITS != 16) {
        // Level accumulators carry the probability boost; the bias sums sit in row `group` of
        // bias_acc, i.e. in register `group` of the lane group 0 lane that owns this lane's query row.
        constexpr int TILES_PER_GROUP = RowState<D, NT>::MT / (D / 64);
#pragma unroll
        for (int grp = 0; grp < D / 64; ++grp) {
            const float group_bias = __shfl(bias_acc[grp], li);
#pragma unroll
            for (int mt = grp * TILES_PER_GROUP; mt < (grp + 1) * TILES_PER_GROUP; ++mt)
                st.o[mt] = st.o[mt] * (1.0f / kProbBoost) + group_bias;
        }
    }

    // A launch of one split ends in the output rows: the gate's values of this thread's items, all asked for ahead of the staging and its
    // barrier.  (Each asked for where it was stored, the items waited for memory one behind the other: a layer's three launches over 99 keys,
    // 2 rows of 16/2 heads of 256, 15.3 us then and 13.9 now; 4 rows over 200 keys 17.1 / 15.7, 20 rows of a prompt 17.4 / 15.9.)
    const int n_valid = ti.tile_rows * a.gh;
    constexpr int D4 = D / 4, ITEMS = NT * D4 / (WAVES * 64), ROUND = WAVES * 64 / D4;
    const bool last = a.n_splits_max == 1;
    h4 gate[ITEMS];
    if (last && out.gate) {
        const global_halves rows = (global_halves)(out.gate + seq * out.g_seq_stride + ti.t0 * out.g_tok_stride + (long long)(ti.kvh * a.group + ti.hsub * a.gh) * D);
        const int d = threadIdx.x % D4 * 4;
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            if (i * ROUND >= n_valid) break;
            const int n = min(i * ROUND + (int)threadIdx.x / D4, n_valid - 1), tl = (n * a.gh_inv) >> 16;
            gate[i] = *(const __attribute__((address_space(1))) h4_unaligned *)(rows + (tl * out.g_tok_stride + (n - tl * a.gh) * D + d));
        }
    }

    // Stage this wave's state in LDS.
    float l = st.l;
    l = (NT == 32) ? sum_across_halves(l) : sum_across_quarters(l);
    float *region = lds + wave * REGION;
    if (!valid) {
        // padding row: nothing to merge
    } else if constexpr (NT == 32) {
#pragma unroll
        for (int mt = 0; mt < D / 32; ++mt)
#pragma unroll
            for (int vq = 0; vq < 4; ++vq) {
                f4 x = {st.o[mt][4 * vq], st.o[mt][4 * vq + 1], st.o[mt][4 * vq + 2], st.o[mt][4 * vq + 3]};
                *reinterpret_cast<f4 *>(region + li * ROW + v_tile_dim(mt, PAIRED) + v_row_dim(8 * vq + 4 * g, PAIRED)) = x;
            }
    } else {
#pragma unroll
        for (int mt = 0; mt < D / 16; ++mt) *reinterpret_cast<f4 *>(region + li * ROW + 16 * mt + 4 * g) = st.o[mt];
    }
    if (g == 0 && valid) {
        region[NT * ROW + 2 * li] = st.m;
        region[NT * ROW + 2 * li + 1] = l;
    }
    __syncthreads();

    // Merge the waves' states; every thread takes (row, 4 dims) items.
    const size_t pbase = (((size_t)sq.first_split + split) * a.n_tiles + tile) * NT;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const int n = i * ROUND + threadIdx.x / D4, d = threadIdx.x % D4 * 4;
        if (n >= n_valid) break;
        float mw[WAVES];
        float ms = kNegBig;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            mw[w] = lds[w * REGION + NT * ROW + 2 * n];
            ms = fmaxf(ms, mw[w]);
        }
        f4 acc = (f4)0.0f;
        float lsum = 0.0f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float f = fast_exp2(mw[w] - ms);
            lsum += f * lds[w * REGION + NT * ROW + 2 * n + 1];
            acc += f * *reinterpret_cast<const f4 *>(lds + w * REGION + n * ROW + d);
        }
        if (last) {
            const int tl = (n * a.gh_inv) >> 16;
            const int hh = ti.kvh * a.group + ti.hsub * a.gh + (n - tl * a.gh);
            store_out4_gated(out, seq, ti.t0 + tl, hh, d, D, acc, lsum > 0.0f ? 1.0f / lsum : 0.0f, (a.flags & kHotAligned) != 0, gate[i]);
        } else {
            *reinterpret_cast<f4 *>(a.part_o + (pbase + n) * D + d) = acc;
            if (d == 0) {
                a.part_ml[(pbase + n) * 2] = ms;
                a.part_ml[(pbase + n) * 2 + 1] = lsum;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Pass 2: cross-split log-sum-exp combine, gate and fp16 store.
// grid = (row within tile * D/64 + dim chunk, tile, sequence), 256 threads.
// Every wave first finds the row's global max over all splits (a few scalars
// per lane), which makes the per-split terms independent: a thread owns 4
// output dims (lane % 16) of the workgroup's 64-dim chunk and the splits
// 4 * wave + lane / 16, + 16, ..., all loads in flight at once; the 16 split
// groups add up through two shuffles and LDS.  All-empty input yields zeros
// (sources/TinyTitanCore/Metal/Attention/attention.metal:418-427).
// ---------------------------------------------------------------------------
// What such a pass takes is its chain of trips to memory, and it is two: the arguments, then the gate, the
// maxima and the partial rows together -- with the gate converted where it was loaded, its arguments read in a trip of
// their own and the second 64 maxima behind the first they were five.  A decode step's launch 0.2 us less (two layers of 7
// sequences of 300 .. 9,000 keys over 4 bits 40.8 -> 40.0 us, four of one of 20,010 over 8 bits 78.2 -> 77.4), the rows kernel
// behind a chunk of 128 rows over key ranges 2.2 (two layers behind 32,640 keys 240.5 -> 236.1).
typedef float f2 __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(1))) f2 *global_pairs;  // part_ml: a partial row's (max, sum)
typedef const __attribute__((address_space(1))) char *global_bytes;

// What attn_combine_kernel reads in the place of a split that is not there: a partial row of zeros.  (Any other row's values would do but for
// infinite ones, which a factor of zero makes NaN of; a select behind the load is instructions on every value, a branch around it a wait of its own.)
static __device__ __align__(256) float no_split[256];
__device__ __forceinline__ global_bytes no_row() {
    global_bytes at = (global_bytes)no_split;
    asm("" : "+s"(at));  // (an address like the others, not zeros the compiler knows of and branches to)
    return at;
}

__device__ __forceinline__ int splits_of(const TileInfo &ti, int split_len) {
    return (int)((unsigned)(max(ti.tile_end - ti.k0, 1) + split_len - 1) / (unsigned)split_len);  // (an empty range has one, of zeros)
}

template <int D, int NT>
__global__ __launch_bounds__(256) void attn_combine_kernel([[maybe_unused]] const SplitKArgs args) {  // (load_args reads them)
    constexpr int DCH = D / 64;
    __shared__ float sm[4][68];
    const int n = blockIdx.x / DCH, dchunk = blockIdx.x - n * DCH;
    const int tile = blockIdx.y, seq = blockIdx.z;
    SplitKHot a;
    SplitKSeq sq;
    SplitKOut out;
    load_args(a, sq, out, seq);
    const TileInfo ti = tile_info(a, sq, tile);
    if (n >= ti.tile_rows * a.gh) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n_splits = splits_of(ti, a.split_len);
    // partial rows of split s: ((first_split + s) * n_tiles + tile) * NT + n
    const size_t tstride = (size_t)a.n_tiles * NT;
    const size_t first_row = (size_t)sq.first_split * tstride + (size_t)tile * NT + n;
    const int d = dchunk * 64 + (lane & 15) * 4;
    const global_pairs ml = (global_pairs)a.part_ml + first_row;
    const global_bytes rows = (global_bytes)a.part_o + (first_row * D + d) * sizeof(float);
    const global_bytes zeros = no_row() + d * sizeof(float);
    auto partial_row = [&](int s) {
        return *(const __attribute__((address_space(1))) f4 *)(s < n_splits ? rows + s * tstride * (D * sizeof(float)) : zeros);
    };
    // the gate of the dim that a thread of the first wavefront stores at the end, first of all requests
    const int tl = (n * a.gh_inv) >> 16;
    const int hh = ti.kvh * a.group + ti.hsub * a.gh + (n - tl * a.gh);
    const long long out_dim = (long long)hh * D + dchunk * 64 + lane;
    const bool gated = wave == 0 && out.gate;
    _Float16 gate = (_Float16)0.0f;
    if (gated) gate = ((global_halves)out.gate)[seq * out.g_seq_stride + (ti.t0 + tl) * out.g_tok_stride + out_dim];
    const int s0 = wave * 4 + (lane >> 4);
    f4 acc = (f4)0.0f;
    float l = 0.0f, factor = 1.0f;
    // This thread's first BATCH splits are requested BEFORE the global max is known: their
    // addresses do not depend on it, so the max's loads and these share one trip to memory.
    auto sum_splits = [&](auto batch) {
        constexpr int BATCH = decltype(batch)::value, MAXIMA = (BATCH * 16 + 63) / 64;
        f4 po[BATCH];
        f2 pml[BATCH];
        float maxima[MAXIMA];
#pragma unroll
        for (int i = 0; i < MAXIMA; ++i) maxima[i] = ml[min(lane + 64 * i, n_splits - 1) * tstride][0];
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
            const int s = s0 + 16 * i;
            pml[i] = ml[(s < n_splits ? s : 0) * tstride];
            po[i] = partial_row(s);
        }
        __builtin_amdgcn_sched_barrier(0);  // (the maximum's wait is not to come in front of the rest of the requests)
        if (gated) {
            factor = sigmoid((float)gate);
            asm volatile("" : "+v"(factor));  // (here, while the rows are on their way, and not behind their sums)
        }
        float mg = maxima[0];
#pragma unroll
        for (int i = 1; i < MAXIMA; ++i) mg = fmaxf(mg, maxima[i]);
        for (int s = lane + 64 * MAXIMA; s < n_splits; s += 64) mg = fmaxf(mg, ml[s * tstride][0]);
        mg = wave_max_f32(mg, lane);
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
            const float f = s0 + 16 * i < n_splits ? fast_exp2(pml[i][0] - mg) : 0.0f;
            l += f * pml[i][1];
            acc += f * po[i];
        }
#pragma unroll 4
        for (int s = s0 + 16 * BATCH; s < n_splits; s += 16) {
            const f2 p = ml[s * tstride];
            const float f = fast_exp2(p[0] - mg);
            l += f * p[1];
            acc += f * partial_row(s);
        }
    };
    // (few splits: requests for the places of more would each pass through the CU's vector memory path; 34 splits in places for 64,
    // four layers of 4 rows behind 8,190 keys over 8 bits, 83.8 us, in places for 128 84.3)
    if (n_splits <= 32) sum_splits(std::integral_constant<int, 2>{});
    else if (n_splits <= 64) sum_splits(std::integral_constant<int, 4>{});
    else sum_splits(std::integral_constant<int, 8>{});
    // (lanes l, l ^ 16, l ^ 32, l ^ 48, added in that order: v_permlane16_swap / v_permlane32_swap, no trip through LDS)
    l = sum_across_quarters(l);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = sum_across_quarters(acc[i]);
    if (lane < 16) *reinterpret_cast<f4 *>(&sm[wave][lane * 4]) = acc;
    if (lane == 0) sm[wave][64] = l;
    __syncthreads();
    if (wave == 0) {
        float o = 0.0f, lsum = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            lsum += sm[w][64];
            o += sm[w][lane];
        }
        o *= lsum > 0.0f ? 1.0f / lsum : 0.0f;
        if (gated) o *= factor;
        typedef __attribute__((address_space(1))) _Float16 *global_out;
        ((global_out)out.out)[seq * out.o_seq_stride + (ti.t0 + tl) * out.o_tok_stride + out_dim] = (_Float16)o;
    }
}

// Pass 2 for launches of many tiles with few splits each (a chunk through the split-K tiles, or through the chunk
// kernel over key ranges): one workgroup per four rows of a tile instead of one per (row, 64 dims) -- the many tiny
// workgroups of attn_combine_kernel cost more to dispatch than these take to run.  A thread owns one (row, 4 dims)
// item and all of its splits, up to kCombineRowsSplits at a time: their loads are requested together, so a thread makes
// one trip to memory per turn, not one per split (the host sends more than two turns' worth to the other kernel).
// grid = (NT / 4, tile, sequence), 256 threads.
constexpr int kCombineRowsSplits = 16;

template <int D, int NT>
__global__ __launch_bounds__(256) void attn_combine_rows_kernel([[maybe_unused]] const SplitKArgs args) {  // (load_args reads them)
    constexpr int D4 = D / 4, ROWS = 4;
    static_assert(ROWS * D4 <= 256, "an item a thread");
    const int tile = blockIdx.y, seq = blockIdx.z;
    SplitKHot a;
    SplitKSeq sq;
    SplitKOut out;
    load_args(a, sq, out, seq);
    const TileInfo ti = tile_info(a, sq, tile);
    const int n = blockIdx.x * ROWS + (int)threadIdx.x / D4, d = ((int)threadIdx.x % D4) * 4;
    if ((int)threadIdx.x >= ROWS * D4 || n >= ti.tile_rows * a.gh) return;
    const int n_splits = splits_of(ti, a.split_len);
    const size_t tstride = (size_t)a.n_tiles * NT;
    const size_t first_row = (size_t)sq.first_split * tstride + (size_t)tile * NT + blockIdx.x * ROWS;
    const unsigned row_at = threadIdx.x * 16u, ml_at = threadIdx.x / D4 * 8u;  // this thread's in a split's four rows and pairs
    const int tl = (n * a.gh_inv) >> 16;
    const int hh = ti.kvh * a.group + ti.hsub * a.gh + (n - tl * a.gh);
    const bool aligned = (a.flags & kHotAligned) != 0;
    const h4 gate4 = load_gate4(out, seq, ti.t0 + tl, hh, d, D);
    float mg = kNegBig, l = 0.0f;
    f4 acc = (f4)0.0f;
    auto turn = [&](auto splits, int first) {
        constexpr int SPLITS = decltype(splits)::value;
        // Places past the row's last split read as zeros: the descriptors end behind it.  (Any other row's values times a factor of zero
        // would do but for infinite ones, which become NaN; the host keeps 16 places of a launch within 4 GiB.)
        const size_t base = first_row + first * tstride;
        const unsigned there = min(n_splits - first, SPLITS) * (unsigned)tstride;
        const __amdgpu_buffer_rsrc_t rows = make_rsrc(a.part_o + base * D, there * (unsigned)(D * sizeof(float)));
        const __amdgpu_buffer_rsrc_t pairs = make_rsrc(a.part_ml + base * 2, there * (unsigned)(2 * sizeof(float)));
        unsigned row_next = row_at, ml_next = ml_at, stride = (unsigned)tstride;
        f2 pml[SPLITS];
        f4 po[SPLITS];
        // Requests in this order: six pairs and rows in turn, the other pairs, the other rows.  (16 ranges of 128 rows of 16/2 heads of 256, 33 MB: 7.4 us,
        // all in turn 7.9, all rows in front 8.2, all pairs 7.85.)
        constexpr int IN_TURN = SPLITS < 6 ? SPLITS : 6;
        auto ask_row = [&](int i) {
            po[i] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rows, row_next, 0, 0));
            row_next += stride * (unsigned)(D * sizeof(float));
        };
#pragma unroll
        for (int i = 0; i < SPLITS; ++i) {
            pml[i] = __builtin_bit_cast(f2, __builtin_amdgcn_raw_buffer_load_b64(pairs, ml_next, 0, 0));
            asm volatile("" : "+s"(stride));  // (a place's offset is worked out here, not in front of all of them in a register of its own)
            ml_next += stride * (unsigned)sizeof(f2);
            if (i < IN_TURN) ask_row(i);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = IN_TURN; i < SPLITS; ++i) {
            asm volatile("" : "+s"(stride));
            ask_row(i);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_sched_barrier(0);  // (left alone, a request goes out when a row before it has come: fewer registers)
        float m_new = mg;
#pragma unroll
        for (int i = 0; i < SPLITS; ++i) m_new = fmaxf(m_new, first + i < n_splits ? pml[i][0] : kNegBig);
        const float keep = fast_exp2(mg - m_new);  // (first turn: what is kept is zero anyway)
        l *= keep;
        acc *= keep;
        mg = m_new;
#pragma unroll
        for (int i = 0; i < SPLITS; ++i) {
            const float f = first + i < n_splits ? fast_exp2(pml[i][0] - mg) : 0.0f;
            l += f * pml[i][1];
            acc += f * po[i];
        }
    };
    // (one turn up to kCombineRowsSplits splits, of four places where there are no more)
    if (n_splits <= 4) turn(std::integral_constant<int, 4>{}, 0);
    else
        for (int first = 0; first < n_splits; first += kCombineRowsSplits) turn(std::integral_constant<int, kCombineRowsSplits>{}, first);
    store_out4_gated(out, seq, ti.t0 + tl, hh, d, D, acc, l > 0.0f ? 1.0f / l : 0.0f, aligned, gate4);
}

// ---------------------------------------------------------------------------
// Host side: planning and launch.
// ---------------------------------------------------------------------------

// Behind the merge regions: the lists of touched blocks of a per-query selection, one per wave.
static constexpr size_t keep_list_bytes(int keep, int waves) { return keep == 2 ? (size_t)waves * kKeepWindows * (64 + 1) * sizeof(int) : 0; }

static size_t lds_bytes_for(int D, int NT, int waves) {
    // one merge region per wave; a wave's copy of the query fragments lives in its own region until then
    return (size_t)waves * ((size_t)NT * (D + kLdsPad) + (size_t)NT * 2) * sizeof(float);
}

int plan_launch(const tt_hip_ctx *ctx, int kind, int n_seq, int n_q_heads, int n_kv_heads, int head_dim, int rows,
                long long total_keys, int min_keys, int max_keys, LaunchPlan *plan, int kv_bits, bool small_tiles_ok) {
    if (n_kv_heads <= 0 || n_q_heads <= 0 || n_q_heads % n_kv_heads != 0) return TT_HIP_ERR_SHAPE;
    if (head_dim != 64 && head_dim != 128 && head_dim != 256) return TT_HIP_ERR_SHAPE;
    if (rows <= 0 || n_seq <= 0) return TT_HIP_ERR_INVALID_ARGUMENT;
    const int group = n_q_heads / n_kv_heads;
    LaunchPlan p{};
    if (kind == 1) {  // prefill: 32 tokens of one q head per tile
        p.nt = 32;
        p.gh = 1;
    } else {
        // GQA-packed rows: all q heads of a KV head (times the tile's tokens) share one pass over K/V.
        p.gh = packed_heads(group);
        p.nt = (rows * p.gh <= 16) ? 16 : 32;
        // Tiles of 16 rows although the rows would fill tiles of 32, while the launch reads little: the 32-row
        // kernel's fixed costs (one workgroup per CU, 32 rows x D floats per wavefront merged through LDS and left as
        // the partial result) then outweigh reading the cache once per tile of 16.  "Little" is counted in keys walked
        // by tiles of 16 over the whole launch, keys x tiles of 16 x KV heads (figures for 2 KV heads of 256, fp16):
        //  * A few verify rows (up to four tiles of 16 per KV head, whose reads all come from HBM): 4 rows at 8k keys
        //    16.4 -> 13.8 us, at 2k keys 13.5 -> 9.8, 4 sequences x 4 rows at 4k keys 19.5 -> 16.7, 8 rows at 8k keys
        //    18.6 -> 16.0; at 36k keys 24.1 against 24.3, at 64k keys 32.6 against 35.5 the other way.  Over quantised
        //    pages the 32-row tile is dearer still (4 rows at 64k keys over 8 bits 28.6 -> 24.6 us).
        //  * A short chunk behind a short context (more tiles, which re-read the same keys from L2), as long as the
        //    tiles are one round of workgroups: 32 rows from position 0 11.0 -> 6.5 us, 128 rows behind 1024 keys
        //    18.7 -> 15.0, 256 rows behind 1024 keys 22.8 -> 17.4; 128 rows behind 3072 keys 26.4 against 29.2 the
        //    other way, and 512 rows from position 0 were 17.0 against 19.7.
        // With 8 KV heads of 128 the same counts hold per KV head four times earlier (4 sequences x 16 rows at 4k keys:
        // 22.2 us in tiles of 32, 27.2 in tiles of 16; 8 rows at 8k keys 15.1 against 13.9), with 4 of 64 twice.
        if (small_tiles_ok && p.nt == 32 && p.gh <= 16) {
            const long long tiles16 = (rows + 16 / p.gh - 1) / (16 / p.gh);
            const long long launch_tiles16 = tiles16 * n_kv_heads * (group / p.gh);  // per sequence
            long long limit;  // of keys x tiles of 16 over the launch (the rows' own keys included)
            if (tiles16 <= 4) limit = kv_bits == 16 ? 144 * 1024 : 288 * 1024;
            else if (launch_tiles16 * n_seq <= ctx->n_cus) limit = kv_bits == 16 ? 320 * 1024 : 384 * 1024;
            else limit = 0;
            if (total_keys * launch_tiles16 <= limit) p.nt = 16;
        }
    }
    p.tt = p.nt / p.gh;
    p.hsubs = group / p.gh;
    p.tok_tiles = (rows + p.tt - 1) / p.tt;
    p.n_tiles = n_kv_heads * p.hsubs * p.tok_tiles;
    p.waves = 4;
    const int min_split = 32 * p.waves;  // one key block per wave
    // Workgroup slots of the chip: the 16-row kernel fits two workgroups per CU, the 32-row one.
    p.slots_per_cu = p.nt == 16 ? 2 : 1;
    const long long slots = (long long)ctx->n_cus * p.slots_per_cu;
    int split_len;
    if (ctx->split_override > 0) {
        split_len = ((ctx->split_override + 31) / 32) * 32;
    } else if (kind == 1) {
        split_len = ((max_keys + 31) / 32) * 32;  // prefill tiles are plentiful: no split
    } else if (min_keys == max_keys) {
        // Equal lengths: give every (sequence, tile) the same whole number of splits so that the
        // launch is exactly one round of at most n_cus workgroups -- a 257th workgroup would wait
        // for a CU and double the kernel's time.
        const long long pairs = (long long)n_seq * p.n_tiles;
        long long per_pair = ctx->n_cus / pairs;
        // Two rounds, side by side on a CU, where a workgroup's loads are few bytes and its walk is long (131k keys over 8 bits
        // with 16/4 heads of 64 23.4 -> 18.0 us, over 4 bits with 32/8 heads of 128 43.0 -> 35.6; with 16/2 of 256 27.4 -> 30.1).
        // Twice the partial results have to be worth it, which is a walk the longer the more rows and dims they have (before the
        // line / at it: 16 rows of 64, 920 keys a workgroup 12.8 -> 13.0 us, 1080 15.2 -> 13.0; 16 of 128 or 32 of 64, 860 keys
        // 14.9 -> 15.8, 1300 19.0 -> 16.2; 32 of 128, 1400 keys 26.3 -> 28.3, 1730 39.2 -> 30.3), and where there was one
        // workgroup a tile, and no combine, a longer one still (1613 keys 21.0 -> 27.0, 3416 25.9 -> 29.2, 8486 87 -> 61).
        const long long walk = per_pair <= 1 ? 4096 : p.nt * head_dim <= 1024 ? 1024 : p.nt * head_dim <= 2048 ? 1280 : 1536;
        if (head_dim * kv_bits <= 512 && pairs <= ctx->n_cus && max_keys >= walk * per_pair) per_pair = 2 * ctx->n_cus / pairs;
        if (per_pair < 1) per_pair = 1;
        split_len = (int)((max_keys + per_pair - 1) / per_pair);
        split_len = ((split_len + min_split - 1) / min_split) * min_split;
    } else {
        // Ragged lengths: about two workgroups per slot evens out the unequal last splits.
        const long long target_wgs = 2 * slots;
        const long long key_work = total_keys * p.n_tiles;
        long long per_wg = (key_work + target_wgs - 1) / target_wgs;
        // ... and at most 256 splits for the longest sequence: the grid is (splits of the longest, tiles,
        // sequences), and one long sequence beside many short ones would otherwise launch a grid of
        // workgroups that find nothing to do.
        if (per_wg < (max_keys + 255) / 256) per_wg = (max_keys + 255) / 256;
        split_len = (int)(((per_wg + min_split - 1) / min_split) * min_split);
    }
    // Up to 384 keys: one split, whose workgroup writes the final rows itself -- a wavefront's three blocks cost less
    // than the second launch (one decode row at 128 keys 8.6 -> 6.3 us a step, at 256 keys 8.7 -> 7.4; at 512 keys
    // 10.3 against 8.7 the other way).
    if (ctx->split_override <= 0 && kind == 0 && max_keys <= 384) split_len = ((max_keys + 31) / 32) * 32;
    if (split_len < 32) split_len = 32;
    p.split_len = split_len;
    p.n_splits_max = max_keys > 0 ? (max_keys + split_len - 1) / split_len : 1;
    if (p.n_splits_max < 1) p.n_splits_max = 1;
    p.workgroups = (long long)p.n_splits_max * p.n_tiles * n_seq;
    p.xcd_grid = false;
    p.lds_bytes = lds_bytes_for(head_dim, p.nt, p.waves);
    *plan = p;
    return TT_HIP_OK;
}

template <int D, int NT>
static int launch_combine_one(tt_hip_ctx *ctx, const LaunchPlan &plan, int n_seq, const SplitKArgs &args) {
    // Many tiles with few splits each: from 64 of its workgroups on (8 sequences' decode rows, 4 sequences' verify
    // rows; a verify pass of 8 x 4 rows at 65k keys 174.5 -> 170.1 us a step, 8 sequences x 8 rows at 4k keys 36.9 ->
    // 30.0 us; with 32 workgroups -- 4 sequences' decode rows -- the other kernel is ahead, 13.1 against 14.3 us).
    // (a turn's places are offsets of 32 bits)
    const bool near = (unsigned long long)plan.n_tiles * NT * D * sizeof(float) * kCombineRowsSplits <= 0xffffffffull;
    if (near && plan.n_splits_max <= 2 * kCombineRowsSplits && (long long)plan.n_tiles * n_seq * (NT / 4) >= 64) {
        dim3 cgrid((unsigned)(NT / 4), (unsigned)plan.n_tiles, (unsigned)n_seq);
        hipLaunchKernelGGL((attn_combine_rows_kernel<D, NT>), cgrid, dim3(256), 0, ctx->stream, args);
    } else {
        // (a workgroup per row that a tile can have and 64 dims of it: tiles of 16 with 8 rows in use launch no idle half)
        const int tile_rows = args.hot.rows < plan.tt ? args.hot.rows : plan.tt;
        dim3 cgrid((unsigned)(tile_rows * plan.gh * (D / 64)), (unsigned)plan.n_tiles, (unsigned)n_seq);
        hipLaunchKernelGGL((attn_combine_kernel<D, NT>), cgrid, dim3(256), 0, ctx->stream, args);
    }
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? TT_HIP_OK : hip_fail(ctx, e, "attn_combine_kernel launch");
}

template <int D, int NT, int WAVES, int BITS, int KEEP = 0, int STREAM = 0>
static int launch_one(tt_hip_ctx *ctx, const LaunchPlan &plan, int n_seq, const SplitKArgs &args) {
    auto kernel = attn_splitk_kernel<D, NT, WAVES, BITS, KEEP, STREAM>;  // its LDS limit was raised when the context was created
    dim3 grid((unsigned)plan.n_splits_max, (unsigned)plan.n_tiles, (unsigned)n_seq);
    if (plan.packed_splits > 0) grid = dim3((unsigned)plan.packed_splits, (unsigned)plan.n_tiles);
    if (plan.xcd_grid) grid = dim3((unsigned)(((long long)plan.n_splits_max * plan.n_tiles + 7) / 8 * 8), 1u, (unsigned)n_seq);
    launch_profiled(ctx, kernel, grid, dim3(WAVES * 64), (unsigned)(plan.lds_bytes + keep_list_bytes(KEEP, WAVES)), args);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(ctx, e, "attn_splitk_kernel launch");
    if (plan.n_splits_max > 1 && !ctx->pass_only) return launch_combine_one<D, NT>(ctx, plan, n_seq, args);
    return TT_HIP_OK;
}


// Every instantiation's dynamic LDS limit (a compile-time constant of the kernel), set once per device when a
// context is created on it: no launch has to configure anything, so none is refused inside a graph capture
// and nothing is remembered outside the context.
template <int D, int NT, int BITS, int KEEP>
static hipError_t configure_one() {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(attn_splitk_kernel<D, NT, 4, BITS, KEEP, 0>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)(lds_bytes_for(D, NT, 4) + keep_list_bytes(KEEP, 4)));
    if constexpr (D == 256 && NT == 32 && BITS == 16 && KEEP == 0) {
        if (e == hipSuccess)
            e = hipFuncSetAttribute(reinterpret_cast<const void *>(attn_splitk_kernel<D, NT, 4, BITS, KEEP, 2>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes_for(D, NT, 4));
    }
    if constexpr (KEEP < 2) {  // (a chunk's per-query selections come with many token tiles: never streamed)
        if (e == hipSuccess)
            e = hipFuncSetAttribute(reinterpret_cast<const void *>(attn_splitk_kernel<D, NT, 4, BITS, KEEP, 1>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes_for(D, NT, 4));
    }
    return e;
}
template <int D, int NT>
static hipError_t configure_tile() {
    hipError_t e = hipSuccess;
#define TT_CFG(BB, KK) \
    if (e == hipSuccess) e = configure_one<D, NT, BB, KK>();
    TT_CFG(16, 0) TT_CFG(8, 0) TT_CFG(4, 0)
    TT_CFG(16, 1) TT_CFG(8, 1) TT_CFG(4, 1)
    TT_CFG(16, 2) TT_CFG(8, 2) TT_CFG(4, 2)
    if constexpr (D != 256) { TT_CFG(16, 3) }  // (heads of 256: by key always)
    TT_CFG(8, 3) TT_CFG(4, 3)
    if constexpr (NT == 32) { TT_CFG(16, 4) }
    if constexpr (lists_fetch_by_key(D, 16)) { TT_CFG(16, 5) }
#undef TT_CFG
    return e;
}
int configure_splitk_kernels(tt_hip_ctx *ctx) {
    hipError_t e = configure_tile<256, 16>();
    if (e == hipSuccess) e = configure_tile<256, 32>();
    if (e == hipSuccess) e = configure_tile<128, 16>();
    if (e == hipSuccess) e = configure_tile<128, 32>();
    if (e == hipSuccess) e = configure_tile<64, 16>();
    if (e == hipSuccess) e = configure_tile<64, 32>();
    return e == hipSuccess ? TT_HIP_OK : hip_fail(ctx, e, "hipFuncSetAttribute(split-K max dynamic LDS)");
}

// The combine pass on its own: for partials written by another kernel in this kernel's layout.
int launch_combine(tt_hip_ctx *ctx, const LaunchPlan &plan, int head_dim, int n_seq, const SplitKArgs &args) {
    if (plan.n_tiles > 65535 || n_seq > 65535) return TT_HIP_ERR_SHAPE;
#define TT_CASE(DD, NN) \
    if (head_dim == DD && plan.nt == NN) return launch_combine_one<DD, NN>(ctx, plan, n_seq, args);
    TT_CASE(256, 16)
    TT_CASE(256, 32)
    TT_CASE(128, 16)
    TT_CASE(128, 32)
    TT_CASE(64, 16)
    TT_CASE(64, 32)
#undef TT_CASE
    return TT_HIP_ERR_SHAPE;
}

int launch_splitk(tt_hip_ctx *ctx, const LaunchPlan &plan, int head_dim, int n_seq, const SplitKArgs &args, int kv_bits) {
    if (n_seq > kMaxSeqPerLaunch || plan.waves != 4) return TT_HIP_ERR_INVALID_ARGUMENT;
    if (plan.n_tiles > 65535 || n_seq > 65535) return TT_HIP_ERR_SHAPE;
#define TT_CASE(DD, NN)                                                                              \
    if (head_dim == DD && plan.nt == NN) {                                                           \
        if constexpr (NN == 32) {                                                                    \
            if (args.plan_blocks && args.plan_groups) return launch_one<DD, NN, 4, 16, 4>(ctx, plan, n_seq, args); \
        }                                                                                            \
        if constexpr (lists_fetch_by_key(DD, 16)) {                                                  \
            if (args.plan_blocks && args.plan_by_key) return launch_one<DD, NN, 4, 16, 5>(ctx, plan, n_seq, args); \
        }                                                                                            \
        if (args.plan_blocks) {                                                                      \
            if constexpr (DD != 256) {                                                               \
                if (kv_bits == 16) return launch_one<DD, NN, 4, 16, 3>(ctx, plan, n_seq, args);      \
            }                                                                                        \
            if (kv_bits == 8) return launch_one<DD, NN, 4, 8, 3>(ctx, plan, n_seq, args);            \
            if (kv_bits == 4) return launch_one<DD, NN, 4, 4, 3>(ctx, plan, n_seq, args);            \
        }                                                                                            \
        if (args.keep && args.keep_row_stride > 0) {                                                 \
            if (kv_bits == 16) return launch_one<DD, NN, 4, 16, 2>(ctx, plan, n_seq, args);          \
            if (kv_bits == 8) return launch_one<DD, NN, 4, 8, 2>(ctx, plan, n_seq, args);            \
            if (kv_bits == 4) return launch_one<DD, NN, 4, 4, 2>(ctx, plan, n_seq, args);            \
        }                                                                                            \
        if (args.keep && plan.stream) {                                                              \
            if (kv_bits == 16) return launch_one<DD, NN, 4, 16, 1, 1>(ctx, plan, n_seq, args);       \
            if (kv_bits == 8) return launch_one<DD, NN, 4, 8, 1, 1>(ctx, plan, n_seq, args);         \
            if (kv_bits == 4) return launch_one<DD, NN, 4, 4, 1, 1>(ctx, plan, n_seq, args);         \
        }                                                                                            \
        if (args.keep) {                                                                             \
            if (kv_bits == 16) return launch_one<DD, NN, 4, 16, 1>(ctx, plan, n_seq, args);          \
            if (kv_bits == 8) return launch_one<DD, NN, 4, 8, 1>(ctx, plan, n_seq, args);            \
            if (kv_bits == 4) return launch_one<DD, NN, 4, 4, 1>(ctx, plan, n_seq, args);            \
        }                                                                                            \
        if (plan.stream) {                                                                           \
            if constexpr (DD == 256 && NN == 32) {                                                   \
                if (kv_bits == 16 && plan.paired) return launch_one<DD, NN, 4, 16, 0, 2>(ctx, plan, n_seq, args); \
            }                                                                                        \
            if (kv_bits == 16) return launch_one<DD, NN, 4, 16, 0, 1>(ctx, plan, n_seq, args);       \
            if (kv_bits == 8) return launch_one<DD, NN, 4, 8, 0, 1>(ctx, plan, n_seq, args);         \
            if (kv_bits == 4) return launch_one<DD, NN, 4, 4, 0, 1>(ctx, plan, n_seq, args);         \
        }                                                                                            \
        if (kv_bits == 16) return launch_one<DD, NN, 4, 16>(ctx, plan, n_seq, args);                 \
        if (kv_bits == 8) return launch_one<DD, NN, 4, 8>(ctx, plan, n_seq, args);                   \
        if (kv_bits == 4) return launch_one<DD, NN, 4, 4>(ctx, plan, n_seq, args);                   \
    }
    TT_CASE(256, 16)
    TT_CASE(256, 32)
    TT_CASE(128, 16)
    TT_CASE(128, 32)
    TT_CASE(64, 16)
    TT_CASE(64, 32)
#undef TT_CASE
    return TT_HIP_ERR_SHAPE;
}

}  // namespace tt
