// The projection behind the gate: y[t] = W x[t] with W stored as affine levels (4 or 8 bits, one
// bf16 scale and one bf16 bias per group of 64 columns), the runner's o_proj.
//
// Reference: RealForwardRunner.encodeAffineProjection
// (sources/TinyTitan/Runtime/Inference/RealForwardRunner+PrefillProjection.swift:53-66) as called for
// family .o (+PrefillAttention.swift:424-436) and the decode / batched-decode GEMVs behind it
// (DequantInt4GEMV.encode / encodeTwoRows, sources/TinyTitan/Kernels/Quant/DequantInt4GEMV.swift:72-143;
// kernels dequant_int4_gemv_simd / dequant_int4_gemv2_simd, sources/TinyTitanCore/Metal/Quant/dequant_int4.metal:101-280;
// CPU form tinytitan_int4_affine_gemv / tinytitan_int8_affine_gemv, sources/TinyTitanKernelsC).
// Arithmetic, as there: per row and group  scale * sum(level * x) + bias * sum(x)  in fp32, the row
// summed over its groups in fp32 and rounded to fp16 once.
//
// Three kernels by token count: a dot-product GEMV (1 to 4 tokens), tiles on the matrix cores (5 to 512), a GEMM over
// half weights (513 and more).
#include <cstdint>

#include "internal.h"
#include "wave_ops.h"

namespace tt {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef unsigned u4v __attribute__((ext_vector_type(4)));

constexpr int kProjGroup = 64;      // Quantization.groupSize

struct ProjArgs {
    const uint8_t *weights;
    const uint16_t *scales, *biases;
    const _Float16 *x;
    _Float16 *y;
    long long x_stride, y_stride;
    int rows, columns, tokens;
    int pass_tiles, pass_rows;  // > 0: the grid is one-dimensional, passes over the rows (affine_tile_kernel)
};

// Eight bytes -> eight halves holding 0..255 exactly: byte b under exponent byte 0x64 is 1024 + b.
__device__ __forceinline__ h8 levels_of_bytes(unsigned w0, unsigned w1) {
    const unsigned e = 0x64646464u;
    const u4v v = {__builtin_amdgcn_perm(e, w0, 0x04010400u), __builtin_amdgcn_perm(e, w0, 0x04030402u),
                   __builtin_amdgcn_perm(e, w1, 0x04010400u), __builtin_amdgcn_perm(e, w1, 0x04030402u)};
    return __builtin_bit_cast(h8, v) - (h8)(_Float16)1024;
}
// Eight nibbles of one dword in element order (element 2 k in the low nibble of byte k).
__device__ __forceinline__ h8 levels_of_nibbles(unsigned w) {
    const unsigned lo = w & 0x0f0f0f0fu, hi = (w >> 4) & 0x0f0f0f0fu, e = 0x64006400u;
    const u4v v = {__builtin_amdgcn_perm(hi, lo, 0x0c040c00u) | e, __builtin_amdgcn_perm(hi, lo, 0x0c050c01u) | e,
                   __builtin_amdgcn_perm(hi, lo, 0x0c060c02u) | e, __builtin_amdgcn_perm(hi, lo, 0x0c070c03u) | e};
    return __builtin_bit_cast(h8, v) - (h8)(_Float16)1024;
}

__device__ __forceinline__ float bf16_value(uint16_t bits) { return __builtin_bit_cast(float, (unsigned)bits << 16); }

// A lane's half group of levels: BITS * 4 bytes.  The reference only promises 2-byte alignment of a
// weight tensor inside its file (DequantInt4GEMV.swift:87-92); ALIGNED = false reads it that way.
template <int BITS, bool ALIGNED>
__device__ __forceinline__ void load_levels(unsigned (&w)[BITS], const uint8_t *src) {
    if constexpr (ALIGNED) {
#pragma unroll
        for (int i = 0; i < BITS / 4; ++i) {
            const u4v v = reinterpret_cast<const u4v *>(src)[i];
            w[4 * i] = v[0];
            w[4 * i + 1] = v[1];
            w[4 * i + 2] = v[2];
            w[4 * i + 3] = v[3];
        }
    } else {
        const uint16_t *p = reinterpret_cast<const uint16_t *>(src);
#pragma unroll
        for (int i = 0; i < BITS; ++i) w[i] = (unsigned)p[2 * i] | ((unsigned)p[2 * i + 1] << 16);
    }
}

// N consecutive bf16 values of a row, two to a register (the even group in the low half); past the row's
// end the last value again.
template <int N>
__device__ __forceinline__ void load_params(unsigned (&dst)[N / 2], const uint16_t *row, int first, int groups, bool vector) {
    if (vector) {
        if constexpr (N == 8) {
            const u4v v = *reinterpret_cast<const u4v *>(row + first);
            dst[0] = v[0];
            dst[1] = v[1];
            dst[2] = v[2];
            dst[3] = v[3];
        } else if constexpr (N == 4) {
            typedef unsigned u2v __attribute__((ext_vector_type(2)));
            const u2v v = *reinterpret_cast<const u2v *>(row + first);
            dst[0] = v[0];
            dst[1] = v[1];
        } else {
            static_assert(N == 2, "8, 4 or 2 values");
            dst[0] = *reinterpret_cast<const unsigned *>(row + first);
        }
    } else {
#pragma unroll
        for (int i = 0; i < N / 2; ++i)
            dst[i] = (unsigned)row[min(first + 2 * i, groups - 1)] | ((unsigned)row[min(first + 2 * i + 1, groups - 1)] << 16);
    }
}

typedef float f4v __attribute__((ext_vector_type(4)));
typedef unsigned u2v __attribute__((ext_vector_type(2)));

// ---------------------------------------------------------------------------
// 5 to 512 tokens (a draft's rows of several sequences, a decode batch, the default prefill chunk): tiles of 16 MT tokens x
// 16 NR weight rows.  A workgroup's eight wavefronts split the columns, a wavefront's groups in order; per group
// v_mfma_f32_16x16x32_f16 twice with A = x (16 tokens x 32 columns) and B = the levels, so that a lane's accumulators are
// four tokens of ONE row and the group's scale and bias are one value per lane, and twice against a constant for sum(x)
// in the same layout: acc += scale * dot + bias * sum(x).  The wavefronts' partial tiles are added through LDS in
// wavefront order: a token's bits depend neither on the tile's form nor on its neighbours.
//
// What bounds it is how its rows get into a CU.  Fragments straight from global memory put 16 lanes -- one token or row
// each, strides of whole lines -- on the same 16 bytes of 16 lines, which the vector cache serves a line at a time: 16 tokens
// (2048 x 4096, 4 bits) took 7.9 us a launch that way, and 6.0 with token strides 16 bytes off a multiple of a line.
// So x and the levels go to LDS by LDS-direct loads in whole lines, their 16-byte pieces permuted by row on the way so
// that the fragment reads hit every bank.
// A 4-bit level left where it lies in a half is a subnormal number; a multiplication makes it level / 512 (exact; nine
// instructions for eight levels, whose pairs (k, k + 4) x follows by a permute), biases are taken by 512 less as well and
// the tile's sums times 512 at the end.  (The matrix cores themselves lose low bits of subnormal halves: 95.5 % of the outputs
// bit-equal to the oracle instead of 99.85.  Levels in the mantissa of 16.0, with a sum that starts from -16 sum(x), cost an
// instruction less, but are rounded at up to three times their size, and an infinite x is a NaN in them.)
// The rest is bytes per CU, 16 MT x 8 KiB of x + 16 NR x 2.25 KiB of levels, at 35-40 KB/us.  us a launch, before (tiles of
// 32 x 32, x through registers and private patches of LDS) -> now:
//   2048 x 4096, 4 bits:   5 tokens 6.2 -> 4.7, 16: 9.7 -> 4.8, 32: 9.8 -> 5.0, 64: 9.9 -> 7.0, 128: 10.1 -> 8.7,
//                          256: 18.1 -> 14.7, 512: 29.5 -> 26.1
//   2048 x 4096, 8 bits:   32: 10.8 -> 5.3, 128: 10.9 -> 9.3, 512: 33.0 -> 27.7
//   2048 x 6144, 4 bits:   16: 13.7 -> 6.3, 128: 14.6 -> 11.0;  512 x 2048, 4 bits: 5: 4.8 -> 3.5, 128: 7.2 -> 3.8
// ---------------------------------------------------------------------------
constexpr int kTileWaves = 8;  // wavefronts that share a row's groups
// A wavefront's part of LDS: x [token tile][group][16 tokens][128 B], then levels [16 NR rows][SPAN groups].
constexpr int tile_x_bytes(int mt, int span) { return mt * span * 16 * 2 * kProjGroup; }
constexpr int tile_w_bytes(int bits, bool aligned, int nr, int span) { return aligned ? nr * 16 * span * 8 * bits : 0; }
constexpr int tile_lds_bytes(int bits, bool aligned, int mt, int nr, int span, int ring) {
    const int sums = kTileWaves * 16 * mt * (16 * nr + 4) * 4;  // the partial tiles take the rows' place
    const int staged = kTileWaves * ring * (tile_x_bytes(mt, span) + tile_w_bytes(bits, aligned, nr, span));
    return sums > staged ? sums : staged;
}

// Four registers of one 16-byte piece per lane group of 16 lanes -> register r of lane group k holds word k of lane group
// r's piece.
__device__ __forceinline__ void transpose_quarters(unsigned (&v)[4]) {
    auto swap32 = [](unsigned &a, unsigned &b) {
        const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        a = r[0];
        b = r[1];
    };
    auto swap16 = [](unsigned &a, unsigned &b) {
        const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        a = r[0];
        b = r[1];
    };
    swap32(v[0], v[2]);
    swap32(v[1], v[3]);
    swap16(v[0], v[1]);
    swap16(v[2], v[3]);
}

// N copies of 16 bytes a lane, global -> LDS, the i-th to lds_addr + 1024 i + 16 lane.  (An instruction's offset counts for both places, so the
// i-th source comes 1024 i below itself.)  In assembly: the compiler, seeing a copy into LDS, guards every later LDS read with a wait for
// all of them.  m0 is the compiler's (naming it as a clobber is not honoured): saved and put back.
template <int N>
__device__ __forceinline__ void copies_to_lds(const char *const (&src)[N], unsigned lds_addr) {
    static_assert(N >= 2 && N <= 4, "two to four copies");
    lds_addr = (unsigned)__builtin_amdgcn_readfirstlane((int)lds_addr);
    unsigned saved_m0;
    if constexpr (N == 2)
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off\n\tglobal_load_lds_dwordx4 %3, off offset:1024\n\t"
                     "s_mov_b32 m0, %0"
                     : "=&s"(saved_m0)
                     : "s"(lds_addr), "v"(src[0]), "v"(src[1])
                     : "memory");
    else if constexpr (N == 3)
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off\n\tglobal_load_lds_dwordx4 %3, off offset:1024\n\t"
                     "global_load_lds_dwordx4 %4, off offset:2048\n\ts_mov_b32 m0, %0"
                     : "=&s"(saved_m0)
                     : "s"(lds_addr), "v"(src[0]), "v"(src[1]), "v"(src[2])
                     : "memory");
    else
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, off\n\tglobal_load_lds_dwordx4 %3, off offset:1024\n\t"
                     "global_load_lds_dwordx4 %4, off offset:2048\n\tglobal_load_lds_dwordx4 %5, off offset:3072\n\ts_mov_b32 m0, %0"
                     : "=&s"(saved_m0)
                     : "s"(lds_addr), "v"(src[0]), "v"(src[1]), "v"(src[2]), "v"(src[3])
                     : "memory");
}

// RING = 2: a wavefront's next span is on its way into a second place while this one is worked on.
template <int BITS, bool ALIGNED, int MT, int NR, int SPAN, int RING>
__global__ __launch_bounds__(kTileWaves * 64) void affine_tile_kernel(const ProjArgs a) {
    static_assert(RING == 1 || ALIGNED, "levels that come through registers are waited for where they are asked for");
    constexpr int kTokens = 16 * MT, kRows = 16 * NR, kPitch = kRows + 4;
    constexpr int kXBytes = tile_x_bytes(MT, SPAN), kWaveBytes = kXBytes + tile_w_bytes(BITS, ALIGNED, NR, SPAN);
    constexpr int kRowPitch = SPAN * 8 * BITS, kRowPieces = kRowPitch / 16, kCopyRows = 64 / kRowPieces;  // of the levels in LDS
    constexpr int kSwizzle = kRowPieces < 8 ? kRowPieces - 1 : 7;
    extern __shared__ __attribute__((aligned(16))) unsigned char tile_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int n = lane & 15, kq = lane >> 4;
    int row_tile = blockIdx.x, token_tile = blockIdx.y;
    if (a.pass_tiles > 0) {
        // A pass is `pass_tiles` token tiles over all rows; an XCD takes every eighth row tile, with all of a pass's token
        // tiles one after the other.
        const int at = (int)(blockIdx.x >> 3), pass = at / (a.pass_tiles * a.pass_rows), in_pass = at - pass * (a.pass_tiles * a.pass_rows);
        token_tile = pass * a.pass_tiles + in_pass % a.pass_tiles;
        row_tile = 8 * (in_pass / a.pass_tiles) + (int)(blockIdx.x & 7);
        if (row_tile * kRows >= a.rows || token_tile * kTokens >= a.tokens) return;  // the whole workgroup: padding of the grid
    }
    const int row0 = row_tile * kRows, token0 = token_tile * kTokens;
    const int groups = a.columns / kProjGroup;
    int per_wave = (groups + kTileWaves - 1) / kTileWaves;
    if (groups >= 4 * kTileWaves) per_wave = (per_wave + 3) / 4 * 4;
    const int g_begin = min(groups, wave * per_wave), g_end = min(groups, g_begin + per_wave);
    const size_t row_bytes = (size_t)a.columns * BITS / 8;

    // copies: lane -> 16 bytes of token lane / 8 (+ 8): piece (lane % 8) ^ (lane / 8) of a group's 128 bytes
    const _Float16 *x_src[2 * MT];
#pragma unroll
    for (int c = 0; c < 2 * MT; ++c)
        x_src[c] = a.x + (long long)min(token0 + 8 * c + (lane >> 3), a.tokens - 1) * a.x_stride + 8 * ((lane & 7) ^ (lane >> 3));
    unsigned char *const wave_lds = tile_lds + wave * (RING * kWaveBytes);
    const unsigned lds_base = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)tile_lds, wave_lds_at = lds_base + wave * (RING * kWaveBytes);
    const uint8_t *w_src[NR];
    size_t p_at[NR];
#pragma unroll
    for (int nr = 0; nr < NR; ++nr) {
        const int row = min(row0 + 16 * nr + n, a.rows - 1);
        w_src[nr] = a.weights + (size_t)row * row_bytes;
        p_at[nr] = (size_t)row * groups;
    }
    // A row's next four scales (or biases) in one load where every such run is aligned, in pairs where those are (1024
    // columns, whose 16 groups are two a wavefront: 300 tokens over 8 bits 22.3 -> 15.4 us, over 4 bits 16.4 -> 10.8).
    const bool by_fours = groups % 4 == 0 && per_wave % 4 == 0 && (uintptr_t)a.scales % 8 == 0 && (uintptr_t)a.biases % 8 == 0;
    const bool by_twos = groups % 2 == 0 && per_wave % 2 == 0 && (uintptr_t)a.scales % 4 == 0 && (uintptr_t)a.biases % 4 == 0;
    auto next_params = [&](unsigned (&dst)[2], const uint16_t *row, int g0) {
        if (by_fours || !by_twos) return load_params<4>(dst, row, g0, groups, by_fours);
#pragma unroll
        for (int i = 0; i < 2; ++i) dst[i] = *reinterpret_cast<const unsigned *>(row + min(g0 + 2 * i, groups - 2));
    };
    const f4v zero = {0.f, 0.f, 0.f, 0.f};
    f4v acc[MT][NR];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nr = 0; nr < NR; ++nr) acc[mt][nr] = zero;
    const h8 ones = (h8)(_Float16)1;
    const h8 to_levels = {0x1p15f16, 0x1p15f16, 0x1p11f16, 0x1p11f16, 0x1p15f16, 0x1p15f16, 0x1p11f16, 0x1p11f16};
    constexpr float kBiasUnit = BITS == 4 ? 0x1p-9f : 1.0f, kSumUnit = BITS == 4 ? 0x1p9f : 1.0f;

    // Tiles of 32 x 32 and two places: in assembly (4 bits, 2048 x 4096, 400 tokens 27.3 -> 25.8 us: not in front of every LDS read of the
    // span a wait).  The others, where that wait costs nothing, by the builtin, which takes fewer instructions (16 tokens 5.10 against 5.18).
    constexpr bool kAssembly = RING == 2 || (MT == 2 && NR == 2);
    auto copies = [&](const auto &src, unsigned to) {  // the i-th to `to` + 1024 i + 16 lane
        constexpr int N = sizeof(src) / sizeof(src[0]);
        if constexpr (kAssembly) {
            const char *below[N];
#pragma unroll
            for (int c = 0; c < N; ++c) below[c] = src[c] - 1024 * c;
            copies_to_lds<N>(below, to);
        } else {
#pragma unroll
            for (int c = 0; c < N; ++c)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src[c],
                                                 (__attribute__((address_space(3))) void *)(tile_lds + (to - lds_base) + 1024 * c), 16, 0, 0);
        }
    };
    auto copy_span = [&](int gs, int place) {  // groups gs .. gs + SPAN - 1
        const unsigned x_at = wave_lds_at + place * kWaveBytes;
#pragma unroll
        for (int gi = 0; gi < SPAN; ++gi) {
            if (gs + gi >= g_end) break;
            const char *src[2 * MT];
#pragma unroll
            for (int c = 0; c < 2 * MT; ++c) src[c] = reinterpret_cast<const char *>(x_src[c] + kProjGroup * (gs + gi));
            copies(src, x_at + gi * (2048 * MT));
        }
        if constexpr (ALIGNED) {
            constexpr int kCopies = kRows / kCopyRows, kRun = kCopies < 4 ? kCopies : 4;
#pragma unroll
            for (int c0 = 0; c0 < kCopies; c0 += kRun) {
                const char *src[kRun];
#pragma unroll
                for (int c = 0; c < kRun; ++c) {
                    const int local = kCopyRows * (c0 + c) + lane / kRowPieces, row = min(row0 + local, a.rows - 1);
                    const unsigned at = min((unsigned)gs * (8 * BITS) + 16 * ((lane % kRowPieces) ^ (local & kSwizzle)), (unsigned)row_bytes - 16);
                    src[c] = reinterpret_cast<const char *>(a.weights + (size_t)row * row_bytes + at);
                }
                copies(src, x_at + kXBytes + 1024 * c0);
            }
        }
    };
    unsigned scales[NR][2], biases[NR][2], next_scales[NR][2], next_biases[NR][2];
    auto ask_params = [&](unsigned (&sc)[NR][2], unsigned (&bi)[NR][2], int g0) {  // of groups g0 .. g0 + 3
#pragma unroll
        for (int nr = 0; nr < NR; ++nr) {
            next_params(sc[nr], a.scales + p_at[nr], g0);
            next_params(bi[nr], a.biases + p_at[nr], g0);
        }
    };
    auto take_params = [&] {  // (touched here: waited for where they are used, they would be behind the next span's copies)
#pragma unroll
        for (int nr = 0; nr < NR; ++nr)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                asm volatile("" : "+v"(next_scales[nr][i]), "+v"(next_biases[nr][i]));
                scales[nr][i] = next_scales[nr][i];
                biases[nr][i] = next_biases[nr][i];
            }
    };
    int place = 0;
    if (RING == 2 && g_begin < g_end) {
        ask_params(next_scales, next_biases, g_begin);
        copy_span(g_begin, 0);
    }
    for (int g0 = g_begin; g0 < g_end; g0 += 4) {
#pragma unroll
        for (int sub = 0; sub < 4; sub += SPAN) {
            if (g0 + sub >= g_end) break;
            const int gs = g0 + sub;
            unsigned w[NR][SPAN * BITS / 2];
            if constexpr (RING == 2) {
                asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // this span is here, the last one's fragments have been read
                if (sub == 0) take_params();
                if (gs + SPAN < g_end) {
                    if (sub + SPAN == 4) ask_params(next_scales, next_biases, g0 + 4);
                    copy_span(gs + SPAN, place ^ 1);
                }
                __builtin_amdgcn_sched_barrier(0);
            } else {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the last span's fragments have been read
                copy_span(gs, 0);
                if (sub == 0) ask_params(scales, biases, g0);
                if constexpr (!ALIGNED) {
#pragma unroll
                    for (int nr = 0; nr < NR; ++nr)
#pragma unroll
                        for (int j = 0; j < SPAN * BITS / 8; ++j) {
                            unsigned v[4];
                            if constexpr (BITS == 4) load_levels<4, false>(v, w_src[nr] + (size_t)min(gs + 2 * j + (kq >> 1), groups - 1) * 32 + 16 * (kq & 1));
                            else load_levels<4, false>(v, w_src[nr] + (size_t)min(gs + j, groups - 1) * 64 + 16 * kq);
#pragma unroll
                            for (int i = 0; i < 4; ++i) w[nr][4 * j + i] = v[i];
                        }
                }
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the wavefront's own copies: no barrier
            }
            __builtin_amdgcn_wave_barrier();
            const unsigned char *const x_lds = wave_lds + place * kWaveBytes, *const w_lds = x_lds + kXBytes;
            if constexpr (RING == 2) place ^= 1;
#pragma unroll
            for (int nr = 0; nr < NR; ++nr)
#pragma unroll
                for (int j = 0; j < SPAN * BITS / 8; ++j) {
                    unsigned v[4] = {w[nr][4 * j], w[nr][4 * j + 1], w[nr][4 * j + 2], w[nr][4 * j + 3]};
                    if constexpr (ALIGNED) {
                        const u4v r = *reinterpret_cast<const u4v *>(w_lds + (16 * nr + n) * kRowPitch + (((4 * j + kq) ^ (n & kSwizzle)) << 4));
#pragma unroll
                        for (int i = 0; i < 4; ++i) v[i] = r[i];
                    }
                    if constexpr (BITS == 4) transpose_quarters(v);
#pragma unroll
                    for (int i = 0; i < 4; ++i) w[nr][4 * j + i] = v[i];
                }
#pragma unroll
            for (int gi = 0; gi < SPAN; ++gi) {
                if (gs + gi >= g_end) break;  // the whole wavefront
                const int g4 = sub + gi;
                h8 xf[MT][2];
                f4v xsum[MT];
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        const int piece = BITS == 4 ? 4 * i + kq : 2 * kq + i;
                        const h8 v = *reinterpret_cast<const h8 *>(x_lds + gi * (2048 * MT) + (16 * mt + n) * 128 + ((piece ^ (n & 7)) << 4));
                        if constexpr (BITS == 4) xf[mt][i] = h8{v[0], v[4], v[1], v[5], v[2], v[6], v[3], v[7]};
                        else xf[mt][i] = v;
                    }
                    xsum[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[mt][0], ones, zero, 0, 0, 0);
                    xsum[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[mt][1], ones, xsum[mt], 0, 0, 0);
                }
#pragma unroll
                for (int nr = 0; nr < NR; ++nr) {
                    const unsigned sp = scales[nr][g4 / 2], bp = biases[nr][g4 / 2];
                    const float bias = __builtin_bit_cast(float, (g4 & 1) ? (bp & 0xffff0000u) : (bp << 16)) * kBiasUnit;
                    const float scale = __builtin_bit_cast(float, (g4 & 1) ? (sp & 0xffff0000u) : (sp << 16));
                    h8 levels[2];
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        if constexpr (BITS == 4) {
                            const unsigned v = w[nr][2 * gi + i], u = v >> 8;
                            const u4v low = {v & 0x000f000fu, v & 0x00f000f0u, u & 0x000f000fu, u & 0x00f000f0u};  // level / 2^24, level / 2^20
                            levels[i] = __builtin_bit_cast(h8, low) * to_levels;
                        } else {
                            levels[i] = levels_of_bytes(w[nr][4 * gi + 2 * i], w[nr][4 * gi + 2 * i + 1]);
                        }
                    }
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) {
                        f4v dot = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[mt][0], levels[0], zero, 0, 0, 0);
                        dot = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[mt][1], levels[1], dot, 0, 0, 0);
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc[mt][nr][j] = fmaf(bias, xsum[mt][j], fmaf(scale, dot[j], acc[mt][nr][j]));
                    }
                }
            }
        }
    }
    __syncthreads();
    float *const sums = reinterpret_cast<float *>(tile_lds);  // [wavefront][token][kPitch]
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nr = 0; nr < NR; ++nr)
#pragma unroll
            for (int j = 0; j < 4; ++j) sums[(wave * kTokens + 16 * mt + 4 * kq + j) * kPitch + 16 * nr + n] = acc[mt][nr][j];
    __syncthreads();
    for (int at = threadIdx.x; at < kTokens * kRows; at += kTileWaves * 64) {
        const int t = at / kRows, r = at % kRows;
        float sum = 0.0f;
#pragma unroll
        for (int w2 = 0; w2 < kTileWaves; ++w2) sum += sums[(w2 * kTokens + t) * kPitch + r];
        if (token0 + t < a.tokens && row0 + r < a.rows) a.y[(long long)(token0 + t) * a.y_stride + row0 + r] = (_Float16)(sum * kSumUnit);
    }
}

// The smallest tile whose workgroups find a CU each -- a wider tile reads less per output but takes longer: 32 tokens
// 5.1 us in tiles of 16 x 16 (256 workgroups), 7.0 in 16 x 32, 8.7 in 32 x 32; 64 tokens 7.4 / 7.0 / 8.7; 128 tokens
// 12.2 / 12.3 / 8.8 (9.8 with two groups instead of four in LDS at a time, which lets two workgroups share a CU) -- and
// beyond that 32 x 32, two workgroups to a CU (256 tokens 14.7 us, with four groups in LDS 16.1), or over 8 bits, whose levels weigh twice as much, 32 x 64 (256 tokens 13.2 against 16.0 us).
template <int BITS, bool ALIGNED>
void launch_tile(tt_hip_ctx *ctx, const ProjArgs &a) {
    auto tiles = [&](int mt, int nr) { return (long long)((a.rows + 16 * nr - 1) / (16 * nr)) * ((a.tokens + 16 * mt - 1) / (16 * mt)); };
    auto launch = [&](auto kernel, int mt, int nr, int lds) {
        dim3 grid((unsigned)((a.rows + 16 * nr - 1) / (16 * nr)), (unsigned)((a.tokens + 16 * mt - 1) / (16 * mt)));
        // Many rows: their weights outlast no L2 from one token tile to the next, so the token tiles of some rows follow each
        // other on one XCD, eight at a time (the x of 256 tokens and the weights in flight still fit its L2).  4 bits, 4096
        // columns: 8192 rows x 256 tokens 50.8 -> 47.9 us, 512 98.3 -> 93.2, 16,384 x 128 52.2 -> 47.9, 512 195.1 -> 181.5; 8
        // bits 16,384 x 256 111.7 -> 106.8.  Fewer rows stay in the L2s as they are: 2048 x 64 7.15 against 7.36, 512 25.8 against 26.4.
        ProjArgs b = a;
        if (a.rows >= 8192 && grid.y > 1) {
            const unsigned pass = grid.y < 8 ? grid.y : 8, passes = (grid.y + pass - 1) / pass, per_xcd = (grid.x + 7) / 8;
            if ((unsigned long long)per_xcd * 8 * pass * passes <= 1u << 22) {  // (a grid of 2^31 threads)
                b.pass_tiles = (int)pass;
                b.pass_rows = (int)per_xcd;
                grid = dim3(per_xcd * 8 * pass * passes);
            }
        }
        launch_profiled(ctx, kernel, grid, dim3(kTileWaves * 64), (unsigned)lds, b);
    };
    // 8 bits: two places in LDS, the next span on its way beside the arithmetic (5 / 32 / 64 / 128 tokens 5.62 / 6.15 / 9.1 / 10.2 -> 5.08 / 5.28 / 7.6 / 9.3
    // us).  4 bits, half the bytes and twice the widening, are the arithmetic anyway: 16 / 64 / 128 tokens 5.1 / 7.25 / 9.0 in one place, 5.2 / 7.3 / 9.3 in two.
    constexpr int kRing = ALIGNED && BITS == 8 ? 2 : 1, kSpan = kRing == 2 ? 2 : 4, kLarge = BITS == 4 ? 4 : ALIGNED ? 1 : 2;
#define TT_TILE(mt, nr, span, ring) launch(affine_tile_kernel<BITS, ALIGNED, mt, nr, span, ring>, mt, nr, tile_lds_bytes(BITS, ALIGNED, mt, nr, span, ring))
    if (tiles(1, 1) <= ctx->n_cus) TT_TILE(1, 1, kSpan, kRing);
    else if (tiles(1, 2) <= ctx->n_cus) TT_TILE(1, 2, kSpan, kRing);
    else if (tiles(2, 2) <= ctx->n_cus) TT_TILE(2, 2, kLarge, kRing);
    else if constexpr (BITS == 4) TT_TILE(2, 2, 2, 1);
    else TT_TILE(2, 4, 2, 1);
#undef TT_TILE
}

// ---------------------------------------------------------------------------
// Up to four tokens (a decode row, the two-row and four-row verify passes): the matrix cores have little to amortise, and
// tiles of 16 rows would leave half of the chip idle at 2048 rows.
// Here a workgroup owns 8 weight rows and its eight wavefronts take the columns 512 at a time in
// turn: a lane takes 8 consecutive columns of each row (one dword of nibbles or two of bytes,
// coalesced; they lie in one group), widens them to fp16 levels and contracts them with its 8 x
// values by v_dot2_f32_f16 (products exact, fp32 accumulation), then
// acc += scale * dot + bias * sum(x) as above.  All of a wavefront's loads for a 512-column chunk
// are independent, so they are in flight together; the lanes' 8 x TOK sums are added by moves between lanes that pack two values
// into one at every step (wave_sums; a chain of six DPP moves for each was most of a launch of four tokens: 2048 x 4096 over 4
// bits, launch to launch, one token 3.60 -> 3.33 us, two 4.23 -> 3.72, four 5.62 -> 4.59, where five take the tiles above 4.91),
// wavefronts through LDS in a fixed order.  256 workgroups at 2048 rows.
// ---------------------------------------------------------------------------
constexpr int kGemvWaves = 8, kGemvRows = 8, kGemvMaxTokens = 4;

__device__ __forceinline__ float dot8(h8 a, h8 b) {
    float d = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const h2 ai = {a[2 * i], a[2 * i + 1]}, bi = {b[2 * i], b[2 * i + 1]};
        d = __builtin_amdgcn_fdot2(ai, bi, d, false);
    }
    return d;
}

template <int BITS, int TOK, bool ALIGNED>
__global__ __launch_bounds__(kGemvWaves * 64) void affine_gemv_kernel(const ProjArgs a) {
    __shared__ float partial[kGemvWaves][kGemvRows * TOK];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row0 = blockIdx.x * kGemvRows;
    const int groups = a.columns / kProjGroup;
    const int chunks = (a.columns + 511) / 512;
    const unsigned row_bytes = (unsigned)a.columns / (8 / BITS);
    const unsigned last = (unsigned)(a.rows - 1 - row0);  // the workgroup's last row there is
    // A workgroup's addresses are one of its first row and what a row adds; eight rows' scales lie within 32 bits of it.  (Each row's
    // from the front of the matrix was products of 64 bits for all three, 60 to 80 scalar instructions in front of the first load:
    // one token over 4 bits, 2048 x 4096 3.12 -> 2.94 us, 16,384 x 2048 6.05 -> 5.42, over 8 bits 7.46 -> 6.28.)
    const uint8_t *const block_weights = a.weights + (unsigned long long)(unsigned)row0 * row_bytes;
    const uint16_t *const block_scales = a.scales + (unsigned long long)(unsigned)row0 * (unsigned)groups;
    const uint16_t *const block_biases = a.biases + (unsigned long long)(unsigned)row0 * (unsigned)groups;
    const h8 ones = (h8)(_Float16)1;
    float acc[kGemvRows][TOK];
#pragma unroll
    for (int r = 0; r < kGemvRows; ++r)
#pragma unroll
        for (int t = 0; t < TOK; ++t) acc[r][t] = 0.0f;
#pragma unroll 1  // one straight-line body: every load of a chunk is issued before the first use
    for (int chunk = wave; chunk < chunks; chunk += kGemvWaves) {
        const int wanted = 512 * chunk + 8 * lane;
        const bool inside = wanted < a.columns;
        const int column = inside ? wanted : 0;  // a valid address always
        h8 xv[TOK];
        float xsum[TOK];
#pragma unroll
        for (int t = 0; t < TOK; ++t) {  // loaded from a valid address; zeroed below where the lane is past the row
            xv[t] = *reinterpret_cast<const h8 *>(a.x + (long long)t * a.x_stride + column);
        }
        const unsigned g = (unsigned)column / kProjGroup;
        unsigned w[kGemvRows][BITS / 4];
        uint16_t scale_bits[kGemvRows], bias_bits[kGemvRows];
#pragma unroll
        for (int r = 0; r < kGemvRows; ++r) {
            const unsigned row = min((unsigned)r, last);
            const uint8_t *src = block_weights + (unsigned long long)row * row_bytes + (unsigned)column / (8 / BITS);
#pragma unroll
            for (int i = 0; i < BITS / 4; ++i) {
                if constexpr (ALIGNED) w[r][i] = reinterpret_cast<const unsigned *>(src)[i];
                else w[r][i] = (unsigned)reinterpret_cast<const uint16_t *>(src)[2 * i] |
                               ((unsigned)reinterpret_cast<const uint16_t *>(src)[2 * i + 1] << 16);
            }
            const unsigned at = (row * (unsigned)groups + g) * (unsigned)sizeof(uint16_t);
            scale_bits[r] = *reinterpret_cast<const uint16_t *>(reinterpret_cast<const char *>(block_scales) + at);
            bias_bits[r] = *reinterpret_cast<const uint16_t *>(reinterpret_cast<const char *>(block_biases) + at);
        }
        // Every load above is issued before anything below: left to itself the scheduler sinks each
        // load to its use to save registers and the wavefront then waits for them one by one.
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < TOK; ++t) {
            xv[t] = inside ? xv[t] : (h8)(_Float16)0;
            xsum[t] = dot8(xv[t], ones);
        }
#pragma unroll
        for (int r = 0; r < kGemvRows; ++r) {
            h8 levels;
            if constexpr (BITS == 4) levels = levels_of_nibbles(w[r][0]);
            else levels = levels_of_bytes(w[r][0], w[r][1]);
            const float scale = bf16_value(scale_bits[r]), bias = bf16_value(bias_bits[r]);
#pragma unroll
            for (int t = 0; t < TOK; ++t) acc[r][t] = fmaf(bias, xsum[t], fmaf(scale, dot8(xv[t], levels), acc[r][t]));
        }
    }
    float v[kGemvRows * TOK];
#pragma unroll
    for (int i = 0; i < kGemvRows * TOK; ++i) v[i] = acc[i / TOK][i % TOK];
    int mine;  // the sum that this lane ends up with
    const float sum = wave_sums<kGemvRows * TOK>(v, lane, mine);
    if (mine >= 0) partial[wave][mine] = sum;
    __syncthreads();
    if (threadIdx.x < kGemvRows * TOK) {
        const int r = threadIdx.x / TOK, t = threadIdx.x % TOK;
        float v = 0.0f;
#pragma unroll
        for (int w2 = 0; w2 < kGemvWaves; ++w2) v += partial[w2][threadIdx.x];
        if (row0 + r < a.rows) a.y[(long long)t * a.y_stride + row0 + r] = (_Float16)v;
    }
}

template <int BITS, bool ALIGNED>
void launch_gemv(tt_hip_ctx *ctx, const ProjArgs &a) {
    const dim3 grid((unsigned)((a.rows + kGemvRows - 1) / kGemvRows));
    const dim3 block(kGemvWaves * 64);
    switch (a.tokens) {
        case 1: launch_profiled(ctx, affine_gemv_kernel<BITS, 1, ALIGNED>, grid, block, 0u, a); break;
        case 2: launch_profiled(ctx, affine_gemv_kernel<BITS, 2, ALIGNED>, grid, block, 0u, a); break;
        case 3: launch_profiled(ctx, affine_gemv_kernel<BITS, 3, ALIGNED>, grid, block, 0u, a); break;
        default: launch_profiled(ctx, affine_gemv_kernel<BITS, 4, ALIGNED>, grid, block, 0u, a); break;
    }
}

// ---------------------------------------------------------------------------
// A prefill chunk (513 tokens and more): a GEMM.  The reference's tensor-operation path for these
// (MPPPrefillInt4QMM, kernel sources/TinyTitanCore/Metal/TensorCore/tensorops.metal:60-125, taken from 32
// tokens on) dequantises a weight tile to HALF -- weightTile = half(fma(float(q), scale, bias)) --
// and multiplies half tiles into an fp32 accumulator; this kernel does the same: a level becomes
// the fp16 number level * scale + bias (one fused fp16 multiply-add: the exact value rounded once,
// where the reference rounds through fp32 first; scale and bias are bf16 values, exact in fp16
// within its range), and x . w accumulates in fp32 on the matrix cores.
//
// A workgroup of 4 wavefronts owns 128 tokens x 128 weight rows; a wavefront 32 of the rows against all
// 128 tokens, four 32x32 accumulators (no row's levels are widened twice).  Per group of 64 columns:
// the x tile (128 x 64) goes straight into LDS (one copy per workgroup, a ring of three, a group's copies issued two groups ahead) and is
// read as A fragments; a wavefront's levels go there too, whole lines of its rows for four groups of 4 bits (two of 8) at a time, a span
// ahead, and a lane reads its row's from there, widens and scales them in registers into the B fragments of a group, and 16 MFMAs per
// group follow (4 contraction steps x 4 token tiles), each step's A fragments read while the step before it
// multiplies (tiles of fewer tokens: two steps before); the rows' scales and biases come from a block in LDS, converted to fp16 once.  One barrier per
// group.  The output tile leaves through LDS, [token][row], as 16-byte stores.
// Before, x went through registers and a lane read its own 16 bytes of levels, 32 rows an instruction, with the MFMAs of a step in runs of three behind
// one run of widening.  2048 x 4096 over 4 bits, 513 / 777 / 1,024 / 1,500 / 2,048 / 4,096 tokens 26.9 / 27.6 / 29.0 / 36.9 / 43.6 / 74.4 -> 23.7 / 25.3 /
// 27.0 / 33.3 / 40.2 / 70.6 us (0.97 PFLOP/s), over 8 bits 29.3 / 29.7 / 30.9 / 39.2 / 46.5 / 76.7 -> 24.2 / 26.3 / 28.4 / 34.7 / 41.7 / 74.4.  What is left, from
// builds without one thing (4,096 tokens; 1,024): MFMAs 21 us; 5, fragment reads 14; 3, widening 11; 5, copies 11; 3, the barrier 0; 0.
// ---------------------------------------------------------------------------
constexpr int kGemmTokens = 128, kGemmWaves = 4, kGemmRows = 32 * kGemmWaves;
// From here on the chunk is a GEMM: 24-27 us up to 1024 tokens, 33 beyond and 40 at 2048, where its grid fills the chip, against
// 26 us at 512 tokens for the tiles above, whose time goes on growing by 25 us per 512 tokens.
constexpr int kGemmMinTokens = 513;
constexpr int kGemmThreads = kGemmWaves * 64;
constexpr int kGemmRing = 3;           // groups of x in LDS: read, landed, on their way
constexpr int kGemmLevelBytes = 4096;  // a wavefront's levels in LDS: 32 rows x 128 bytes
constexpr int gemm_tile_bytes(int tokens) { return tokens * 2 * kProjGroup; }
// Groups whose scales and biases sit in LDS at a time: 64, over the parts that walk columns of their own; half as many where two workgroups share a CU.
constexpr int gemm_param_groups(int ks, bool rs) { return rs ? 64 : ks == 1 ? 32 : 64 / ks; }
// KS = parts the columns are split into inside a workgroup (1 or 2): KS x 4 wavefronts, part p's four take the
// groups [p x part_groups, (p + 1) x part_groups) with x tiles and a block of scales and biases of their own, and
// the parts' accumulators are added through LDS at the end, in a fixed order.  For chunks whose tiles number no
// more than the CUs: a workgroup's time is that of ONE wavefront's walk over the columns (44 us at 4096 columns,
// whatever the number of tiles); in two parts it is 39-40 us, and 48-51 us instead of 56-57 at 2048 tokens, where
// every CU has a workgroup.
// Its time goes with the tokens of its tile more than with its columns' parts (a third and fourth part of a tile of 64
// tokens: 31.3 us against 29.1 at 777 tokens, its registers halved), so a chunk that leaves CUs without a workgroup takes
// tiles of 64 or 96 (TOKENS).
constexpr int gemm_lds_bytes(int ks, bool rs, int tokens) {
    const int x = (rs ? 1 : ks) * kGemmRing * gemm_tile_bytes(tokens), rows = rs ? ks * kGemmRows : kGemmRows;
    return x + ks * kGemmWaves * kGemmLevelBytes + (rs ? 1 : ks) * gemm_param_groups(ks, rs) * rows * 4;
}
static_assert(gemm_lds_bytes(1, false, kGemmTokens) <= 80 * 1024, "two workgroups to a CU");

// vmcnt(n) only: leaves the LDS and export counters alone.
#define TT_WAIT_COPIES(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | (0x7 << 4) | (0xF << 8))

template <int BITS, bool ALIGNED, int KS, bool RS = false, int TOKENS = kGemmTokens>
__global__ __launch_bounds__(kGemmThreads * KS, 2) void affine_gemm_kernel(const ProjArgs a) {
    // RS (with KS = 2): the two parts split the ROWS instead of the columns -- a tile of 128 tokens x 256 rows, one x
    // tile for all eight wavefronts.
    constexpr int kThreads = kGemmThreads * KS, kPartParamGroups = gemm_param_groups(KS, RS);
    constexpr int kRows = RS ? kGemmRows * KS : kGemmRows;
    constexpr int kStageThreads = RS ? kThreads : kGemmThreads, kCopies = TOKENS * 8 / kStageThreads;  // x copies of a wavefront per group
    constexpr int TT = TOKENS / 32;  // 32-token tiles: accumulators of a wavefront
    static_assert(kGemmWaves * 64 * 16 * TT * (int)sizeof(float) <= gemm_lds_bytes(2, false, TOKENS), "the parts' accumulators meet in the store");
    // per part kGemmRing x tiles of TOKENS x 128 bytes, then per wavefront its levels, then per part [kPartParamGroups][kRows] (scale, bias)
    // pairs as fp16.  A token's (a row's) 16-byte pieces are permuted by its number, so that the fragment reads hit every bank.
    extern __shared__ __attribute__((aligned(16))) _Float16 lds_store[];
    const int part = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kGemmThreads);
    const int tid = threadIdx.x % kGemmThreads, lane = tid & 63, wave = tid >> 6;  // tid, wave: inside the part
    const int stage_tid = RS ? (int)threadIdx.x : tid;
    constexpr int kXBytes = kGemmRing * gemm_tile_bytes(TOKENS), kXParts = RS ? 1 : KS;
    char *const lds_bytes = reinterpret_cast<char *>(lds_store), *const x_tiles = lds_bytes + (RS ? 0 : part * kXBytes);
    char *const level_tile = lds_bytes + kXParts * kXBytes + (kGemmWaves * part + wave) * kGemmLevelBytes;
    unsigned *const params = reinterpret_cast<unsigned *>(lds_bytes + kXParts * kXBytes + KS * kGemmWaves * kGemmLevelBytes) + (RS ? 0 : part * kPartParamGroups * kRows);
    const int c = lane & 31, h = lane >> 5;
    // A wavefront owns 32 weight rows against all 128 tokens: every row's levels are widened by exactly one wavefront.
    // Workgroups are dealt to the 8 XCDs in turn, each with its own L2: the workgroups that share a token block
    // (its x rows are what they all read) get ids congruent modulo 8, i.e. one XCD.
    const int row_blocks = (a.rows + kRows - 1) / kRows;
    const int id = blockIdx.x;
    const int token_block = (id & 7) + 8 * (id / (8 * row_blocks));
    if (token_block * TOKENS >= a.tokens) return;  // the whole workgroup, before any barrier: padding of the grid
    const int token0 = token_block * TOKENS, row0 = ((id >> 3) % row_blocks) * kRows;
    const int groups = a.columns / kProjGroup;
    constexpr int kHalfGroupBytes = BITS * 4;
    // Levels are read kSpan groups at a time: a lane's 64 contiguous bytes of its row, so that a 128-byte line
    // is fetched once and used whole (16 bytes per group would touch the line again for each of its groups).
    constexpr int kSpan = BITS == 4 ? 4 : 2;
    // This part's groups: [first_group, first_group + part_groups), whole spans; below, g counts from first_group.
    constexpr int kColumnParts = RS ? 1 : KS;
    const int part_groups = (groups + kColumnParts * kSpan - 1) / (kColumnParts * kSpan) * kSpan, first_group = RS ? 0 : part * part_groups;
    const size_t row_bytes = (size_t)a.columns * BITS / 8;

    // x: a copy of a wavefront is eight tokens' 128 bytes of a group.
    const unsigned lds_base = (unsigned)(size_t)(__attribute__((address_space(3))) void *)lds_store;
    const unsigned x_lds = lds_base + (unsigned)(x_tiles - lds_bytes) + (unsigned)((stage_tid >> 6) * kCopies * 1024);
    const char *x_src[kCopies];
#pragma unroll
    for (int p = 0; p < kCopies; ++p) {
        const int local = 8 * ((stage_tid >> 6) * kCopies + p) + (lane >> 3);
        x_src[p] = reinterpret_cast<const char *>(a.x + (long long)min(token0 + local, a.tokens - 1) * a.x_stride) + 16 * ((lane & 7) ^ (lane >> 3)) - 1024 * p;
    }
    auto copy_x = [&](int g, unsigned slot) {  // slot: the tile's offset in the ring
        const int gc = min(first_group + g, groups - 1);  // past the end: the last group again, a valid address, unused
        const char *src[kCopies];
#pragma unroll
        for (int p = 0; p < kCopies; ++p) src[p] = x_src[p] + 2 * kProjGroup * gc;
        copies_to_lds<kCopies>(src, x_lds + slot);
    };
    const int param_at = (RS ? kGemmRows * part : 0) + 32 * wave + c;  // this lane's weight row inside the workgroup's tile
    // Levels: the 128 bytes of a span of the wavefront's 32 rows, a line each, in four copies of eight rows.  (Read by the lanes themselves, 16
    // bytes of 32 rows an instruction, they were 32 lines for every KiB, and a CU's path to memory takes two cycles a line whatever is wanted of it:
    // copies of 32, 64 and 128 bytes a row run at 34, 69 and 115 KB/us a CU.)
    const unsigned level_lds = lds_base + (unsigned)(level_tile - lds_bytes);
    const uint8_t *const w_row = a.weights + (size_t)min(row0 + param_at, a.rows - 1) * row_bytes;
    const char *w_src[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = (RS ? kGemmRows * part : 0) + 32 * wave + 8 * i + (lane >> 3);
        w_src[i] = reinterpret_cast<const char *>(a.weights + (size_t)min(row0 + row, a.rows - 1) * row_bytes) - 1024 * i;
    }
    auto copy_levels = [&](int first) {  // of groups [first, first + kSpan)
        const size_t at = min((size_t)(first_group + first) * (8 * BITS) + 16 * ((lane & 7) ^ (lane >> 3)), row_bytes - 16);
        const char *const src[4] = {w_src[0] + at, w_src[1] + at, w_src[2] + at, w_src[3] + at};
        copies_to_lds<4>(src, level_lds);
    };
    // Scales and biases of this workgroup's rows for groups [first, first + kPartParamGroups): a thread takes eight
    // consecutive groups of a row, 16 bytes of scales and 16 of biases, and eight threads a row's 128 bytes, so the
    // rows are read as whole lines (one value per thread and load made 64 loads of 2 bytes per thread, every lane on
    // a line of its own: 16 us of a 107 us launch at 4096 tokens).  Converted to fp16 and stored [group][row], so that
    // the lanes of a wavefront -- consecutive rows -- read consecutive words.
    constexpr int kRowThreads = kPartParamGroups / 8, kPassRows = kStageThreads / kRowThreads;
    static_assert(kPartParamGroups % 8 == 0 && kRows % kPassRows == 0, "eight groups a thread");
    const bool params_vector = (uintptr_t)a.scales % 16 == 0 && (uintptr_t)a.biases % 16 == 0 && groups % 8 == 0;
    auto stage_params = [&](int first) {
        const int k = 8 * (stage_tid % kRowThreads), g = first_group + first + k;
        // All of a thread's loads before its first store, and one question for all of them: asked row by row it was a branch around
        // every load, and the wavefront waited for each (2048 rows, 777 tokens: 1024 columns 12.1 -> 10.7 us, 2048 16.8 -> 15.9, 6144 40.4
        // -> 39.1; 4096 tokens over 4096 columns 71.7 -> 71.1).
        constexpr int kPasses = kRows / kPassRows;
        unsigned scale_bits[kPasses][4], bias_bits[kPasses][4];
        auto load = [&](int at_group, bool vector) {
#pragma unroll
            for (int i = 0; i < kPasses; ++i) {
                const size_t at = (size_t)min(row0 + stage_tid / kRowThreads + kPassRows * i, a.rows - 1) * groups;
                load_params<8>(scale_bits[i], a.scales + at, at_group, groups, vector);
                load_params<8>(bias_bits[i], a.biases + at, at_group, groups, vector);
            }
        };
        // (Eight groups that are all past the matrix's last are not read back.  Eight that reach over it, where a second part starts
        // between eights -- 24 groups: at the 12th -- are, in part, and are loaded one by one: 1536 columns, 777 tokens 14.2 us, where
        // the question row by row took 14.6.)
        if (params_vector && (g >= groups || g + 8 <= groups)) load(min(g, groups - 8), true);
        else load(g, false);
#pragma unroll
        for (int i = 0; i < kPasses; ++i) {
            const int local = stage_tid / kRowThreads + kPassRows * i;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const _Float16 scale = (_Float16)bf16_value((uint16_t)(scale_bits[i][j / 2] >> (16 * (j & 1))));
                const _Float16 bias = (_Float16)bf16_value((uint16_t)(bias_bits[i][j / 2] >> (16 * (j & 1))));
                params[(k + j) * kRows + local] = (unsigned)__builtin_bit_cast(uint16_t, scale) |
                                                      ((unsigned)__builtin_bit_cast(uint16_t, bias) << 16);
            }
        }
    };
    const f16v zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    f16v acc[TT];  // one per 32-token tile
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) acc[tt] = zero;

    unsigned w_now[kSpan][BITS], w_later[kSpan][BITS];  // (w_later: levels that are not aligned come by register, a span ahead)
    auto load_span = [&](unsigned (&w)[kSpan][BITS], int first) {
#pragma unroll
        for (int k = 0; k < kSpan; ++k) {
            const int g = min(first_group + first + k, groups - 1);  // past the end: the last group again, a valid address, unused
            load_levels<BITS, false>(w[k], w_row + (size_t)g * (2 * kHalfGroupBytes) + h * kHalfGroupBytes);
        }
    };
    auto read_span = [&]() {
#pragma unroll
        for (int k = 0; k < kSpan; ++k)
#pragma unroll
            for (int i = 0; i < BITS / 4; ++i) {
                const int piece = (BITS / 4) * (2 * k + h) + i;
                const u4v v = *reinterpret_cast<const u4v *>(level_tile + c * 128 + ((piece ^ (c & 7)) << 4));
                w_now[k][4 * i] = v[0];
                w_now[k][4 * i + 1] = v[1];
                w_now[k][4 * i + 2] = v[2];
                w_now[k][4 * i + 3] = v[3];
            }
    };
    if constexpr (ALIGNED) {
        copy_levels(0);
    } else {
        load_span(w_now, 0);
        load_span(w_later, kSpan);
    }
    copy_x(0, 0);
    copy_x(1, gemm_tile_bytes(TOKENS));
    stage_params(0);
    TT_WAIT_COPIES(0);
    __syncthreads();
    if constexpr (ALIGNED) {
        read_span();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (part_groups > kSpan) copy_levels(kSpan);
    }

    // B fragments of a group: its levels widened and scaled, bw[g % 2], four registers of two halves each.  They are made one group ahead, a
    // pair at a time behind the current group's MFMAs.
    unsigned bw[2][4][4];
    unsigned exponents = BITS == 4 ? 0x54006400u : 0x64646464u;  // (in a vector register: an instruction takes one scalar one)
    asm volatile("" : "+v"(exponents));
    auto widen_pair = [&](unsigned &dst, const unsigned (&w)[BITS], int t, int p, h2 scale, h2 bias) {  // columns 2 p, 2 p + 1 of a lane's eight
        unsigned v;
        h2 zero_level;
        if constexpr (BITS == 4) {  // byte p twice: the low nibble under the exponent of 1024, the high one, four places up, under that of 64
            v = (__builtin_amdgcn_perm(w[t], w[t], 0x0c000c00u + 0x00010001u * p) & 0x00f0000fu) | exponents;
            zero_level = h2{1024, 64};
        } else {
            v = __builtin_amdgcn_perm(exponents, w[2 * t + p / 2], p % 2 ? 0x04030402u : 0x04010400u);
            zero_level = h2{1024, 1024};
        }
        dst = __builtin_bit_cast(unsigned, __builtin_elementwise_fma(__builtin_bit_cast(h2, v) - zero_level, scale, bias));
    };
    // Past the matrix's last group the scale and the bias are zero: such a group's products add nothing, and the
    // loop over a span needs no exit in its middle.
    auto pair_of = [&](int g) { return first_group + g < groups ? params[(g % kPartParamGroups) * kRows + param_at] : 0u; };
    auto scale_of = [&](unsigned pair) { return (h2)__builtin_bit_cast(_Float16, (uint16_t)(pair & 0xffffu)); };
    auto bias_of = [&](unsigned pair) { return (h2)__builtin_bit_cast(_Float16, (uint16_t)(pair >> 16)); };
    {
        const unsigned pair = pair_of(0);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int p = 0; p < 4; ++p) widen_pair(bw[0][t][p], w_now[0], t, p, scale_of(pair), bias_of(pair));
    }
    // A fragments of contraction step t of a group: 32 tokens x 16 columns per token tile, af[t]; a step's
    // fragments are read from LDS kAhead steps before they multiply.
    constexpr int kAhead = TT >= 4 ? 1 : 2;
    h8 af[4][TT];
    const int fragment_at = c * 128 + (((4 * h) ^ (c & 7)) << 4);
    auto fragment = [&](unsigned slot, int t, int tt) { return *reinterpret_cast<const h8 *>(x_tiles + slot + (fragment_at ^ (t << 4)) + 4096 * tt); };
    // The ring's places: of the group in hand, of the next (landed at the barrier) and of the one whose copies go out now.
    unsigned here = 0, next = gemm_tile_bytes(TOKENS), ahead = 2 * gemm_tile_bytes(TOKENS);
#pragma unroll
    for (int t = 0; t < kAhead; ++t)
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) af[t][tt] = fragment(here, t, tt);

    for (int g0 = 0; g0 < part_groups; g0 += kSpan) {
        const bool more_spans = g0 + kSpan < part_groups, still_more = g0 + 2 * kSpan < part_groups;
#pragma unroll
        for (int k = 0; k < kSpan; ++k) {
            const int g = g0 + k;
            static_assert(kSpan % 2 == 0, "a group's fragments must not depend on the span");
            const unsigned pair_next = pair_of(g + 1);
            const h2 scale_next = scale_of(pair_next), bias_next = bias_of(pair_next);
            // The copies of this group: x of group g + 2 into the place that group g - 1 was read from (every wavefront is past that group's barrier), and in
            // a span's last group, when the next span's levels have gone to their registers, those of the span behind it.
            const bool more_x = g + 2 < part_groups;
            if (k == kSpan - 1 && more_spans) {
                if constexpr (ALIGNED) {
                    read_span();
                } else {
#pragma unroll
                    for (int i = 0; i < kSpan; ++i)
#pragma unroll
                        for (int j = 0; j < BITS; ++j) w_now[i][j] = w_later[i][j];
                }
            }
            const unsigned(&w_of_next)[BITS] = w_now[(k + 1) % kSpan];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if (t == 0 && more_x) copy_x(g + 2, ahead);
                const bool levels_out = k == kSpan - 1 && still_more;
                if (t == 1 && levels_out) {
                    if constexpr (ALIGNED) {
                        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (read_span's)
                        copy_levels(g0 + 2 * kSpan);
                    } else {
                        load_span(w_later, g0 + 2 * kSpan);
                    }
                }
                if (t == 4 - kAhead) {
                    // Everybody's rows of group g + 1 are in LDS from here on: of the copies only this group's may still be on their way.
                    if (ALIGNED && levels_out) TT_WAIT_COPIES(kCopies + 4);  // (a span behind the next: there is more x)
                    else if (more_x) TT_WAIT_COPIES(kCopies);
                    else TT_WAIT_COPIES(0);
                    __syncthreads();
                }
                const h8 b = __builtin_bit_cast(h8, u4v{bw[k & 1][t][0], bw[k & 1][t][1], bw[k & 1][t][2], bw[k & 1][t][3]});
#pragma unroll
                for (int tt = 0; tt < TT; ++tt) {
                    // One MFMA, one fragment read and a share of the next group's widening, in this order: the two wavefronts of a SIMD then have
                    // something else to issue between any two MFMAs.
                    acc[tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[t][tt], b, acc[tt], 0, 0, 0);
                    af[(t + kAhead) % 4][tt] = fragment(t + kAhead < 4 ? here : next, (t + kAhead) % 4, tt);
#pragma unroll
                    for (int p = tt * 4 / TT; p < (tt + 1) * 4 / TT; ++p) widen_pair(bw[(k + 1) & 1][t][p], w_of_next, t, p, scale_next, bias_next);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            const unsigned done = here;
            here = next;
            next = ahead;
            ahead = done;
            // The next block of scales and biases is first read one step before its first group is multiplied.
            if ((g + 2) % kPartParamGroups == 0 && g + 2 < part_groups) {  // the whole workgroup
                __syncthreads();                                       // everyone has read this block
                stage_params(g + 2);
                __syncthreads();
            }
        }
    }
    // The tile leaves through LDS: a lane holds 16 tokens of ONE row, 2 bytes of a token's output each; laid out
    // [token][row] in the space of the x tiles, a thread then writes 16 bytes -- eight rows of a token -- and 16
    // threads a token's 256 bytes (64 stores of 2 bytes per lane took 8 us of the launch at 4096 tokens).
    __syncthreads();  // nobody reads an x tile any more
    if constexpr (KS == 2 && !RS) {
        // part 1's accumulators join part 0's: [wavefront][value][lane] floats, every lane its own words
        float *const sums = reinterpret_cast<float *>(lds_store) + wave * 64 * 16 * TT + lane;
        if (part == 1) {
#pragma unroll
            for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                for (int j = 0; j < 16; ++j) sums[(16 * tt + j) * 64] = acc[tt][j];
        }
        __syncthreads();
        if (part == 0) {
#pragma unroll
            for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                for (int j = 0; j < 16; ++j) acc[tt][j] += sums[(16 * tt + j) * 64];
        }
        __syncthreads();  // the sums are read: the output tile may take their place
    }
    _Float16 *const out_tile = lds_store;
    constexpr int kOutPitch = kRows + 8;
    static_assert(TOKENS * kOutPitch * (int)sizeof(_Float16) <= gemm_lds_bytes(KS, RS, TOKENS), "the output tile takes the store's space");
    if (part == 0 || RS) {
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int j = 0; j < 16; ++j)
                out_tile[(32 * tt + 8 * (j / 4) + 4 * h + (j % 4)) * kOutPitch + param_at] = (_Float16)acc[tt][j];
    }
    __syncthreads();
    const bool y_vector = (uintptr_t)a.y % 16 == 0 && a.y_stride % 8 == 0;
    const int thread = threadIdx.x;
    constexpr int kPieces = kRows / 8;
#pragma unroll
    for (int i = 0; i < TOKENS * kPieces / kThreads; ++i) {
        const int at = thread + kThreads * i, local = at / kPieces, piece = at % kPieces;
        const int token = token0 + local, row = row0 + 8 * piece;
        if (token >= a.tokens || row >= a.rows) continue;
        const h8 v = *reinterpret_cast<const h8 *>(out_tile + local * kOutPitch + 8 * piece);
        _Float16 *dst = a.y + (long long)token * a.y_stride + row;
        if (y_vector && row + 8 <= a.rows) {
            *reinterpret_cast<h8 *>(dst) = v;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (row + e < a.rows) dst[e] = v[e];
        }
    }
}

// 80 to 160 KiB of LDS: above the 64 KiB a kernel gets without asking.
template <int BITS, bool ALIGNED, int KS, bool RS = false, int TOKENS = kGemmTokens>
int launch_gemm(tt_hip_ctx *ctx, const ProjArgs &a, dim3 grid) {
    auto kernel = affine_gemm_kernel<BITS, ALIGNED, KS, RS, TOKENS>;  // its LDS limit was raised when the context was created
    launch_profiled(ctx, kernel, grid, dim3(kGemmThreads * KS), (unsigned)gemm_lds_bytes(KS, RS, TOKENS), a);
    return TT_HIP_OK;
}

}  // namespace

// The MFMA kernels' dynamic LDS limits, set once per device when a context is created on it.
int configure_affine_kernels(tt_hip_ctx *ctx) {
    hipError_t e = hipSuccess;
#define TT_CFG(KERNEL, BYTES) \
    if (e == hipSuccess) e = hipFuncSetAttribute(reinterpret_cast<const void *>(KERNEL), hipFuncAttributeMaxDynamicSharedMemorySize, BYTES);
    TT_CFG((affine_gemm_kernel<4, true, 1>), gemm_lds_bytes(1, false, 128))
    TT_CFG((affine_gemm_kernel<4, false, 1>), gemm_lds_bytes(1, false, 128))
    TT_CFG((affine_gemm_kernel<8, true, 1>), gemm_lds_bytes(1, false, 128))
    TT_CFG((affine_gemm_kernel<8, false, 1>), gemm_lds_bytes(1, false, 128))
    TT_CFG((affine_gemm_kernel<4, true, 2>), gemm_lds_bytes(2, false, 128))
    TT_CFG((affine_gemm_kernel<4, false, 2>), gemm_lds_bytes(2, false, 128))
    TT_CFG((affine_gemm_kernel<8, true, 2>), gemm_lds_bytes(2, false, 128))
    TT_CFG((affine_gemm_kernel<8, false, 2>), gemm_lds_bytes(2, false, 128))
    TT_CFG((affine_gemm_kernel<4, true, 2, false, 64>), gemm_lds_bytes(2, false, 64))
    TT_CFG((affine_gemm_kernel<4, true, 2, false, 96>), gemm_lds_bytes(2, false, 96))
    TT_CFG((affine_gemm_kernel<4, false, 2, false, 64>), gemm_lds_bytes(2, false, 64))
    TT_CFG((affine_gemm_kernel<4, false, 2, false, 96>), gemm_lds_bytes(2, false, 96))
    TT_CFG((affine_gemm_kernel<8, true, 2, false, 64>), gemm_lds_bytes(2, false, 64))
    TT_CFG((affine_gemm_kernel<8, true, 2, false, 96>), gemm_lds_bytes(2, false, 96))
    TT_CFG((affine_gemm_kernel<8, false, 2, false, 64>), gemm_lds_bytes(2, false, 64))
    TT_CFG((affine_gemm_kernel<8, false, 2, false, 96>), gemm_lds_bytes(2, false, 96))
    TT_CFG((affine_gemm_kernel<4, true, 2, true>), gemm_lds_bytes(2, true, 128))
    TT_CFG((affine_gemm_kernel<4, false, 2, true>), gemm_lds_bytes(2, true, 128))
    TT_CFG((affine_gemm_kernel<8, true, 2, true>), gemm_lds_bytes(2, true, 128))
    TT_CFG((affine_gemm_kernel<8, false, 2, true>), gemm_lds_bytes(2, true, 128))
    TT_CFG((affine_tile_kernel<4, true, 1, 1, 4, 1>), tile_lds_bytes(4, true, 1, 1, 4, 1))
    TT_CFG((affine_tile_kernel<4, true, 1, 2, 4, 1>), tile_lds_bytes(4, true, 1, 2, 4, 1))
    TT_CFG((affine_tile_kernel<4, true, 2, 2, 4, 1>), tile_lds_bytes(4, true, 2, 2, 4, 1))
    TT_CFG((affine_tile_kernel<4, true, 2, 2, 2, 1>), tile_lds_bytes(4, true, 2, 2, 2, 1))
    TT_CFG((affine_tile_kernel<4, false, 1, 1, 4, 1>), tile_lds_bytes(4, false, 1, 1, 4, 1))
    TT_CFG((affine_tile_kernel<4, false, 1, 2, 4, 1>), tile_lds_bytes(4, false, 1, 2, 4, 1))
    TT_CFG((affine_tile_kernel<4, false, 2, 2, 4, 1>), tile_lds_bytes(4, false, 2, 2, 4, 1))
    TT_CFG((affine_tile_kernel<4, false, 2, 2, 2, 1>), tile_lds_bytes(4, false, 2, 2, 2, 1))
    TT_CFG((affine_tile_kernel<8, true, 1, 1, 2, 2>), tile_lds_bytes(8, true, 1, 1, 2, 2))
    TT_CFG((affine_tile_kernel<8, true, 1, 2, 2, 2>), tile_lds_bytes(8, true, 1, 2, 2, 2))
    TT_CFG((affine_tile_kernel<8, true, 2, 2, 1, 2>), tile_lds_bytes(8, true, 2, 2, 1, 2))
    TT_CFG((affine_tile_kernel<8, true, 2, 4, 2, 1>), tile_lds_bytes(8, true, 2, 4, 2, 1))
    TT_CFG((affine_tile_kernel<8, false, 1, 1, 4, 1>), tile_lds_bytes(8, false, 1, 1, 4, 1))
    TT_CFG((affine_tile_kernel<8, false, 1, 2, 4, 1>), tile_lds_bytes(8, false, 1, 2, 4, 1))
    TT_CFG((affine_tile_kernel<8, false, 2, 2, 2, 1>), tile_lds_bytes(8, false, 2, 2, 2, 1))
    TT_CFG((affine_tile_kernel<8, false, 2, 4, 2, 1>), tile_lds_bytes(8, false, 2, 4, 2, 1))
#undef TT_CFG
    return e == hipSuccess ? TT_HIP_OK : hip_fail(ctx, e, "hipFuncSetAttribute(o_proj max dynamic LDS)");
}

}  // namespace tt

using namespace tt;

extern "C" int tt_hip_affine_projection(tt_hip_ctx *ctx, int weight_bits, const void *weights, const uint16_t *scales_bf16,
                                        const uint16_t *biases_bf16, const tt_half *x, tt_half *y, int rows, int columns,
                                        int token_count, size_t x_stride_, size_t y_stride_) {
    if (!ctx || !weights || !scales_bf16 || !biases_bf16 || !x || !y) return TT_HIP_ERR_INVALID_ARGUMENT;
    if (rows <= 0 || columns <= 0 || token_count < 0) return TT_HIP_ERR_INVALID_ARGUMENT;
    if (weight_bits != 4 && weight_bits != 8) return TT_HIP_ERR_SHAPE;
    // Quantization.groupSize: the reference's precondition (DequantInt4GEMV.swift:84-86).
    if (columns % kProjGroup != 0) return TT_HIP_ERR_SHAPE;
    const long long x_stride = (long long)x_stride_, y_stride = (long long)y_stride_;
    if (x_stride < columns || y_stride < rows) return TT_HIP_ERR_SHAPE;
    // x rows are read 16 bytes at a time; weights at least 2-byte aligned, scales and biases are 16-bit values.
    if ((uintptr_t)x % 16 != 0 || x_stride % 8 != 0 || (uintptr_t)weights % 2 != 0 || (uintptr_t)y % 2 != 0 ||
        (uintptr_t)scales_bf16 % 2 != 0 || (uintptr_t)biases_bf16 % 2 != 0)
        return TT_HIP_ERR_SHAPE;
    if (token_count == 0) return TT_HIP_OK;
    BusyGuard guard(ctx);
    if (!guard.ok) return TT_HIP_ERR_BUSY;
    ProjArgs a{};
    a.weights = static_cast<const uint8_t *>(weights);
    a.scales = scales_bf16;
    a.biases = biases_bf16;
    a.x = reinterpret_cast<const _Float16 *>(x);
    a.y = reinterpret_cast<_Float16 *>(y);
    a.x_stride = x_stride;
    a.y_stride = y_stride;
    a.rows = rows;
    a.columns = columns;
    a.tokens = token_count;
    if (token_count > 32 * 65535) return TT_HIP_ERR_SHAPE;
    const bool aligned = (uintptr_t)weights % 16 == 0;
    if (token_count >= kGemmMinTokens) {
        const long long row_blocks = (rows + kGemmRows - 1) / kGemmRows, token_blocks = (token_count + kGemmTokens - 1) / kGemmTokens;
        const long long padded = (token_blocks + 7) / 8 * 8 * row_blocks;  // token blocks in eights: see the kernel's id mapping
        if (padded > 0x7fffffffLL) return TT_HIP_ERR_SHAPE;
        const dim3 tiles_grid((unsigned)padded);
        // Four forms of the kernel.  Tiles of 128 rows for no more than the CUs: the columns in two parts inside a
        // workgroup.  More than that: tiles of 256 rows, eight wavefronts, one workgroup per CU -- the x tile is then
        // fetched once for twice the rows, and what the card's power limit charges for is traffic (4096 tokens 94.5 ->
        // 87.7 us on one box, 92.7 -> 92.0 on another; 3072 tokens 82.1 -> 75.7; 8192 tokens 176 -> 167) -- unless their
        // last round of several would leave most of the chip idle (5120 tokens, 320 such tiles: 134.8 us against 125.4 with tiles
        // of 128 rows, two workgroups per CU).
        const long long wide_blocks = (rows + 2 * kGemmRows - 1) / (2 * kGemmRows), wide_tiles = token_blocks * wide_blocks;
        const long long last_round = wide_tiles % ctx->n_cus;
        const bool two_parts = columns / kProjGroup >= 16;
        const auto tiles = [&](int tokens) { return (token_count + tokens - 1) / tokens * row_blocks; };
        const auto grid_of = [&](int tokens) { return dim3((unsigned)(((token_count + tokens - 1) / tokens + 7) / 8 * 8 * row_blocks)); };
        int status;
        if (two_parts && tiles(64) <= ctx->n_cus) {
            // ... and with fewer tokens a tile while those tiles number no more than the CUs either: at 2048 rows x 4096 columns
            // tiles of 64 38.0 -> 28.7 us up to 1024 tokens (8-bit levels 41.8 -> 30.5; at 1024 columns 14.4 -> 11.5; at
            // 1100 tokens, a second workgroup on some CUs, 51.0 against 37.5 the other way), tiles of 96 41.3 -> 35.7 up to 1536.
            if (weight_bits == 4) status = aligned ? launch_gemm<4, true, 2, false, 64>(ctx, a, grid_of(64)) : launch_gemm<4, false, 2, false, 64>(ctx, a, grid_of(64));
            else status = aligned ? launch_gemm<8, true, 2, false, 64>(ctx, a, grid_of(64)) : launch_gemm<8, false, 2, false, 64>(ctx, a, grid_of(64));
        } else if (two_parts && tiles(96) <= ctx->n_cus) {
            if (weight_bits == 4) status = aligned ? launch_gemm<4, true, 2, false, 96>(ctx, a, grid_of(96)) : launch_gemm<4, false, 2, false, 96>(ctx, a, grid_of(96));
            else status = aligned ? launch_gemm<8, true, 2, false, 96>(ctx, a, grid_of(96)) : launch_gemm<8, false, 2, false, 96>(ctx, a, grid_of(96));
        } else if (two_parts && token_blocks * row_blocks <= ctx->n_cus) {
            if (weight_bits == 4) status = aligned ? launch_gemm<4, true, 2>(ctx, a, tiles_grid) : launch_gemm<4, false, 2>(ctx, a, tiles_grid);
            else status = aligned ? launch_gemm<8, true, 2>(ctx, a, tiles_grid) : launch_gemm<8, false, 2>(ctx, a, tiles_grid);
        } else if (wide_tiles <= ctx->n_cus || last_round == 0 || 10 * last_round > 6 * ctx->n_cus) {
            const dim3 wide_grid((unsigned)((token_blocks + 7) / 8 * 8 * wide_blocks));  // (padded <= 0x7fffffff holds for these too)
            if (weight_bits == 4) status = aligned ? launch_gemm<4, true, 2, true>(ctx, a, wide_grid) : launch_gemm<4, false, 2, true>(ctx, a, wide_grid);
            else status = aligned ? launch_gemm<8, true, 2, true>(ctx, a, wide_grid) : launch_gemm<8, false, 2, true>(ctx, a, wide_grid);
        } else {
            if (weight_bits == 4) status = aligned ? launch_gemm<4, true, 1>(ctx, a, tiles_grid) : launch_gemm<4, false, 1>(ctx, a, tiles_grid);
            else status = aligned ? launch_gemm<8, true, 1>(ctx, a, tiles_grid) : launch_gemm<8, false, 1>(ctx, a, tiles_grid);
        }
        if (status != TT_HIP_OK) return status;
    } else if (token_count <= kGemvMaxTokens) {
        // unaligned weights: a lane's dword sits at a 2-byte boundary
        const bool words = (uintptr_t)weights % 4 == 0;
        if (weight_bits == 4) {
            if (words) launch_gemv<4, true>(ctx, a);
            else launch_gemv<4, false>(ctx, a);
        } else {
            if (words) launch_gemv<8, true>(ctx, a);
            else launch_gemv<8, false>(ctx, a);
        }
    } else {
        // (aligned: rows of levels are then whole 16-byte pieces, too)
        if (weight_bits == 4) {
            if (aligned) launch_tile<4, true>(ctx, a);
            else launch_tile<4, false>(ctx, a);
        } else {
            if (aligned) launch_tile<8, true>(ctx, a);
            else launch_tile<8, false>(ctx, a);
        }
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? TT_HIP_OK : hip_fail(ctx, e, "affine projection launch");
}
