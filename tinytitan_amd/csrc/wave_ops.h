// Cross-lane reductions over the 2 (32-row tiles) or 4 (16-row tiles) lanes that share a query
// row, with gfx950's v_permlane32_swap / v_permlane16_swap: no lane-index register, no LDS trip.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

namespace tt {

// The output gate's factor, 1 / (1 + e^-x), rounded as the fp32 division rounds it: the hardware's reciprocal (one unit in the last
// place) and a Newton step, over a quarter of the denominator (exact) so that no reciprocal is subnormal; an infinite denominator
// is the fixup's.  Every fp16 gate gives the division's bits (of the factors below 2^-126, which round any fp16 value to zero, all
// but their last place): the bare reciprocal was off in 3,597 of them.  A pass of 4,096 rows of
// 16/2 heads of 256 (245 us) and one of 777 rows of 32/8 of 128 (97.4 us) take 0.8 and 0.3 % more than with the bare reciprocal, with a full division
// (a dozen instructions for every element of an output, 128 a lane in the chunk kernel) 1.6 and 1.0 %.
__device__ __forceinline__ float sigmoid(float x) {
    float scale = 0.25f;
    asm("" : "+s"(scale));  // (kept in a vector register it was the one too many in the chunk kernel of heads of 256, which then spilled)
    const float quarter = __builtin_fmaf(scale, __expf(-x), scale), r = __builtin_amdgcn_rcpf(quarter);
    return scale * __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-quarter, r, 1.0f), r, r), quarter, 1.0f);
}

// v_permlane32_swap(x, x): first result = lanes 0-31 of x in both halves, second = lanes 32-63.
__device__ __forceinline__ void halves_of(float x, float &lo, float &hi) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    lo = __builtin_bit_cast(float, (unsigned)r[0]);
    hi = __builtin_bit_cast(float, (unsigned)r[1]);
}
// v_permlane16_swap(x, x): first result = rows 0,0,2,2 of x (a row is 16 lanes), second = rows 1,1,3,3.
__device__ __forceinline__ void row_pairs_of(float x, float &even, float &odd) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    even = __builtin_bit_cast(float, (unsigned)r[0]);
    odd = __builtin_bit_cast(float, (unsigned)r[1]);
}

// Lanes l and l ^ 32.
__device__ __forceinline__ float max_across_halves(float x) {
    float lo, hi;
    halves_of(x, lo, hi);
    return fmaxf(lo, hi);
}
__device__ __forceinline__ float sum_across_halves(float x) {
    float lo, hi;
    halves_of(x, lo, hi);
    return lo + hi;
}
// Lanes l, l ^ 16, l ^ 32, l ^ 48.
__device__ __forceinline__ float max_across_quarters(float x) {
    float a, b;
    row_pairs_of(x, a, b);
    return max_across_halves(fmaxf(a, b));
}
__device__ __forceinline__ float sum_across_quarters(float x) {
    float a, b;
    row_pairs_of(x, a, b);
    return sum_across_halves(a + b);
}

// The largest value of the 64 lanes, in every lane, by data-parallel-primitive moves: within a row of 16 lanes by
// row_shr 1, 2, 4, 8, then lane 15 of every row into the row after it (row_bcast15) and lane 31 into the upper half
// (row_bcast31) -- a lane takes a step's value only where the move had a source -- then lane 63's.
__device__ __forceinline__ float wave_max_f32(float x, int lane) {
    const int in_row = lane & 15;
    auto moved = [](float v, auto ctrl) {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(ctrl)::value, 0xf, 0xf, false));
    };
    float t;
    t = moved(x, std::integral_constant<int, 0x111>{});
    if (in_row >= 1) x = fmaxf(x, t);
    t = moved(x, std::integral_constant<int, 0x112>{});
    if (in_row >= 2) x = fmaxf(x, t);
    t = moved(x, std::integral_constant<int, 0x114>{});
    if (in_row >= 4) x = fmaxf(x, t);
    t = moved(x, std::integral_constant<int, 0x118>{});
    if (in_row >= 8) x = fmaxf(x, t);
    t = moved(x, std::integral_constant<int, 0x142>{});
    if ((lane & 31) >= 16) x = fmaxf(x, t);
    t = moved(x, std::integral_constant<int, 0x143>{});
    if (lane >= 32) x = fmaxf(x, t);
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 63));
}

// The sum of the 64 lanes, in lane 63 (other lanes hold partial sums): row_shr 1, 2, 4, 8 inside the rows of 16, then
// row_bcast15 and row_bcast31; a lane whose move has no source adds zero.  Six vector instructions, no trip through LDS.
__device__ __forceinline__ float wave_sum_in_lane63(float x) {
    auto moved = [](float v, auto ctrl) {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(ctrl)::value, 0xf, 0xf, false));
    };
    x += moved(x, std::integral_constant<int, 0x111>{});
    x += moved(x, std::integral_constant<int, 0x112>{});
    x += moved(x, std::integral_constant<int, 0x114>{});
    x += moved(x, std::integral_constant<int, 0x118>{});
    x += moved(x, std::integral_constant<int, 0x142>{});
    x += moved(x, std::integral_constant<int, 0x143>{});
    return x;
}

// The sums of the 64 lanes of N <= 32 values, each value's in a lane of its own: `mine` is the value whose sum the lane gets, -1
// in the lanes that are left over.  Six steps, every one of which adds two lanes and, while there are several values, packs two
// of them into one register on the way -- by v_permlane32_swap, v_permlane16_swap, then by picks and DPP moves inside a
// row -- so that the work halves from step to step: 71 instructions for 32 values, where six a value are 192.  A value's
// additions are the same ones whatever N is.
template <int CTRL>
__device__ __forceinline__ float sums_moved(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
template <int N>
__device__ __forceinline__ float wave_sums(float (&v)[N], int lane, int &mine) {
    static_assert(N >= 1 && N <= 32, "a lane bit tells two values apart, and one is left for the last step");
    auto pairs = [&](int count, auto join) {  // the values 2 i and 2 i + 1 become value i; an odd last one stands for both
#pragma unroll
        for (int i = 0; i < N; ++i)
            if (2 * i < count) v[i] = join(v[2 * i], v[2 * i + 1 < count ? 2 * i + 1 : 2 * i]);
        return (count + 1) / 2;
    };
    // lanes l and l ^ 32, then l and l ^ 16: the lower ones keep a's sum, the upper ones b's
    int count = pairs(N, [](float a, float b) {
        const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
        return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
    });
    count = pairs(count, [](float a, float b) {
        const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
        return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
    });
    // inside a row of 16: row_ror:8, row_half_mirror, quad_perm [2,3,0,1]
    const auto step = [&](int bit, auto ctrl) {
        const bool upper = (lane & bit) != 0;
        if (count == 1) {
            v[0] += sums_moved<decltype(ctrl)::value>(v[0]);
            return;
        }
        count = pairs(count, [&](float a, float b) { return (upper ? b : a) + sums_moved<decltype(ctrl)::value>(upper ? a : b); });
    };
    step(8, std::integral_constant<int, 0x128>{});
    step(4, std::integral_constant<int, 0x141>{});
    step(2, std::integral_constant<int, 0x4E>{});
    v[0] += sums_moved<0xB1>(v[0]);
    mine = (lane >> 5) + ((lane >> 4) & 1) * 2 + ((lane >> 3) & 1) * 4;
    int unused = 7;
    if constexpr (N > 8) {
        mine += ((lane >> 2) & 1) * 8;
        unused = 3;
    }
    if constexpr (N > 16) {
        mine += ((lane >> 1) & 1) * 16;
        unused = 1;
    }
    if (mine >= N || (lane & unused)) mine = -1;
    return v[0];
}

// Sums, minima and maxima over aligned groups of 8, 16 or 32 lanes, every lane of a group getting the result, by DPP
// moves: quad_perm [1,0,3,2] and [2,3,0,1] inside a quad; then row_half_mirror (lane i <-> 7 - i: the other quad,
// whose lanes all hold that quad's value by now) and row_mirror (i <-> 15 - i: the other eight); the other row of 16 by
// v_permlane16_swap.  No trip through LDS.
template <int CTRL>
__device__ __forceinline__ float dpp_moved(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
template <int LANES, typename Op>
__device__ __forceinline__ float group_reduce(float x, Op op) {
    static_assert(LANES == 4 || LANES == 8 || LANES == 16 || LANES == 32, "a group of 4, 8, 16 or 32 lanes");
    x = op(x, dpp_moved<0xB1>(x));
    x = op(x, dpp_moved<0x4E>(x));
    if constexpr (LANES >= 8) x = op(x, dpp_moved<0x141>(x));
    if constexpr (LANES >= 16) x = op(x, dpp_moved<0x140>(x));
    if constexpr (LANES >= 32) {
        float even, odd;
        row_pairs_of(x, even, odd);
        x = op(even, odd);
    }
    return x;
}
template <int LANES>
__device__ __forceinline__ float group_sum(float x) {
    return group_reduce<LANES>(x, [](float a, float b) { return a + b; });
}
template <int LANES>
__device__ __forceinline__ float group_min(float x) {
    return group_reduce<LANES>(x, [](float a, float b) { return fminf(a, b); });
}
template <int LANES>
__device__ __forceinline__ float group_max(float x) {
    return group_reduce<LANES>(x, [](float a, float b) { return fmaxf(a, b); });
}

}  // namespace tt
