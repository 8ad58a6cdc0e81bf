// Compare-and-pack primitives shared by the quantizer kernels and the fused 1x1 conv kernel: sixteen lanes (one
// DPP row) turn one row of 64 consecutive channels, read as 16 float4, into its packed element.
#pragma once
#include "tab_common.h"

namespace tab {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));
typedef uint32_t uintx2 __attribute__((ext_vector_type(2)));

// Threshold of an item of the lane's own; for partial sums a lane adds them up alone.
__device__ __forceinline__ float lane_threshold(const Thresholds &t, long item)
{
    if (t.values == nullptr) return 0.f;
    if (t.splits == 0) return t.values[item];
    double sum = 0.0;
    for (int i = 0; i < t.splits; i++) sum += (double)t.values[item * t.splits + i];
    return (float)(sum * t.scale);
}

// The sum of v over the wave (every lane active), in every lane.  Inside the rows of 16 lanes by DPP, then of the four rows: 50
// instructions without a wait, where six exchanges of a double through LDS took 0.4 us of every wave that added up a threshold.
__device__ __forceinline__ double wave_sum_f64(double v)
{
    auto exchanged = [](double x, auto control) {
        const uint64_t u = (uint64_t)__double_as_longlong(x);
        const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, decltype(control)::value, 0xF, 0xF, true);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), decltype(control)::value, 0xF, 0xF, true);
        return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
    };
    v += exchanged(v, std::integral_constant<int, 0xB1>());   // quad_perm [1,0,3,2]
    v += exchanged(v, std::integral_constant<int, 0x4E>());   // quad_perm [2,3,0,1]
    v += exchanged(v, std::integral_constant<int, 0x141>());  // row_half_mirror
    v += exchanged(v, std::integral_constant<int, 0x140>());  // row_mirror
    auto of_row = [&](int row) {
        const uint64_t u = (uint64_t)__double_as_longlong(v);
        const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, 16 * row), hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), 16 * row);
        return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
    };
    return (of_row(0) + of_row(1)) + (of_row(2) + of_row(3));
}

// Threshold of one item for a whole wave (every lane active): the lanes share the partial sums.  The order of the sum
// differs from lane_threshold's; a sum of up to 1024 fp32 values within a factor of 2^19 of each other is exact in fp64.
// In two steps, so that the first 256 partial sums can be requested before what the wave has to wait for longer (loads return in order).
// (One image of 224x224x64, 1024 partial sums: the layer 15.9 -> 13.2 us.)
__device__ __forceinline__ floatx4 request_threshold(const Thresholds &t, long item)
{
    const uint32_t lane = threadIdx.x & 63;
    const float *own = t.values + item * t.splits;  // a power of two of them: past 64 every lane has as many
    floatx4 part = {0.f, 0.f, 0.f, 0.f};
    if ((int)lane < t.splits) part[0] = own[lane];
    if (t.splits > 64) part[1] = own[lane + 64];
    if (t.splits > 128) part[2] = own[lane + 128], part[3] = own[lane + 192];
    return part;
}
__device__ __forceinline__ float finish_threshold(const Thresholds &t, long item, const floatx4 requested)
{
    auto add = [](const floatx4 v) { return ((double)v[0] + (double)v[1]) + ((double)v[2] + (double)v[3]); };
    double sum = add(requested);
    const float *own = t.values + item * t.splits + (threadIdx.x & 63);
    for (int i = 256; i < t.splits; i += 256) sum += add(floatx4{own[i], own[i + 64], own[i + 128], own[i + 192]});
    sum = wave_sum_f64(sum);
    return __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint((float)(sum * t.scale))));
}
__device__ __forceinline__ float given_threshold(const Thresholds &t, long item) { return t.values == nullptr ? 0.f : t.values[item]; }
__device__ __forceinline__ float wave_threshold(const Thresholds &t, long item)
{
    return t.splits == 0 ? given_threshold(t, item) : finish_threshold(t, item, request_threshold(t, item));
}

// Threshold of the lane's item, from partial sums, where the wave's items are first .. last (uniform; every lane active): of two the wave
// adds up both.  (A lane adding its item's partial sums up alone waits for one load after the other: in an NHWC tensor whose items are no
// multiple of 32 rows, the waves at their borders took 20 us: N=72 55x55x64 28.9 -> 11.4.)  More than two items are short ones of few partial sums each.
__device__ __forceinline__ float span_threshold(const Thresholds &t, long item, long first, long last, const floatx4 requested)
{
    if (last - first > 1) return lane_threshold(t, item);
    const float t_first = finish_threshold(t, first, requested);
    if (last == first) return t_first;
    const float t_last = finish_threshold(t, last, request_threshold(t, last));
    return item == first ? t_first : t_last;
}

// Four compares shifted into bits, two instructions each: bits = 2 * bits + (a < b), the carry of an addition being the
// compare's result.  (Select and OR take three to five, which is what bounds a lane that packs bits of its own on small
// tensors.)  The compares stand before the additions because a carry read as a scalar mask needs two other instructions
// between it and the compare that wrote it; the compiler cannot see into the block to put them there.
#define TAB_SHIFT_IN_LESS4(B0, B1, B2, B3, A0, A1, A2, A3, L0, L1, L2, L3)                                                       \
    "v_cmp_lt_f32_e64 %[c0], %[" A0 "], %[" L0 "]\n\tv_cmp_lt_f32_e64 %[c1], %[" A1 "], %[" L1 "]\n\t"                            \
    "v_cmp_lt_f32_e64 %[c2], %[" A2 "], %[" L2 "]\n\tv_cmp_lt_f32_e64 %[c3], %[" A3 "], %[" L3 "]\n\t"                            \
    "v_addc_co_u32_e64 %[" B0 "], %[c0], %[" B0 "], %[" B0 "], %[c0]\n\tv_addc_co_u32_e64 %[" B1 "], %[c1], %[" B1 "], %[" B1 "], %[c1]\n\t" \
    "v_addc_co_u32_e64 %[" B2 "], %[c2], %[" B2 "], %[" B2 "], %[c2]\n\tv_addc_co_u32_e64 %[" B3 "], %[c3], %[" B3 "], %[" B3 "], %[c3]"

// into the bits of four pixels
__device__ __forceinline__ void shift_in_less4(uint32_t (&bits)[4], const float (&a)[4], const float limit)
{
    uint64_t c0, c1, c2, c3;
    asm(TAB_SHIFT_IN_LESS4("b0", "b1", "b2", "b3", "a0", "a1", "a2", "a3", "l", "l", "l", "l")
        : [b0] "+v"(bits[0]), [b1] "+v"(bits[1]), [b2] "+v"(bits[2]), [b3] "+v"(bits[3]), [c0] "=&s"(c0), [c1] "=&s"(c1), [c2] "=&s"(c2), [c3] "=&s"(c3)
        : [a0] "v"(a[0]), [a1] "v"(a[1]), [a2] "v"(a[2]), [a3] "v"(a[3]), [l] "v"(limit));
}
// limit < a
__device__ __forceinline__ void shift_in_more4(uint32_t (&bits)[4], const float (&a)[4], const float limit)
{
    uint64_t c0, c1, c2, c3;
    asm(TAB_SHIFT_IN_LESS4("b0", "b1", "b2", "b3", "l", "l", "l", "l", "a0", "a1", "a2", "a3")
        : [b0] "+v"(bits[0]), [b1] "+v"(bits[1]), [b2] "+v"(bits[2]), [b3] "+v"(bits[3]), [c0] "=&s"(c0), [c1] "=&s"(c1), [c2] "=&s"(c2), [c3] "=&s"(c3)
        : [a0] "v"(a[0]), [a1] "v"(a[1]), [a2] "v"(a[2]), [a3] "v"(a[3]), [l] "v"(limit));
}

// into the bits of one pixel, a0 first
__device__ __forceinline__ void shift_in_less4(uint32_t &bits, const float a0, const float a1, const float a2, const float a3, const float limit)
{
    uint64_t c0, c1, c2, c3;
    asm(TAB_SHIFT_IN_LESS4("b", "b", "b", "b", "a0", "a1", "a2", "a3", "l", "l", "l", "l")
        : [b] "+v"(bits), [c0] "=&s"(c0), [c1] "=&s"(c1), [c2] "=&s"(c2), [c3] "=&s"(c3)
        : [a0] "v"(a0), [a1] "v"(a1), [a2] "v"(a2), [a3] "v"(a3), [l] "v"(limit));
}
__device__ __forceinline__ void shift_in_more4(uint32_t &bits, const float a0, const float a1, const float a2, const float a3, const float limit)
{
    uint64_t c0, c1, c2, c3;
    asm(TAB_SHIFT_IN_LESS4("b", "b", "b", "b", "l", "l", "l", "l", "a0", "a1", "a2", "a3")
        : [b] "+v"(bits), [c0] "=&s"(c0), [c1] "=&s"(c1), [c2] "=&s"(c2), [c3] "=&s"(c3)
        : [a0] "v"(a0), [a1] "v"(a1), [a2] "v"(a2), [a3] "v"(a3), [l] "v"(limit));
}
#undef TAB_SHIFT_IN_LESS4

// OR over the 8 lanes of each half of a 16-lane DPP row; every lane gets the result.
__device__ __forceinline__ uint32_t or_reduce8(uint32_t v)
{
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true);   // quad_perm [1,0,3,2]
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true);   // quad_perm [2,3,0,1]
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, true);  // row_half_mirror
    return v;
}

// value of the lane 8 positions further round the 16-lane DPP row (row_ror:8)
__device__ __forceinline__ uint32_t rotate_row8(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xF, 0xF, true);
}

// Compare one float4 against the threshold; bit e of the result belongs to element e.
// MODE 2, ternary: first test v > t (+1), only then v < -t (-1); both are strict and ordered, so
// ties and NaN give 0 (TAB_GEMM.cu:184-192).  MODE 1, binary: bit = v < t (TAB_GEMM.cu:231).
// MODE 5 (RTN fields) compares like MODE 2.  MODE 4 (2-bit levels): `sign` gets the weight-2 bit and
// `nz` the weight-1 bit of level = (v >= 0.5t) + (v >= 1.5t) + (v >= 2.5t).
template <int MODE>
__device__ __forceinline__ void compare4(const floatx4 v, const float t, uint32_t &sign, uint32_t &nz)
{
    const float e[4] = {v[0], v[1], v[2], v[3]};
    sign = 0;
    nz = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (MODE == 2 || MODE == 5) {
            const bool pos = e[i] > t;
            const bool neg = !pos && (e[i] < -t);
            nz |= (uint32_t)(pos || neg) << i;
            sign |= (uint32_t)neg << i;
        } else if (MODE == 4) {
            const int level = (int)(e[i] >= 0.5f * t) + (int)(e[i] >= 1.5f * t) + (int)(e[i] >= 2.5f * t);
            sign |= (uint32_t)(level >> 1) << i;
            nz |= (uint32_t)(level & 1) << i;
        } else {
            sign |= (uint32_t)(e[i] < t) << i;
        }
    }
}

// The packed output of one 64-channel row from the compare bits of lane l of its 16-lane DPP row; all
// lanes of the row take part, lane 0 gets the complete result: out[0..1] for MODE 1, out[0..3] else.
// MODE 1/2/4: the lane's nibble goes to bit 4*(l%8) and an OR over 8 lanes yields the low (lanes 0-7)
// or high (lanes 8-15) 32 bits of a plane word; a rotate by 8 within the row hands lane 0 the other
// half: (plane 0 low, plane 0 high, plane 1 low, plane 1 high).
// MODE 5: the row is two words of 32 two-bit fields (TAB_CPU.cpp:364-379); the lane's four fields
// (8 bits, even bit = nonzero, odd bit = sign) go to byte l%4 of the low (l%8 < 4) or high half of the
// word lanes 0-7 (channels 0-31) or lanes 8-15 (channels 32-63) build: (word 0 low, high, word 1 low, high).
// MASKED: the bits have been masked, so that the compiler cannot put the compares' results in their places by itself: they are spread.
template <int MODE, bool MASKED = false>
__device__ __forceinline__ void pack_row(uint32_t sign, uint32_t nz, int l, uint32_t (&out)[4])
{
    if (MODE == 5) {
        uint32_t fields = 0;
        if (MASKED) {
            uint32_t both = nz | sign << 16;
            both = (both | both << 2) & 0x00330033u;
            both = (both | both << 1) & 0x00550055u;
            fields = both | both >> 15;
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) fields |= (((nz >> i) & 1u) | (((sign >> i) & 1u) << 1)) << (2 * i);
        }
        const uint32_t placed = (fields & 0xffu) << (8 * (l & 3));
        const uint32_t lo = or_reduce8((l & 4) ? 0u : placed), hi = or_reduce8((l & 4) ? placed : 0u);
        out[0] = lo; out[1] = hi; out[2] = rotate_row8(lo); out[3] = rotate_row8(hi);
        return;
    }
    const int shift = 4 * (l & 7);
    const uint32_t sign_half = or_reduce8(sign << shift);
    out[0] = sign_half;
    out[1] = rotate_row8(sign_half);
    if (MODE != 1) {
        const uint32_t nz_half = or_reduce8(nz << shift);
        out[2] = nz_half;
        out[3] = rotate_row8(nz_half);
    }
}

// Spread the 32 bits of v to the even bits of a 64-bit word.
__device__ __forceinline__ uint64_t spread_bits(uint32_t v)
{
    uint64_t x = v;
    x = (x | x << 16) & 0x0000ffff0000ffffull;
    x = (x | x << 8) & 0x00ff00ff00ff00ffull;
    x = (x | x << 4) & 0x0f0f0f0f0f0f0f0full;
    x = (x | x << 2) & 0x3333333333333333ull;
    return (x | x << 1) & 0x5555555555555555ull;
}

// OR over the 16 lanes of a DPP row; every lane gets the result.
__device__ __forceinline__ uint32_t or_reduce16(uint32_t v)
{
    v = or_reduce8(v);
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, true);  // row_mirror
    return v;
}

// The packed element of one pixel's word, of any channel count, from the 16 lanes of a DPP row, lane l holding channels
// l + 16 * e: what pack_row gives for whole words.  Channels that do not exist stay 0 (TAB_GEMM.cu:203-206).
template <int MODE>
__device__ __forceinline__ void pack_row_strided(const float (&v)[4], float t, int l, int channels, uint32_t (&out)[4])
{
    uint32_t w[4] = {0, 0, 0, 0};  // plane 0 low, high, plane 1 low, high
#pragma unroll
    for (int e = 0; e < 4; e++) {
        uint32_t sign, nz;  // bit 0
        compare4<MODE>(floatx4{v[e], 0.f, 0.f, 0.f}, t, sign, nz);
        const uint32_t valid = l + 16 * e < channels ? 1u : 0u;
        w[e / 2] |= (sign & valid) << (l + 16 * (e % 2));
        if (MODE != 1) w[2 + e / 2] |= (nz & valid) << (l + 16 * (e % 2));
    }
#pragma unroll
    for (int i = 0; i < (MODE == 1 ? 2 : 4); i++) out[i] = or_reduce16(w[i]);
    if (MODE == 5) {
        const uint64_t word0 = spread_bits(out[2]) | spread_bits(out[0]) << 1, word1 = spread_bits(out[3]) | spread_bits(out[1]) << 1;
        out[0] = (uint32_t)word0; out[1] = (uint32_t)(word0 >> 32);
        out[2] = (uint32_t)word1; out[3] = (uint32_t)(word1 >> 32);
    }
}

}  // namespace
}  // namespace tab
