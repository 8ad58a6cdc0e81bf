// Matrix-core conv kernel for launches of few tiles: K split over the waves of a workgroup, operands straight into registers.
//
// Such a launch lasts as long as one wave's chain of waits.  The kernel that had these launches before let four waves share chunks of K in
// LDS, and each chunk was a round trip to memory, a write to LDS and a barrier before its first MFMA; but waves that take different words
// of K share nothing.  So every wave loads its own words, all of the first units' at once, expands and multiplies them as they arrive, and
// the only barrier is the one before the partial sums are added up.
//   * Lane (kb, r) loads the words of pixel r and of filter r that its half-wave feeds, through buffer descriptors (padding, rows past M,
//     filters past KN and words past K are an offset select that reads zeros).  What bounds the loads of a launch of many tiles is the
//     cache lines an instruction touches, 32, so a lane takes two words of an operand of one plane at once: 16 bytes.
//   * Eight waves a tile where a CU gets few tiles, four from about one tile of 32x32 a CU on: more waves only add to the sums in
//     LDS.  64x32 and 32x64 tiles, three expansions for two MFMAs instead of four, where the launch is several rounds of those.
//   * Two units ahead (three of one word): with three (five) the registers leave seven waves a SIMD instead of eight, 5 % on launches of 2000
//     tiles and more.
// Tried and not in the tree: weights requested before the pixels' addresses are worked out, and 16-byte LDS accesses for the sums (3-10 %
// slower); 64x64 tiles, two or sixteen waves a tile, eight on 64x32 (no more than 2 % on few launches).
// In graph replays behind the quantizer, kernel with shared chunks / this, us: 2048->235 linear TNN 4.1 / 2.9, N=4 7x7x512->512 BNN 4.6 / 3.1,
// N=16 5.6 / 4.2, N=5 37x53x100->75 5x5 stride 2 TBN 5.6 / 3.7, N=197 11x7x384->64 stride 2 type 5 9.4 / 3.6; 1900 random layers 0.74.  The rule
// that takes it, conv_waves_or in tab_conv.hip.
#pragma once
#include "tab_conv_mfma.h"

namespace tab {
namespace {

// Words a half-wave takes at once: two where that makes the loads of an operand of one plane 16 bytes.  Types whose operands both have two
// planes gain nothing from it and share the pairs out more evenly.
template <int TYPE> constexpr bool kWavesOneWord = Planes<TYPE>::A == 2 && Planes<TYPE>::B == 2;

// One tile of 32*TM x 32*TN a workgroup.  A unit is 2 * W words of K, W consecutive ones for each half-wave; wave w multiplies units w, w + WAVES, ...
template <int TYPE, int WAVES, int TM, int TN, int W, int AHEAD>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(TM * TN > 1 ? 4 : (TYPE == 2 ? 6 : 8)))) void conv_mfma_waves(const ConvParams k)
{
    constexpr int BM = 32 * TM, BN = 32 * TN;
    const ConvArgs p = unpack_conv<TYPE, false, BM, BN>(k);
    constexpr int APL = Planes<TYPE>::A, BPL = Planes<TYPE>::B;
    constexpr int MINE = 16 / WAVES;  // accumulator elements of a lane and tile that a wave finishes
    __shared__ float partial[WAVES * TM * TN * 17 * 64];  // of each tile 16 accumulators and the BTN count a lane

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int r = lane & 31, kb = lane >> 5;
    int tile_m, tile_n;
    if (!tile_of_workgroup(p, tile_m, tile_n)) return;
    const int m0 = tile_m * BM, n0 = tile_n * BN;

    // the lane's output pixels
    const int pixels = p.OH * p.OW;
    const int n_first = (int)div32((uint32_t)m0, p.div_pixels);  // uniform
    const size_t image_words = (size_t)p.H * p.W * p.PC * APL;
    const size_t a_bytes = (size_t)(p.N - n_first) * image_words * 8;
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(p.qx + (size_t)n_first * image_words), 0,
                                                                            a_bytes > 0xffffffffull ? (int)0xffffffffu : (int)a_bytes, kBufferFlags);
    int ih0[TM], iw0[TM];
    uint32_t a_base[TM];
#pragma unroll
    for (int mt = 0; mt < TM; mt++) {
        const int m = m0 + mt * 32 + r;
        const bool a_live = m < p.M;
        const int mm = a_live ? m : m0;
        const int n = (int)div32((uint32_t)mm, p.div_pixels);
        const int rem = mm - n * pixels;
        const int oh = (int)div32((uint32_t)rem, p.div_ow), ow = rem - oh * p.OW;
        ih0[mt] = a_live ? oh * p.s1 - p.p1 : -(1 << 30);  // a dead row fails every bounds check
        iw0[mt] = ow * p.s2 - p.p2;
        a_base[mt] = (uint32_t)((((n - n_first) * p.H + (oh * p.s1 - p.p1)) * p.W + iw0[mt]) * p.PC) * (uint32_t)(APL * 8);
    }
    const size_t filter_bytes = (size_t)p.G * BPL * 8;
    const size_t b_bytes = (size_t)(p.KN - n0 < BN ? p.KN - n0 : BN) * filter_bytes;
    const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(p.qw + (size_t)n0 * p.G * BPL), 0, (int)b_bytes, kBufferFlags);
    int btn[TN];
#pragma unroll
    for (int nt = 0; nt < TN; nt++) btn[nt] = (TYPE == 2 && n0 + nt * 32 + r < p.KN) ? p.btn[n0 + nt * 32 + r] : 0;
    const ExpandConsts consts;

    struct Unit { uint32_t a[TM][W][2 * APL], b[TN][W][2 * BPL]; };
    const int units = (p.G + 2 * W - 1) / (2 * W);
    auto load = [&](auto &dst, auto planes_constant, __amdgpu_buffer_rsrc_t rsrc, uint32_t offset) {
        constexpr int PL = decltype(planes_constant)::value;
        if constexpr (PL == 1 && W == 1) {
            const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rsrc, offset, 0, 0);
            dst[0][0] = v[0]; dst[0][1] = v[1];
        } else {
#pragma unroll
            for (int i = 0; i < W * PL / 2; i++) {
                const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, offset == kNoData ? kNoData : offset + 16u * i, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; e++) dst[PL == 2 ? i : e / 2][PL == 2 ? e : e % 2] = v[e];
            }
        }
    };
    auto fetch = [&](Unit &u, int unit) {
        const int g = unit * (2 * W) + kb * W;
        const int tap = (int)fastdiv((uint32_t)g, p.div_pc), pc = g - tap * p.PC;
        const int kh = (int)fastdiv((uint32_t)tap, p.div_kw), kw = tap - kh * p.KW;
        const bool there = g < p.G;
        const uint32_t tap_off = (uint32_t)((kh * p.W + kw) * p.PC + pc) * (uint32_t)(APL * 8);
#pragma unroll
        for (int mt = 0; mt < TM; mt++) {
            const bool ok = there && (unsigned)(ih0[mt] + kh) < (unsigned)p.H && (unsigned)(iw0[mt] + kw) < (unsigned)p.W;
            load(u.a[mt], std::integral_constant<int, APL>(), a_rsrc, ok ? a_base[mt] + tap_off : kNoData);
        }
#pragma unroll
        for (int nt = 0; nt < TN; nt++) {
            const bool ok = there && n0 + nt * 32 + r < p.KN;
            load(u.b[nt], std::integral_constant<int, BPL>(), b_rsrc, ok ? (uint32_t)(nt * 32 + r) * (uint32_t)filter_bytes + (uint32_t)g * (uint32_t)(BPL * 8) : kNoData);
        }
    };

    f32x16 acc[TM][TN];
#pragma unroll
    for (int mt = 0; mt < TM; mt++)
#pragma unroll
        for (int nt = 0; nt < TN; nt++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[mt][nt][e] = 0.f;
    int b_nonzero[TN] = {};
    auto multiply = [&](const Unit &u) {
#pragma unroll
        for (int w = 0; w < W; w++)
#pragma unroll
            for (int h = 0; h < (TYPE == 5 ? 1 : 2); h++) {
                i32x8 a[TM], b[TN];
#pragma unroll
                for (int mt = 0; mt < TM; mt++)
                    a[mt] = TYPE == 5 ? expand_operand<TYPE, 0>(u.a[mt][w][0], u.a[mt][w][1], consts) : expand_operand<TYPE, 0>(u.a[mt][w][h], u.a[mt][w][2 * (APL - 1) + h], consts);
#pragma unroll
                for (int nt = 0; nt < TN; nt++) {
                    b[nt] = TYPE == 5 ? expand_operand<TYPE, 1>(u.b[nt][w][0], u.b[nt][w][1], consts) : expand_operand<TYPE, 1>(u.b[nt][w][h], u.b[nt][w][2 * (BPL - 1) + h], consts);
                    if (TYPE == 2) b_nonzero[nt] += __builtin_popcount(u.b[nt][w][2 * (BPL - 1) + h]);
                }
#pragma unroll
                for (int mt = 0; mt < TM; mt++)
#pragma unroll
                    for (int nt = 0; nt < TN; nt++)
                        acc[mt][nt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a[mt], b[nt], acc[mt][nt], 4, 4, 0, 0, 0, 0);
            }
    };

    Unit held[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; i++)
        if (wave + i * WAVES < units) fetch(held[i], wave + i * WAVES);
    for (int u0 = wave; u0 < units; u0 += AHEAD * WAVES)
#pragma unroll
        for (int i = 0; i < AHEAD; i++) {
            if (u0 + i * WAVES >= units) break;
            multiply(held[i]);
            if (u0 + (i + AHEAD) * WAVES < units) fetch(held[i], u0 + (i + AHEAD) * WAVES);
        }
    scale_sums<TYPE>(acc);

    // the waves' sums meet in LDS: wave w finishes elements w * MINE ... of each tile
    auto slot = [&](int w, int t, int e) -> float & { return partial[((w * TM * TN + t) * 17 + e) * 64 + lane]; };
#pragma unroll
    for (int t = 0; t < TM * TN; t++) {
#pragma unroll
        for (int e = 0; e < 16; e++) slot(wave, t, e) = acc[t / TN][t % TN][e];
        if (TYPE == 2) slot(wave, t, 16) = (float)b_nonzero[t % TN];
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TM * TN; t++) {
        auto total = [&](int e) {
            float sum = 0.f;
#pragma unroll
            for (int w = 0; w < WAVES; w++) sum += slot(w, t, e);
            return sum;
        };
        float bias = 0.f;
        if (TYPE == 2) {
            const float nonzero = total(16);
            bias = (float)btn[t % TN] - (nonzero + __shfl_xor(nonzero, 32, 64));
        }
        if (TYPE == 3) bias = (float)(p.num - 64 * (units * 2 * W));
        const int col = n0 + t % TN * 32 + r;
#pragma unroll
        for (int i = 0; i < MINE; i++) {
            const int e = wave * MINE + i;
            const int row = m0 + t / TN * 32 + 8 * (e >> 2) + 4 * kb + (e & 3);
            const float y = total(e) + bias;
            if (col < p.KN && row < p.M) __builtin_nontemporal_store(y, &p.y[(size_t)row * p.KN + col]);
        }
    }
}

template <int TYPE, int WAVES, int TM, int TN, int W, int AHEAD>
hipError_t launch_waves_of(ConvArgs a, hipStream_t stream)
{
    a.kcw = 0;
    a.nchunks = 0;
    a.tiles_m = (a.M + 32 * TM - 1) / (32 * TM);
    const long blocks = order_workgroups<Planes<TYPE>::A>(a, (a.KN + 32 * TN - 1) / (32 * TN));
    if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
    conv_mfma_waves<TYPE, WAVES, TM, TN, W, AHEAD><<<dim3((unsigned)blocks), dim3(64 * WAVES), 0, stream>>>(pack_conv<TYPE, false>(a));
    return hipGetLastError();
}

template <int TYPE, int WAVES, int TM, int TN>
hipError_t launch_waves(const ConvArgs &a, hipStream_t stream)
{
    if (a.qy != nullptr) return hipErrorInvalidValue;  // fp32 output only
    if constexpr (!kWavesOneWord<TYPE>)
        if (a.PC % 2 == 0) return launch_waves_of<TYPE, WAVES, TM, TN, 2, 2>(a, stream);
    return launch_waves_of<TYPE, WAVES, TM, TN, 1, 3>(a, stream);
}

}  // namespace
}  // namespace tab
