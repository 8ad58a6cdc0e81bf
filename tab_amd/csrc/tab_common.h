// Shared declarations of the gfx950 TAB kernels (internal; the public surface is
// include/tab_amd.h).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>
#include <type_traits>

#include "tab_route.h"

namespace tab {

constexpr int kWordBits = 64;  // channels per packed int64 word (CNTBITS, TAB_GEMM.cuh:10)

// Exact x / d for x < 65536 and 1 <= d < 65536 with one multiply-high:
// magic = floor(2^32 / d) + 1 gives floor(x * magic / 2^32) == floor(x / d) whenever
// x * d < 2^32.  d == 1 has no 32-bit magic and is passed through.
struct FastDiv {
    uint32_t magic;
    uint32_t d;
};
inline FastDiv make_fastdiv(uint32_t d)
{
    FastDiv f;
    f.d = d;
    f.magic = d > 1 ? (uint32_t)(0x100000000ull / d) + 1u : 0u;
    return f;
}
__device__ __forceinline__ uint32_t fastdiv(uint32_t x, FastDiv f)
{
    return f.d == 1 ? x : __umulhi(x, f.magic);
}

// Exact x / d for 0 <= x < 2^31 and 1 <= d < 2^31 with one 32x32 -> 64-bit multiply and a shift (a runtime
// divisor otherwise costs some 25 instructions a lane): with s = ceil(log2 d) and mul = floor(2^(31+s) / d) + 1,
// mul * d exceeds 2^(31+s) by at most d <= 2^s, so the quotient's error term x * (mul * d - 2^(31+s)) / (d * 2^(31+s))
// stays below 1 / d for every x < 2^31.
struct Div32 {
    uint32_t mul, shift;
};
inline Div32 make_div32(uint32_t d)
{
    const uint32_t s = d > 1 ? 32u - (uint32_t)__builtin_clz(d - 1) : 0u;
    Div32 f;
    f.shift = 31 + s;
    f.mul = (uint32_t)((((uint64_t)1 << (31 + s)) / d) + 1);
    return f;
}
__host__ __device__ __forceinline__ uint32_t div32(uint32_t x, Div32 f)
{
    return (uint32_t)(((uint64_t)x * f.mul) >> f.shift);
}

// Whether an fp32 Y of M rows of KN filters is written through the caches because its rows are no whole cache lines: a line is
// then completed by two waves or two tiles, and non-temporal stores send its parts to memory one by one once Y outgrows what the
// L2s hold (32 MB).  Non-temporal / cached, us: KN = 41 103 MB 83 / 26, KN = 106 115 MB 79 / 28, KN = 70 179 MB 132 / 51, KN = 958 52 MB
// 55 / 43, KN = 517 31 MB 11.4 / 9.5; one launch of quantizer and 1x1 conv: KN = 70 56 MB 51 / 26, KN = 513 26 MB 12.9 / 10.0, but KN = 100
// 20 MB 7.4 / 9.2.  At most 32 filters are one wave's own block of contiguous rows (KN = 25 29 MB 28.6 / 29.4).
__host__ __device__ __forceinline__ bool ragged_rows_cached(long M, int KN)
{
    return KN % 32 != 0 && KN > 32 && M * KN >= (6L << 20);
}

// Arguments of the fused pad + im2row + GEMM kernels; they travel as ConvParams (below).
struct ConvArgs {
    const uint64_t *qx;  // packed activation [N][H][W][PC][APL]; PC = words per pixel and plane
    const uint64_t *qw;  // packed weight     [KN][KH][KW][PC][BPL]
    const int32_t *btn;  // [KN] (BTN only)
    float *y;            // [M][KN]
    // packed output instead of y (matrix-core kernel only): 32-bit halves of [M][ceil(KN/64)][out_bits]
    uint32_t *qy;
    const float *out_ths;  // [N] thresholds applied to the outputs of image n; null: out_th for every image
    float out_th;
    int out_bits;          // 1 or 2
    int N, H, W, PC;
    int KN, KH, KW;
    int p1, p2, s1, s2;
    int OH, OW;
    int M;         // N*OH*OW
    int G;         // KH*KW*PC, packed words along K per plane
    int kcw;       // words per K chunk (at most the kernel's KCH; 6 bits of ConvParams)
    int nchunks;   // ceil(G / kcw)
    int num;       // KH*KW*C (BNN constant)
    int tiles_m;   // ceil(M / BM)
    int tiles_n;   // filter tiles when the workgroups are ordered by rows of Y (LDS-direct kernel, short K), else 0
    Div32 div_tiles_m;  // by tiles_m, or by 8 * tiles_n in that order (set by the launchers)
    int y_cached;       // fp32 output through the caches (1) or with non-temporal stores (0)
    int xcd_share;      // tiles each of the 8 XCDs takes as one contiguous run of rows of Y (0: order not XCD-aware)
    int filter_tiles;   // ceil(KN / BN), with div_filter_tiles, for that order
    Div32 div_filter_tiles;
    int tail_big;       // the mixed launch (conv_mfma_tail): workgroups that take whole 128x128 tiles; the rest take quarters
    int tail_chunks;    // chunks of K of a quarter in that launch
    FastDiv div_pc, div_kw;
    Div32 div_pixels, div_ow;  // by OH*OW and OW: an output row's image and line
};

// ConvArgs as a kernel receives it.  The host writes kernel arguments into device memory, and from 120 bytes on that costs
// 0.6-0.8 us a launch (measured launching back to back: 2.8 us up to 112 bytes, 3.4 at 120-128, 3.6-3.9 beyond; ConvArgs
// itself is 248), a quarter of a small call.  So what a kernel can derive in a few scalar instructions is left out (M and
// the tile counts), divisors are stored once, and small numbers share a dword: 104 bytes, 112 with packed output.  unpack_conv gives the kernels the ConvArgs back; what they do not use of it costs nothing.
struct ConvParams {
    const uint64_t *qx, *qw;
    void *out;             // y or qy
    uint64_t btn_or_num;   // BTN: btn, otherwise num
    int N, H, W, KN, OH, OW;
    int p1, p2, s1, s2;
    uint32_t pc_kw;        // PC | KW << 16
    uint32_t g_chunks;     // G | nchunks << 16
    uint32_t magic_pc, magic_kw, mul_pixels, mul_ow, mul_tiles;
    uint32_t bits;         // 0-4, 5-9, 10-14: shifts of the three divisors; then the flags below
};
struct ConvParamsPacked : ConvParams {
    const float *out_ths;  // or the bits of out_th (kConvOutConstant)
};
static_assert(sizeof(ConvParams) == 104 && sizeof(ConvParamsPacked) == 112, "kernel arguments below 120 bytes");
constexpr uint32_t kConvOutBits2 = 1u << 15;      // packed output of two planes
constexpr uint32_t kConvOutConstant = 1u << 16;   // one output threshold for every image
constexpr uint32_t kConvCachedY = 1u << 17;
constexpr uint32_t kConvXcdOrder = 1u << 18;      // xcd_share != 0
constexpr uint32_t kConvRowsOrder = 1u << 19;     // tiles_n != 0
constexpr int kConvKcwShift = 20;                 // kcw, 6 bits

template <bool PACKED>
using ConvParamsOf = typename std::conditional<PACKED, ConvParamsPacked, ConvParams>::type;

template <int TYPE, bool PACKED>
ConvParamsOf<PACKED> pack_conv(const ConvArgs &a)
{
    ConvParamsOf<PACKED> k;
    k.qx = a.qx;
    k.qw = a.qw;
    k.out = PACKED ? static_cast<void *>(a.qy) : static_cast<void *>(a.y);
    k.btn_or_num = TYPE == 2 ? (uint64_t)(uintptr_t)a.btn : (uint64_t)(uint32_t)a.num;
    k.N = a.N; k.H = a.H; k.W = a.W; k.KN = a.KN; k.OH = a.OH; k.OW = a.OW;
    k.p1 = a.p1; k.p2 = a.p2; k.s1 = a.s1; k.s2 = a.s2;
    k.pc_kw = (uint32_t)a.PC | (uint32_t)a.KW << 16;
    k.g_chunks = (uint32_t)a.G | (uint32_t)a.nchunks << 16;
    k.magic_pc = a.div_pc.magic;
    k.magic_kw = a.div_kw.magic;
    const Div32 tiles = a.xcd_share != 0 ? a.div_filter_tiles : a.div_tiles_m;
    k.mul_pixels = a.div_pixels.mul;
    k.mul_ow = a.div_ow.mul;
    k.mul_tiles = tiles.mul;
    k.bits = (a.div_pixels.shift - 31) | (a.div_ow.shift - 31) << 5 | (tiles.shift - 31) << 10 | (a.y_cached ? kConvCachedY : 0) |
             (a.xcd_share != 0 ? kConvXcdOrder : 0) | (a.tiles_n != 0 ? kConvRowsOrder : 0) | (uint32_t)a.kcw << kConvKcwShift;
    if constexpr (PACKED) {
        k.bits |= (a.out_bits == 2 ? kConvOutBits2 : 0) | (a.out_ths == nullptr ? kConvOutConstant : 0);
        uint32_t th;
        memcpy(&th, &a.out_th, sizeof th);
        k.out_ths = a.out_ths != nullptr ? a.out_ths : reinterpret_cast<const float *>((uintptr_t)th);
    }
    return k;
}

// BM, BN: the workgroup's tile.
template <int TYPE, bool PACKED, int BM, int BN>
__device__ __forceinline__ ConvArgs unpack_conv(const ConvParamsOf<PACKED> &k)
{
    ConvArgs a = {};
    a.qx = k.qx;
    a.qw = k.qw;
    if (PACKED) a.qy = static_cast<uint32_t *>(k.out);
    else a.y = static_cast<float *>(k.out);
    if (TYPE == 2) a.btn = reinterpret_cast<const int32_t *>((uintptr_t)k.btn_or_num);
    else a.num = (int)(uint32_t)k.btn_or_num;
    a.N = k.N; a.H = k.H; a.W = k.W; a.KN = k.KN; a.OH = k.OH; a.OW = k.OW;
    a.p1 = k.p1; a.p2 = k.p2; a.s1 = k.s1; a.s2 = k.s2;
    a.PC = (int)(k.pc_kw & 0xffffu);
    a.KW = (int)(k.pc_kw >> 16);
    a.G = (int)(k.g_chunks & 0xffffu);
    a.nchunks = (int)(k.g_chunks >> 16);
    a.div_pc = FastDiv{k.magic_pc, (uint32_t)a.PC};
    a.div_kw = FastDiv{k.magic_kw, (uint32_t)a.KW};
    a.div_pixels = Div32{k.mul_pixels, 31 + (k.bits & 31u)};
    a.div_ow = Div32{k.mul_ow, 31 + (k.bits >> 5 & 31u)};
    a.div_tiles_m = a.div_filter_tiles = Div32{k.mul_tiles, 31 + (k.bits >> 10 & 31u)};
    a.M = k.N * k.OH * k.OW;
    a.tiles_m = (a.M + BM - 1) / BM;
    a.filter_tiles = (k.KN + BN - 1) / BN;
    a.tiles_n = k.bits & kConvRowsOrder ? a.filter_tiles : 0;
    a.y_cached = (k.bits & kConvCachedY) != 0;
    a.kcw = (int)(k.bits >> kConvKcwShift & 63u);
    if constexpr (PACKED) {
        a.out_bits = k.bits & kConvOutBits2 ? 2 : 1;
        const bool constant = (k.bits & kConvOutConstant) != 0;
        a.out_ths = constant ? nullptr : k.out_ths;
        a.out_th = __uint_as_float((uint32_t)(uintptr_t)k.out_ths);
    }
    a.xcd_share = k.bits & kConvXcdOrder ? (int)((uint32_t)(a.tiles_m * a.filter_tiles) / 8u) : 0;
    return a;
}

// Compute units of the current device (256 on MI355X), looked up once; 256 if the lookup fails.
int device_compute_units();
void set_compute_units(int units);  // test hook of the rules that count them (0: the device's)

// The convolution that keeps the input patch of a tile in LDS (tab_conv_mfma_patch.h) reads the weights in an order of its own, in
// which the quantizer's launch leaves them in the caller's workspace (pack_weights, tab_patch_weights.h): its first `blocks`
// workgroups do that.
struct WeightJob {
    const uint64_t *qw;
    uint64_t *out;
    int KN;
    uint32_t pc_taps;    // PC | KH * KW << 16
    uint32_t blocks;
    uint32_t kc_planes;  // words of a chunk | bit planes << 8
};
static_assert(sizeof(WeightJob) == 32, "quantizers take it beside at most 80 bytes of arguments");

constexpr int kPatchShape = 12;  // shapes (of launch_conv_mfma) from here on are that kernel's
constexpr int kWavesShape = 19;  // and from here on those of the kernel that splits K over the waves of a workgroup
// Whether a call of these sizes may go there at all: the launches for which the plan is worked out.
bool conv_patch_considered(int type, long M, int KN, int KH, int KW);
// The plan of the automatic choice (or of the test hook's); fp32 output.
PatchPlan conv_patch_plan(int type, const ConvArgs &args);
// Bytes that hold the weights of any plan for these sizes.
size_t patch_weight_bytes(int type, int C, int KN, int KH, int KW);
WeightJob patch_weight_job(int type, const ConvArgs &args, const PatchPlan &plan, uint64_t *out);
hipError_t launch_patch_weights(const WeightJob &job, hipStream_t stream);  // the job in a launch of its own

// Launchers (tab_conv.hip / tab_quantize.hip); they enqueue on `stream` and return the
// launch status.
hipError_t launch_conv(int type, const ConvArgs &args, hipStream_t stream);
// Matrix-core (FP4 MFMA) variant; shape picks the workgroup tile.  conv_mfma_exact() says whether K is
// short enough for its fp32 accumulators to hold every partial sum exactly.
bool conv_mfma_exact(const ConvArgs &args);
bool conv_mfma_exact_levels(const ConvArgs &args);  // the same for type 4, whose products reach 9
int conv_mfma_shape(int type, const ConvArgs &args, float *cost_us = nullptr);
// At most 32 filters, fp32 output, an even number of words per pixel: the shapes of 64 filters that exist in a form of 32.
inline bool conv_mfma_narrow(const ConvArgs &a) { return a.KN <= 32 && a.PC % 2 == 0 && a.qy == nullptr; }
hipError_t launch_conv_mfma(int type, const ConvArgs &args, int shape, hipStream_t stream);
// Of the kernel with the weights in registers (tab_conv_mfma_regs.h): workgroups along M for `tiles` 32-pixel tiles: one tile per wave while
// the launch is small; from `cap` workgroups on, the fewest rounds with the waves evenly loaded.
inline unsigned regs_grid_x(int tiles, int cap)
{
    const int wanted = (tiles + 3) / 4;
    if (wanted <= cap) return (unsigned)wanted;
    const int rounds = (tiles + 4 * cap - 1) / (4 * cap);
    return (unsigned)(((tiles + rounds - 1) / rounds + 3) / 4);
}
// Packed output: how many of its workgroups a CU is to get, of `most` that fit.  As many as fit is not the soonest way: every workgroup expands its
// weights first, and the rounds of more waves divide the tiles more roughly.  What the busiest CU takes, in turns of its waves: rounds, each of
// its workgroups' turns and a wait that they do not hide (the longer of turns with few words), and the expansions; fewer only where that gains
// 2 %.  819 measured layers of 6 to 150 us (regs_workgroups_timings.txt): 0.967 of the time with as many as fit, the best count 0.958; seven more than
// 3 % slower, the worst 6 %.  Packing by comparisons, whose registers left room for fewer / by signs and as many as fit / this, us: one plane N=34
// 71x48x256->64 BTN 6.5 / 8.4 / 6.5, N=219 18x38x256->256 BNN 14.6 / 16.3 / 13.8, N=73 48x44x256->512 21.4 / 23.5 / 20.3, N=53 47x43x64->512 13.4 / 11.9 / 8.4.
inline int regs_on_cu(int G, int tiles, int tiles_n, int most, int cus)
{
    const int full = most < 4 ? most : 4;
    int best = full;
    float full_cost = 0.f, best_cost = 0.f;
    for (int n = full; n >= 2; n--) {
        const int cap = n * cus / tiles_n < 1 ? 1 : n * cus / tiles_n;
        const unsigned grid = regs_grid_x(tiles, cap) * (unsigned)tiles_n;
        const int rounds = ((tiles + 3) / 4 + cap - 1) / cap, busiest = (int)((grid + (unsigned)cus - 1) / (unsigned)cus);
        const float cost = (float)rounds * ((float)busiest + 0.2f + 0.3f / (float)G) + (float)busiest;
        if (n == full) full_cost = best_cost = cost;
        if (cost < best_cost) {
            best = n;
            best_cost = cost;
        }
    }
    return best_cost < 0.98f * full_cost ? best : full;
}
// Of the kernel that splits K over the waves of a workgroup (tab_conv_mfma_waves.h): the shape with the lowest predicted duration.
int conv_waves_shape(int type, const ConvArgs &args, float *cost_us);
// The shape of a launch of fp32 output: that kernel's, or the one that conv_mfma_shape picks.
int conv_fp32_shape(int type, const ConvArgs &args);
// What that kernel is predicted to gain over the tiles, microseconds: infinity where it has their place by rank, -infinity where it is not taken.
float conv_waves_gain(int type, const ConvArgs &args);
hipError_t launch_conv_mfma_tnn(const ConvArgs &args, int shape, hipStream_t stream);
hipError_t launch_conv_mfma_tbn(const ConvArgs &args, int shape, hipStream_t stream);
hipError_t launch_conv_mfma_btn(const ConvArgs &args, int shape, hipStream_t stream);
hipError_t launch_conv_mfma_bnn(const ConvArgs &args, int shape, hipStream_t stream);
hipError_t launch_conv_mfma_drf(const ConvArgs &args, int shape, hipStream_t stream);
hipError_t launch_conv_mfma_rtn(const ConvArgs &args, int shape, hipStream_t stream);

// Where a quantizer finds the threshold of item n: values[n] (splits == 0), the scaled sum of the item's `splits` partial
// sums of |x| that launch_abs_sums left (values[n * splits ...]; the quantizer adds them up itself, which saves the launch
// that would), or 0 for every item (values == null).
// eighth: which workgroups of a quantizer take what (see in_eighths); launchers are given 0, 1 or -1 and make it the workgroups of an
// eighth of the launch.
struct Thresholds {
    const float *values;
    double scale;
    int splits;
    int eighth;
};

// Consecutive workgroups go to consecutive XCDs, each with an L2 of its own that keeps its lines from one kernel to the next.  With
// `eighth` != 0 XCD x takes the x-th eighth of a launch's work in order (< 0: backwards), so that two launches over the same data
// find it in the L2s: 25.7 MB read a second time take 2.3 us instead of 5.1 (11 TB/s), and of more than the L2s hold (32 MB) the
// part read last is there for a launch that begins with it.  Workgroups past the eight eighths keep their place.
__host__ __device__ __forceinline__ uint32_t in_eighths(uint32_t block, int eighth)
{
    const uint32_t share = (uint32_t)(eighth < 0 ? -eighth : eighth), at = block >> 3;
    if (at >= share) return block;
    return (block & 7u) * share + (eighth < 0 ? share - 1 - at : at);
}
inline Thresholds ordered(Thresholds t, long blocks)
{
    t.eighth = t.eighth == 0 || blocks < 64 ? 0 : (int)(t.eighth < 0 ? -(blocks / 8) : blocks / 8);
    return t;
}
constexpr int kOwnPixelThresholds = -1;  // splits, conv_small only: images of one pixel, the kernel adds up |x| itself
inline Thresholds given_thresholds(const float *ths) { return Thresholds{ths, 0.0, 0, 0}; }

// count_workspace: quantize_count_workspace bytes for the counts of two planes, or null (they are then taken from the packed
// output, one launch more)
size_t quantize_count_workspace(int bitwidth, long items, long pixels_per_item, int C);
hipError_t launch_quantize(const float *x, const Thresholds &ths, int bitwidth, long pixels_per_item,
                           long items, int C, uint64_t *qx, int32_t *btn, int32_t *count_workspace, hipStream_t stream,
                           const WeightJob *weights = nullptr);  // weights: with btn == null only

// The same quantizer reading x as [N][C][H*W] (the CPU path's input layout, TAB_CPU.cpp:20-206); output as above.
hipError_t launch_quantize_nchw(const float *x, const Thresholds &ths, int bitwidth, int N, int C, long HW, uint64_t *qx,
                                int32_t *btn, int32_t *count_workspace, hipStream_t stream, const WeightJob *weights = nullptr);

// Of an NCHW tensor: whether the form that gathers words takes it (`unit` a thread), else the waves of a last word apart, or 0.
struct PlaneForm {
    bool gather;
    int unit, last;
};
PlaneForm plane_form(int bitwidth, long N, long HW, int C);

// Small items of two planes, a workgroup each (tab_quantize_item.hip): with given thresholds and the counts (btn), or with thresholds
// that it finds itself, scale * mean|x|, as launch_threshold would to the last bit.  own: which of the two.
bool quantize_items_supported(bool own, bool nchw, long items, long pixels, int C);
hipError_t launch_quantize_items(const float *x, const Thresholds &ths, bool nchw, long items, long pixels, int C, uint64_t *qx, int32_t *btn,
                                 hipStream_t stream);
hipError_t launch_quantize_own(const float *x, float scale, bool nchw, long items, long pixels, int C, uint64_t *qx, hipStream_t stream);

// Packers of the CPU-only conv types: format 4 = DoReFa 2-bit levels, 5 = RTN fields.
hipError_t launch_quantize_format(const float *x, const float *ths, int format, long pixels_per_item, long items, int C,
                                  uint64_t *qx, hipStream_t stream, const WeightJob *weights = nullptr);

// Quantize only the pixels (oh*s1, ow*s2) of every image into a compact [N][OH][OW][PC] activation
// (what a 1x1 convolution with stride and no padding reads).
bool quantize_strided_supported(const float *x, int H, int W, int C, int OH, int OW);
hipError_t launch_quantize_strided(const float *x, const Thresholds &ths, int bitwidth, int N, int H, int W, int C, int OH,
                                   int OW, int s1, int s2, uint64_t *qx, hipStream_t stream);

// ths[n] = scale * mean|x[n]| over per_item elements; `partial` holds items * threshold_splits()
// floats of scratch.
int threshold_splits(long items, long per_item);
// The first half of launch_threshold: what a quantizer needs to find the thresholds itself (*source, in `partial`).
hipError_t launch_abs_sums(const float *x, long items, long per_item, float scale, float *partial, Thresholds *source,
                           hipStream_t stream);
// ths[n] from what launch_abs_sums left.
hipError_t launch_threshold_values(const Thresholds &source, long items, float *ths, hipStream_t stream);
hipError_t launch_threshold(const float *x, long items, long per_item, float scale, float *ths, float *partial,
                            hipStream_t stream);

// Quantize + 1x1 conv in one launch (tab_conv_fused1x1.hip), for calls that are bound by their launches.
bool conv1x1_fused_supported(int type, const float *x, int C, int KH, int KW, int p1, int p2, long M, int KN);
hipError_t launch_conv1x1_fused(int type, const float *x, const Thresholds &ths, const uint64_t *qw, const int32_t *btn, float *y, int N,
                                int H, int W, int C, int KN, int s1, int s2, int OH, int OW, hipStream_t stream);

// Quantize + convolution in one launch for the smallest calls (tab_conv_small.hip); x NHWC or NCHW.
bool conv_small_supported(int type, const float *x, bool nchw, int N, int H, int W, int C, int KN, int KH, int KW, int p1, int p2, int s1,
                          int s2, int OH, int OW);
// False where conv_small cannot run the call; cost: the predicted microseconds on the GPU and the three numbers they come from.
bool conv_small_cost(int type, const float *x, bool nchw, int N, int H, int W, int C, int KN, int KH, int KW, int p1, int p2, int s1, int s2,
                     int OH, int OW, float (&cost)[4]);
bool conv_small_in_one_image(int OH, int OW);
// Images of one pixel (H = W = 1, a 1x1 kernel without padding): conv_small takes kOwnPixelThresholds.
bool conv_small_own_thresholds(const float *x, int H, int W, int C, int KH, int KW, int p1, int p2);
hipError_t launch_conv_small(int type, const float *x, bool nchw, const Thresholds &ths, const uint64_t *qw, const int32_t *btn, float *y,
                             int N, int H, int W, int C, int KN, int KH, int KW, int p1, int p2, int s1, int s2, int OH, int OW,
                             hipStream_t stream);

void force_conv_tile(int tm, int ng);  // tuning hook: 0,0 restores the automatic choice
void set_tail_round(int workgroups);   // test hook of the mixed launch: workgroups counted as one round of the chip (0: the CUs)
int tail_round();
bool conv_kernel_forced();             // true while tab_set_conv_kernel holds a choice other than the automatic one

}  // namespace tab
