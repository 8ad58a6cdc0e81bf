// Quantize + 1x1 convolution in one launch: ConvWithCuda_TAB's quantize, pad, im2row and GEMM stages
// (TAB_GEMM.cu:419-509) without the packed activation ever reaching memory.
//
// A 1x1 convolution without padding reads each input pixel (oh*s1, ow*s2) for one output pixel only, so the activation
// a workgroup multiplies is exactly the activation it quantizes.  A workgroup owns 32 output pixels and a run of filter
// tiles:
//   * its four waves read the 32 pixels' channels as fp32, one 64-channel word per 16-lane DPP row, 4 rows per wave
//     instruction (the quantizer's lane layout, tab_pack.h), threshold them with the image's threshold
//     (TAB_GEMM.cu:184-192, 231) and leave the packed words in LDS, [word][pixel].  Where a load belongs to one pixel a lane
//     works out one of the 32 (image, place, threshold) and hands it over as scalars; a wave's loads are all requested before
//     the first is used;
//   * meanwhile every lane has requested its own words of the first filter tile, straight from global memory: lane (kb, r)
//     of a wave feeds word 2j + kb of filter r of the tile for each pair of words j, and multiplies the word's low half in
//     one MFMA and its high half in the next (the order of tab_conv_mfma_direct.h);
//   * after one barrier each wave multiplies the 32 pixels with filter tile after filter tile, the next one's words in
//     flight, and stores a 32x32 block of Y per tile, 128 contiguous bytes of two rows per instruction.
//
// What bounds it and how the work is split: a small launch lasts as long as one workgroup's instructions and its two round
// trips (X, then the drain of its stores), so every wave gets one filter tile and the pixels are quantized again for every 128
// filters; a large one is bound by reading X and writing Y, and a wave walks two filter tiles where that halves the
// readings of X (fused_tiles).  Where the line to the other kernels lies: conv1x1_fused_supported.
#include "tab_conv_mfma.h"
#include "tab_pack.h"

namespace tab {
namespace {

struct Fused1x1Args {
    const float *x;       // fp32 [N][H][W][C]
    Thresholds ths;       // of the N images
    const uint64_t *qw;   // packed weight [KN][PC][BPL]
    const int32_t *btn;   // [KN] (BTN only)
    float *y;             // [M][KN]
    int H, W, C;          // (C: also the BNN constant)
    int KN, s1, s2;
    int pixels, OW, M;    // pixels = OH * OW
    uint32_t mul_pixels, mul_ow, mul_pc;  // mul_pc: x / PC = x * mul_pc >> 16 for x below 2^16 / PC
    uint32_t shifts_tiles;  // shift of the division by pixels (6 bits), by OW (6 bits), filter tiles a wave walks
};
static_assert(sizeof(Fused1x1Args) <= 112, "kernel arguments below 120 bytes (see ConvParams)");

// How a wave reads the pixels' channels.  Which pixel and word a load belongs to is uniform over the wave in the first and
// the last form, so that the addresses are scalar.
enum FusedInput {
    kInputQuads = 0,   // whole 64-channel words, a multiple of four of them: a load is 1 KB of one pixel
    kInputWords = 1,   // whole 64-channel words: 16 bytes a lane, a word per 16-lane row
    kInputRagged = 2   // any channel count or alignment: a word per load, 4 bytes a lane, packed by the compare's wave mask
};

// NP: pairs of words, enough for a pixel's (1, 2 or 4).
// CACHED: Y through the caches (ragged_rows_cached).
template <int TYPE, int NP, int INPUT, bool CACHED, bool OWN>
__global__ __launch_bounds__(kConvThreads) void conv1x1_fused(const Fused1x1Args p)
{
    static_assert(TYPE >= 0 && TYPE <= 3, "types 0..3");
    constexpr int APL = Planes<TYPE>::A, BPL = Planes<TYPE>::B;
    constexpr int MODE = APL;             // ternary or binary activation
    constexpr int WORDS = 2 * NP;         // words a pixel takes in LDS (p.C has at most as many)
    constexpr bool RAGGED = INPUT == kInputRagged;
    constexpr int WIDE = RAGGED ? 1 : 4;  // words per load
    constexpr int LOADS = 32 / 4 * WORDS / WIDE;  // a wave's share of the 32 pixels, all in flight
    extern __shared__ __attribute__((aligned(16))) uint32_t act[];  // [word][pixel][plane][half]

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int r = lane & 31, kb = lane >> 5;
    const int sub = lane >> 4, l = lane & 15;
    const int m0 = (int)(OWN ? in_eighths(blockIdx.x, p.ths.eighth) : blockIdx.x) * 32;
    const int PC = (p.C + kWordBits - 1) / kWordBits;
    const int tiles = (int)(p.shifts_tiles >> 12);
    const int live = p.M - m0 < 32 ? p.M - m0 : 32;
    const ExpandConsts consts;

    // output pixel m -> image and the byte offset of its input pixel
    auto place_of = [&](int m, int &n) {
        m = m < p.M ? m : p.M - 1;
        n = (int)div32((uint32_t)m, Div32{p.mul_pixels, p.shifts_tiles & 63u});
        const int rem = m - n * p.pixels;
        const int oh = (int)div32((uint32_t)rem, Div32{p.mul_ow, p.shifts_tiles >> 6 & 63u}), ow = rem - oh * p.OW;
        return (size_t)(uint32_t)((n * p.H + oh * p.s1) * p.W + ow * p.s2) * (size_t)p.C * 4;  // pixels: < 2^31 (launch check)
    };
    // forms with a uniform pixel per load: lane r works out pixel m0 + r and hands it over
    constexpr bool HANDED = INPUT != kInputWords;
    int n = 0;
    const size_t in_offset = HANDED ? place_of(m0 + r, n) : 0;
    // OWN: thresholds from the layer's own sums: the wave adds up those of its pixels' first and last image, requested before x.  (In a
    // launch of its own it took 2 to 3 us: N=8 56x56x64->256 12.2 -> 10.4, one image of 56x56x64->64 11.2 -> 8.3.  A form of its own,
    // since the code that is not run costs the calls with given thresholds 2 %.)
    int n_first = 0, n_last = 0;
    floatx4 requested = {};
    if (OWN) {
        if (HANDED) {
            n_first = __builtin_amdgcn_readfirstlane(n);
            n_last = __builtin_amdgcn_readlane(n, 31);
        } else {
            place_of(m0, n_first);
            place_of(m0 + live - 1, n_last);
            n_first = __builtin_amdgcn_readfirstlane(n_first);
            n_last = __builtin_amdgcn_readfirstlane(n_last);
        }
        requested = request_threshold(p.ths, n_first);
    }

    // ---- activation: row = pixel * PC + word of the tile; load i of the wave takes the rows (4*i + wave) * WIDE ... ------
    // (ragged: load i is word i % WORDS of the pixel 4 * (i / WORDS) + wave.  Code that runs once costs its instructions: with
    // a division and a 64-bit product per load, 50 a word, the ragged form was four times slower)
    const int rows = live * PC;
    auto row_of = [&](int i) { return (4 * i + wave) * WIDE; };  // the load's first row
    auto last_row = [&](int row) { return row < rows ? row : rows - WIDE; };  // rows past the end: the last again, left out below
    auto pixel_of = [&](int row) { return (int)((uint32_t)row * p.mul_pc >> 16); };  // rows: at most 32 * 8
    auto lane_bits = [](uint32_t v, int from) { return (uint32_t)__builtin_amdgcn_readlane((int)v, from); };
    auto uniform_offset = [&](int pixel) { return (size_t)lane_bits((uint32_t)(in_offset >> 32), pixel) << 32 | lane_bits((uint32_t)in_offset, pixel); };
    const char *const x = reinterpret_cast<const char *>(p.x);
    float v[LOADS][WIDE];
    float th_row[HANDED ? 1 : LOADS];  // thresholds of the loads' rows where no lane hands them over
#pragma unroll
    for (int i = 0; i < LOADS; i++) {
        if constexpr (RAGGED) {
            const int pixel = min(4 * (i / WORDS) + wave, live - 1), w = i % WORDS;
            const int last = p.C - 1 - w * kWordBits;  // past the last channel: that one again, masked below (a word past the last: unused)
            v[i][0] = *reinterpret_cast<const float *>(x + (uniform_offset(pixel) + (uint32_t)(w * 256 + 4 * min(lane, last))));
        } else {
            int pixel, word, off_lane;
            size_t off;
            if constexpr (INPUT == kInputWords) {
                const int row = row_of(i) + sub < rows ? row_of(i) + sub : rows - 1;
                pixel = pixel_of(row);
                word = row - pixel * PC;
                off_lane = l * 16;
                int image;
                off = place_of(m0 + pixel, image);
                th_row[i % (HANDED ? 1 : LOADS)] = OWN ? (n_last - n_first > 1 ? lane_threshold(p.ths, image) : image == n_first ? 0.f : 1.f)
                                                       : given_threshold(p.ths, image);
            } else {
                const int row = last_row(row_of(i));
                pixel = pixel_of(row);
                word = row - pixel * PC;
                off_lane = lane * 16;
                off = uniform_offset(pixel);
            }
            const floatx4 w = *reinterpret_cast<const floatx4 *>(x + (off + (uint32_t)word * 256u) + (uint32_t)off_lane);
#pragma unroll
            for (int e = 0; e < WIDE; e++) v[i][e] = w[e % 4];
        }
    }
    float th = 0.f;
    if (HANDED) {
        th = OWN ? span_threshold(p.ths, n, n_first, n_last, requested) : given_threshold(p.ths, n);
    } else if (OWN && n_last - n_first <= 1) {
        const float t_first = finish_threshold(p.ths, n_first, requested), t_last = n_last == n_first ? t_first : wave_threshold(p.ths, n_last);
#pragma unroll
        for (int i = 0; i < (HANDED ? 1 : LOADS); i++) th_row[i] = th_row[i] == 0.f ? t_first : t_last;
    }

    // ---- weights: filter tile t of this wave --------------------------------------------------------
    const int n_wave = (blockIdx.y * 4 + wave) * tiles * 32;  // first filter of the wave
    uint32_t raw[NP][2 * BPL];
    auto request_weights = [&](int t) {
        int f = n_wave + t * 32 + r;
        f = f < p.KN ? f : p.KN - 1;  // filters past KN repeat the last one and are never stored
#pragma unroll
        for (int j = 0; j < NP; j++) {
            const int word = 2 * j + kb;
            const uint32_t *src = reinterpret_cast<const uint32_t *>(p.qw + ((size_t)f * PC + (word < PC ? word : PC - 1)) * BPL);
            if (BPL == 2) {
                const u32x4 q = *reinterpret_cast<const u32x4 *>(src);
#pragma unroll
                for (int e = 0; e < 4; e++) raw[j][e % (2 * BPL)] = word < PC ? q[e] : 0u;
            } else {
                const u32x2 q = *reinterpret_cast<const u32x2 *>(src);
#pragma unroll
                for (int e = 0; e < 2; e++) raw[j][e] = word < PC ? q[e] : 0u;
            }
        }
    };
    request_weights(0);

    // ---- threshold, pack, deposit -----------------------------------------------------------------------------------
    // words past PC are zeros on both sides (0 for a ternary operand; +64 each for binary x binary, which the bias counts)
    for (int i = tid; i < (WORDS - PC) * 32 * APL * 2; i += kConvThreads) act[PC * 32 * APL * 2 + i] = 0u;
    auto leave = [&](int word, int pixel, const uint32_t (&q)[4]) {
        uint32_t *dst = act + (word * 32 + pixel) * (2 * APL);
        if (APL == 2) *reinterpret_cast<uintx4 *>(dst) = uintx4{q[0], q[1], q[2], q[3]};
        else *reinterpret_cast<uintx2 *>(dst) = uintx2{q[0], q[1]};
    };
    if constexpr (RAGGED) {
        uint32_t mine[4] = {0, 0, 0, 0};  // lane i: the element of load i
#pragma unroll
        for (int i = 0; i < LOADS; i++) {
            const float t = __uint_as_float(lane_bits(__float_as_uint(th), min(4 * (i / WORDS) + wave, live - 1)));
            uint64_t sign, nz = 0;
            if (MODE == 2) {
                const uint64_t pos = __ballot(v[i][0] > t);
                sign = __ballot(v[i][0] < -t) & ~pos;
                nz = pos | sign;
            } else {
                sign = __ballot(v[i][0] < t);
            }
            const bool me = lane == i;
            mine[0] = me ? (uint32_t)sign : mine[0];
            mine[1] = me ? (uint32_t)(sign >> 32) : mine[1];
            if (MODE == 2) {
                mine[2] = me ? (uint32_t)nz : mine[2];
                mine[3] = me ? (uint32_t)(nz >> 32) : mine[3];
            }
        }
        const int word = lane % WORDS, pixel = 4 * (lane / WORDS) + wave;
        const uint64_t exist = word == PC - 1 ? ~(uint64_t)0 >> (PC * kWordBits - p.C) : ~(uint64_t)0;
#pragma unroll
        for (int e = 0; e < 4; e++) mine[e] &= (uint32_t)(exist >> (32 * (e & 1)));
        if (lane < LOADS && word < PC && pixel < live) leave(word, pixel, mine);
    } else {
#pragma unroll
        for (int i = 0; i < LOADS; i++) {
            uint32_t out[4];
            const int row = row_of(i) + (INPUT == kInputWords ? sub : 0);
            const int pixel = pixel_of(INPUT == kInputWords ? (row < rows ? row : rows - 1) : last_row(row));
            const float t = HANDED ? __uint_as_float(lane_bits(__float_as_uint(th), pixel)) : th_row[i % (HANDED ? 1 : LOADS)];
            uint32_t sign, nz;
            compare4<MODE>(floatx4{v[i][0], v[i][1 % WIDE], v[i][2 % WIDE], v[i][3 % WIDE]}, t, sign, nz);
            pack_row<MODE>(sign, nz, l, out);  // lane 0 of the row holds (plane 0 low, high[, plane 1 low, high])
            const int word = row + (INPUT == kInputWords ? 0 : sub) - pixel * PC;
            if (l == 0 && row < rows) leave(word, pixel, out);
        }
    }
    __syncthreads();
    if (n_wave >= p.KN) return;  // no barrier past this point

    // ---- multiply and store, filter tile by filter tile ------------------------------------------------------------
    const uint32_t row_bytes = (uint32_t)p.KN * 4u;
    // a buffer descriptor that ends with the tile's last live row drops the pixels past M; filters past KN get an offset out
    // of range
    const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc((void *)(p.y + (size_t)m0 * p.KN), 0,
                                                                         (int)((uint32_t)live * row_bytes), kBufferFlags);
    for (int t = 0; t < tiles; t++) {
        const int n0 = n_wave + t * 32;
        if (n0 >= p.KN) break;  // uniform over the wave
        f32x16 acc;
        int nonzero = 0;  // BTN: bits set in the nonzero plane of this lane's words of its filter
#pragma unroll
        for (int e = 0; e < 16; e++) acc[e] = 0.f;
        // btn of the lane's filter, in flight with the multiplication
        const int btn = TYPE == 2 ? p.btn[n0 + r < p.KN ? n0 + r : p.KN - 1] : 0;
        uint32_t w[NP][2 * BPL];
#pragma unroll
        for (int j = 0; j < NP; j++)
#pragma unroll
            for (int e = 0; e < 2 * BPL; e++) w[j][e] = raw[j][e];
        if (t + 1 < tiles) request_weights(t + 1);  // (of filters past KN: the last one's, unused)
#pragma unroll
        for (int j = 0; j < NP; j++) {
            const uint32_t *src = act + ((2 * j + kb) * 32 + r) * (2 * APL);
            uint32_t a[2 * APL];
            if (APL == 2) {
                const u32x4 q = *reinterpret_cast<const u32x4 *>(src);
#pragma unroll
                for (int e = 0; e < 4; e++) a[e % (2 * APL)] = q[e];
            } else {
                const u32x2 q = *reinterpret_cast<const u32x2 *>(src);
                a[0] = q[0]; a[1] = q[1];
            }
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const i32x8 af = expand_operand<TYPE, 0>(a[h], a[2 * (APL - 1) + h], consts);
                const i32x8 bf = expand_operand<TYPE, 1>(w[j][h], w[j][2 * (BPL - 1) + h], consts);
                if (TYPE == 2) nonzero += __builtin_popcount(w[j][2 * (BPL - 1) + h]);
                acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(af, bf, acc, 4, 4, 0, 0, 0, 0);
            }
        }
        if (TYPE == 0) acc *= 0.25f;  // both operands are +-2: four times the sums

        // BTN btn[f] - popcount(b1 of f), BNN NUM - 64 per word (TAB_GEMM.cu:116, 144)
        float bias = TYPE == 3 ? (float)(p.C - 64 * WORDS) : 0.f;
        if (TYPE == 2) bias = (float)(btn - (nonzero + __shfl_xor(nonzero, 32, 64)));
        const uint32_t lane_off = n0 + r < p.KN ? (uint32_t)(4 * kb) * row_bytes + (uint32_t)(n0 + r) * 4u : kNoFilter;
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int i = 0; i < 4; i++)  // accumulator element 4j+i of lane (kb, r) is pixel 8j+4kb+i, filter n0 + r
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[4 * j + i] + bias), out, lane_off + (uint32_t)(8 * j + i) * row_bytes, 0,
                                                      CACHED ? 0 : kStreamingStore);
    }
}

// Filter tiles a wave walks.  Two once a launch of three or four words a pixel is several rounds of the chip: X is then read
// (and quantized) half as often (N=128 28x28x256->512 s2 BTN 16.2 -> 13.6 us); with fewer words reading X again is cheaper
// than the longer waves (N=32 28x28x128->512 TNN 10.6 us with one tile, 12.1 with two), and four tiles gain nothing more.
int fused_tiles(int PC, long blocks, int KN) { return PC >= 3 && blocks >= 1024 && KN > 128 ? 2 : 1; }

long fused_blocks(long M, int KN) { return (M + 31) / 32 * ((KN + 127) / 128); }

template <int TYPE, int NP, bool CACHED, bool OWN>
hipError_t launch_fused_rows(const Fused1x1Args &a, hipStream_t stream)
{
    const int PC = (a.C + kWordBits - 1) / kWordBits;
    const int tiles = (int)(a.shifts_tiles >> 12);
    const dim3 grid((unsigned)((a.M + 31) / 32), (unsigned)((a.KN + 128 * tiles - 1) / (128 * tiles)));
    const unsigned lds = 2 * NP * 32 * Planes<TYPE>::A * 8;
    if (a.C % kWordBits != 0 || (uintptr_t)a.x % 16 != 0) {
        if constexpr (NP == 1) conv1x1_fused<TYPE, NP, kInputRagged, CACHED, OWN><<<grid, dim3(kConvThreads), lds, stream>>>(a);
        else return hipErrorInvalidValue;
    } else if (NP >= 2 && PC % 4 == 0) {
        if constexpr (NP >= 2) conv1x1_fused<TYPE, NP, kInputQuads, CACHED, OWN><<<grid, dim3(kConvThreads), lds, stream>>>(a);
    } else {
        conv1x1_fused<TYPE, NP, kInputWords, CACHED, OWN><<<grid, dim3(kConvThreads), lds, stream>>>(a);
    }
    return hipGetLastError();
}

template <int TYPE, bool CACHED, bool OWN>
hipError_t launch_fused_words(const Fused1x1Args &a, hipStream_t stream)
{
    const int PC = (a.C + kWordBits - 1) / kWordBits;
    if (PC <= 2) return launch_fused_rows<TYPE, 1, CACHED, OWN>(a, stream);
    if (PC <= 4) return launch_fused_rows<TYPE, 2, CACHED, OWN>(a, stream);
    return launch_fused_rows<TYPE, 4, CACHED, OWN>(a, stream);
}

template <int TYPE>
hipError_t launch_fused_type(const Fused1x1Args &a, hipStream_t stream)
{
    const bool cached = ragged_rows_cached(a.M, a.KN);
    if constexpr (Planes<TYPE>::A == 2)
        if (a.ths.splits > 0) return cached ? launch_fused_words<TYPE, true, true>(a, stream) : launch_fused_words<TYPE, false, true>(a, stream);
    return cached ? launch_fused_words<TYPE, true, false>(a, stream) : launch_fused_words<TYPE, false, false>(a, stream);
}

}  // namespace

// True when conv1x1_fused takes the call: a 1x1 kernel without padding, types 0..3, up to eight words a pixel.  A block is a
// tile of 32 pixels x 128 filters.  With one, two or four words the one launch is the faster one up to some 4096 blocks
// (beyond, the two-kernel path, whose quantizer streams X and whose conv kernel tiles the filters, is level or better).
// With more words a workgroup's serial quantizing grows (eight: N=32 28x28x512->512 34 us against 18.6 in two launches), so
// that only launches within a round of the chip save more than they lose; three words have no wide loads, and channels
// that are no whole words take 4-byte loads: both pay where the launch itself is the cost.
bool conv1x1_fused_supported(int type, const float *x, int C, int KH, int KW, int p1, int p2, long M, int KN)
{
    if (type < 0 || type > 3 || KH != 1 || KW != 1 || p1 != 0 || p2 != 0) return false;
    const int PC = (C + kWordBits - 1) / kWordBits;
    const long blocks = fused_blocks(M, KN);
    if (C % kWordBits != 0 || (uintptr_t)x % 16 != 0) return PC <= 2 && blocks <= 64;
    if (PC == 1 || PC == 2 || PC == 4) return blocks <= 4096;
    return PC <= 8 && blocks <= (PC == 8 ? 256 : 64);
}

hipError_t launch_conv1x1_fused(int type, const float *x, const Thresholds &ths, const uint64_t *qw, const int32_t *btn, float *y, int N,
                                int H, int W, int C, int KN, int s1, int s2, int OH, int OW, hipStream_t stream)
{
    Fused1x1Args a;
    a.x = x; a.qw = qw; a.btn = btn; a.y = y;
    a.H = H; a.W = W; a.C = C; a.KN = KN; a.s1 = s1; a.s2 = s2; a.pixels = OH * OW; a.OW = OW;
    a.M = N * OH * OW;
    a.ths = ordered(ths, (a.M + 31) / 32);
    const Div32 by_pixels = make_div32((uint32_t)a.pixels), by_ow = make_div32((uint32_t)OW);
    a.mul_pixels = by_pixels.mul;
    a.mul_ow = by_ow.mul;
    const uint32_t PC = (uint32_t)((C + kWordBits - 1) / kWordBits);
    a.mul_pc = (65536u + PC - 1) / PC;
    a.shifts_tiles = by_pixels.shift | by_ow.shift << 6 | (uint32_t)fused_tiles((int)PC, fused_blocks(a.M, KN), KN) << 12;
    switch (type) {
    case 0: return launch_fused_type<0>(a, stream);
    case 1: return launch_fused_type<1>(a, stream);
    case 2: return launch_fused_type<2>(a, stream);
    case 3: return launch_fused_type<3>(a, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace tab
