// Quantize + convolution in one launch for the smallest calls (all types, any kernel, stride and padding): all stages of
// ConvWithCuda_TAB (TAB_GEMM.cu:419-509), the packed activation never reaching memory.
//
// Such a call is bound by what a launch costs the host (2.4-2.8 us each) and by the instructions a wave runs one after the
// other: alone on its SIMD a wave takes some 2.5 ns per instruction, and the chip is mostly idle.  So the work is cut fine:
// a workgroup owns 16 output pixels (a block of tl lines x tc columns) and 64 filters, and
//   * its four waves quantize the patch of input pixels that block reads - "slots", row by row, padding included as zero
//     words (TAB_CPU.cpp:39,155) - into LDS, each input pixel once per workgroup;
//   * each wave multiplies the 16 pixels with its 16 filters (v_mfma_f32_16x16x128_f8f6f4: two words of K per
//     instruction, an operand is four lanes' 32 bits of one pixel or filter), the weights straight from global memory,
//     requested before the activation.
// A patch is quantized again by the workgroups of the other filters and, at its rim, of the neighbouring blocks; where that
// outweighs the saved launch the two-kernel path is taken (conv_small_supported).
#include "tab_conv_mfma_direct.h"
#include "tab_pack.h"

namespace tab {
namespace {

typedef float f32x4v __attribute__((ext_vector_type(4)));

struct SmallConvArgs {
    const float *x;
    Thresholds ths;       // of the N images
    const uint64_t *qw;   // packed weight [KN][KH][KW][PC][BPL]
    const int32_t *btn;   // [KN] (BTN only)
    float *y;             // [N*OH*OW][KN]
    int N, H, W, C, KN, OH, OW;
    uint32_t s12, p12;    // strides and paddings, 16 bits each
    uint32_t kernel;      // KH | KW << 8 | tl << 16 | tc << 24
    uint32_t magic_pw, magic_pc, magic_blocks;  // divisions by the patch width, PC and the column blocks (fastdiv)
};
static_assert(sizeof(SmallConvArgs) <= 112, "kernel arguments below 120 bytes (see ConvParams)");

// The slots of a patch.  Along an axis, outputs i and taps k share input rows (columns) where the stride is below the kernel:
// slot = i * stride + k; otherwise, and for lines of different images, every output has its own: slot = i * K + k.
__host__ __device__ __forceinline__ int slot_step(bool shared, int stride, int K) { return shared && stride < K ? stride : K; }

enum SmallInput {
    kNhwcWords = 0,   // whole 64-channel words aligned for 16-byte loads
    kNhwcRagged = 1,  // any channel count and alignment
    kNchw = 2         // [N][C][H][W]
};

// PAIRS: pairs of words of K multiplied per turn of the loop; the weights come from registers, refilled a turn ahead (WLDS
// false), or from LDS, where all of them are sent at the start (WLDS: longer K, granules of 16 bytes; with a turn of the
// registers ahead each of the N=1 14x14x256 layer's four turns waited for its own round trip).
template <int TYPE, int INPUT, int PAIRS, bool WLDS>
__global__ __launch_bounds__(kConvThreads) void conv_small(const SmallConvArgs p)
{
    // Type 5 goes like the two-plane types, over words of 64 channels: its two words of 32 fields are as long, and where
    // another lane takes 32 bits of both planes its lane takes a word, low and high half for plane 0 and 1.
    constexpr bool FIELDS = TYPE == 5;
    constexpr int APL = FIELDS ? 2 : Planes<TYPE>::A, BPL = FIELDS ? 2 : Planes<TYPE>::B;
    constexpr int MODE = TYPE > 3 ? TYPE : APL;  // ternary or binary activation, or the type's own format
    constexpr int kHalf = FIELDS ? 2 : 1, kPlane = FIELDS ? 1 : 2;  // dwords between the halves and the planes of a weight word
    // [slot][word][half][plane], then per slot its input pixel (-1: padding) and threshold, per word of K its place in a window
    extern __shared__ __attribute__((aligned(16))) uint32_t act[];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int r = lane & 15, q = lane >> 4;  // pixel or filter of a tile; which 32 bits of a pair of words this lane feeds
    const int KH = (int)(p.kernel & 255u), KW = (int)(p.kernel >> 8 & 255u), tl = (int)(p.kernel >> 16 & 255u), tc = (int)(p.kernel >> 24);
    const int s1 = (int)(p.s12 & 0xffffu), s2 = (int)(p.s12 >> 16), p1 = (int)(p.p12 & 0xffffu), p2 = (int)(p.p12 >> 16);
    const int PC = (p.C + kWordBits - 1) / kWordBits;
    const int G = KH * KW * PC;
    const int chunks = ((G + 1) / 2 + PAIRS - 1) / PAIRS;

    // ---- the block of outputs: lines line0 .. (of image n0, or of all images where they are shorter than a block) --------
    const bool own_image = p.OH >= tl;
    const int lb = (int)fastdiv(blockIdx.x, FastDiv{p.magic_blocks, p.OW <= tc ? 1u : 2u});  // (only d == 1 matters to fastdiv)
    const int cb = p.OW <= tc ? 0 : (int)blockIdx.x - lb * ((p.OW + tc - 1) / tc);
    const int n0 = own_image ? (int)blockIdx.y : 0;
    const int line0 = lb * tl, lines = own_image ? p.OH : p.N * p.OH;
    const int col0 = cb * tc;
    const int rs = slot_step(own_image, s1, KH), cs = slot_step(true, s2, KW);
    const int pw = (tc - 1) * cs + KW, ph = (tl - 1) * rs + KH;
    const int slots = pw * ph;
    const int stride = PC * 2 * APL + APL;  // dwords per slot: an odd number of elements, against bank conflicts
    int *const pixel_of = reinterpret_cast<int *>(act + slots * stride);
    float *const th_of = reinterpret_cast<float *>(pixel_of + slots);
    int *const place_of = reinterpret_cast<int *>(th_of + slots);
    const ExpandConsts consts;

    // ---- weights: the wave's filters from f0 on, pair of words j: lane (q, r) feeds half q % 2 of word 2j + q / 2 -----------
    const int f0 = (blockIdx.z * 4 + wave) * 16;
    const uint32_t *qw32 = reinterpret_cast<const uint32_t *>(p.qw);
    uint32_t raw[WLDS ? 1 : PAIRS][BPL];
    auto request_weights = [&](int j0) {
        const int f = f0 + r < p.KN ? f0 + r : p.KN - 1;  // filters past KN repeat the last one and are never stored
        const uint32_t *row = qw32 + (size_t)f * G * (2 * BPL) + (q & 1) * kHalf;
#pragma unroll
        for (int j = 0; j < PAIRS; j++) {
            const int g = 2 * (j0 + j) + (q >> 1), at = (g < G ? g : G - 1) * (2 * BPL);
#pragma unroll
            for (int pl = 0; pl < BPL; pl++) raw[j % (WLDS ? 1 : PAIRS)][pl] = row[at + kPlane * pl];
        }
    };
    // WLDS: granule k of filter f of the workgroup's 64 at ((k * 64) + f) * 16 bytes: two words of one plane or one of two
    const int granules = G * BPL / 2;
    uint32_t *const weights = act + ((slots * (stride + 2) + chunks * PAIRS * 2 + 3) & ~3);
    if constexpr (WLDS) {
        const int fw = blockIdx.z * 64 + lane;
        const size_t b_bytes = (size_t)p.KN * G * (BPL * 8);
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)p.qw, 0, (int)(uint32_t)b_bytes, kBufferFlags);
        const uint32_t row = fw < p.KN ? (uint32_t)fw * (uint32_t)(G * BPL * 8) : kNoFilter;  // (filters past KN: zeros)
        for (int k = wave; k < granules; k += 4)
            load16_to_lds(rsrc, weights + k * 256, fw < p.KN ? row + (uint32_t)k * 16u : kNoFilter);
    } else {
        request_weights(0);
    }

    // ---- tables: a thread works out a slot and a word of K once, where every load and every multiplication would again -------
    for (int slot = tid; slot < slots; slot += kConvThreads) {
        const int sr = (int)fastdiv((uint32_t)slot, FastDiv{p.magic_pw, (uint32_t)pw}), sc = slot - sr * pw;
        int line = line0, kh = sr;  // shared rows: from the block's first line on
        if (rs == KH && tl > 1) {
            line = line0 + sr / KH;
            kh = sr % KH;
        }
        int n = n0, oh = line;
        if (!own_image) {
            n = line / p.OH;
            oh = line - n * p.OH;
        }
        int ow = col0, kw = sc;
        if (cs == KW && tc > 1) {
            ow = col0 + sc / KW;
            kw = sc % KW;
        }
        const int ih = oh * s1 - p1 + kh, iw = ow * s2 - p2 + kw;
        const bool ok = line < lines && (unsigned)ih < (unsigned)p.H && (unsigned)iw < (unsigned)p.W && n < p.N;
        pixel_of[slot] = ok ? (n * p.H + ih) * p.W + iw : -1;  // < 2^31 (launch check)
        if (!own_image && p.ths.splits >= 0) th_of[slot] = lane_threshold(p.ths, ok ? n : 0);
    }
    for (int g = tid; g < chunks * PAIRS * 2; g += kConvThreads) {
        const int tap = (int)fastdiv((uint32_t)g, FastDiv{p.magic_pc, (uint32_t)PC}), kh = tap / KW;
        place_of[g] = g < G ? (kh * pw + tap - kh * KW) * stride + (g - tap * PC) * 2 * APL : 0;
    }
    const float t_image = own_image ? wave_threshold(p.ths, n0) : 0.f;
    __syncthreads();
    if constexpr (INPUT == kNhwcWords && MODE == 2) {
        if (p.ths.splits == kOwnPixelThresholds) {
            // Images of one pixel: a 16-lane row adds up |x| of its slot's image, in the order of abs_sum_partial (whose 256
            // threads take every 256th float4, i.e. every 16th word: words w, w + 16, ... in turn, then a tree over the four
            // words of a wave, then the waves), so that the thresholds are the same to the last bit.
            const int slot = wave * 4 + q;
            const int pixel = slot < slots ? pixel_of[slot] : -1;
            const float *src = p.x + (size_t)(uint32_t)(pixel < 0 ? 0 : pixel) * p.C + r * 4;
            float sum[4][4];
#pragma unroll
            for (int b = 0; b < 4; b++)
#pragma unroll
                for (int w = 0; w < 4; w++) sum[b][w] = 0.f;
            for (int w0 = 0; w0 < PC; w0 += 16)
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    if (w0 + 4 * b >= PC) break;  // uniform
#pragma unroll
                    for (int w = 0; w < 4; w++) {
                        const int word = w0 + 4 * b + w;
                        const floatx4 v = *reinterpret_cast<const floatx4 *>(src + (word < PC ? word : PC - 1) * kWordBits);
                        const float s = (__builtin_fabsf(v[0]) + __builtin_fabsf(v[1])) + (__builtin_fabsf(v[2]) + __builtin_fabsf(v[3]));
                        sum[b][w] += word < PC ? s : 0.f;
                    }
                }
            float total = 0.f;
#pragma unroll
            for (int b = 0; b < 4; b++) {
                float s = (sum[b][0] + sum[b][2]) + (sum[b][1] + sum[b][3]);
#pragma unroll
                for (int off = 8; off > 0; off >>= 1) s += __shfl_xor(s, off, 16);
                total += s;
            }
            if (r == 0 && slot < slots) th_of[slot] = (float)((double)total * p.ths.scale);
            __syncthreads();
        }
    }

    // ---- the patch ----------------------------------------------------------------------------------------------------
    if constexpr (INPUT == kNchw) {
        // unit: 64 slots (a lane each) x 16 channels of one word; the unit's bits are a quarter of the word
        const int slot_groups = (slots + 63) / 64, units = slot_groups * PC * 4;
        uint16_t *act16 = reinterpret_cast<uint16_t *>(act);
        for (int u = wave; u < units; u += 4) {
            const int quarter = u & 3, w = (u >> 2) % PC, sg = (u >> 2) / PC;
            const int slot = sg * 64 + lane;
            const int pixel = slot < slots ? pixel_of[slot] : -1;
            const int c0 = w * kWordBits + quarter * 16;
            const long HW = (long)p.H * p.W;
            const int n = own_image ? n0 : (int)((uint32_t)(pixel < 0 ? 0 : pixel) / (uint32_t)HW);
            const float *src = p.x + (pixel < 0 ? 0 : (size_t)pixel + (size_t)n * (p.C - 1) * HW);
            float v[16];
#pragma unroll
            for (int k = 0; k < 16; k++) v[k] = src[(c0 + k < p.C ? c0 + k : p.C - 1) * HW];
            const float t = own_image ? t_image : th_of[slot < slots ? slot : 0];
            uint32_t sign = 0, nz = 0;
#pragma unroll
            for (int k = 0; k < 16; k++) {
                const uint32_t bit = c0 + k < p.C ? 1u << k : 0u;
                if (MODE == 2) {
                    const bool pos = v[k] > t, neg = !pos && v[k] < -t;
                    sign |= neg ? bit : 0u;
                    nz |= pos || neg ? bit : 0u;
                } else {
                    sign |= v[k] < t ? bit : 0u;
                }
            }
            if (slot < slots) {  // 16 bits `quarter` of (half, plane)
                const int at = 2 * (slot * stride + w * 2 * APL + (quarter >> 1) * APL) + (quarter & 1);
                act16[at] = (uint16_t)(pixel < 0 ? 0u : sign);
                if (APL == 2) act16[at + 2] = (uint16_t)(pixel < 0 ? 0u : nz);
            }
        }
    } else {
        // row = slot * PC + word; a 16-lane DPP row takes one, a wave four per pass
        constexpr int LOADS = 4;  // in flight (eight: more passes past the end, 0.1-0.8 us slower)
        const int rows = slots * PC;
        for (int row0 = wave * 4 * LOADS; row0 < rows; row0 += 16 * LOADS) {
            float v[LOADS][4], t[LOADS];
            int at[LOADS], channels[LOADS];
            bool ok[LOADS];
#pragma unroll
            for (int i = 0; i < LOADS; i++) {
                const int row = row0 + 4 * i + q, row_c = row < rows ? row : rows - 1;
                const int slot = (int)fastdiv((uint32_t)row_c, FastDiv{p.magic_pc, (uint32_t)PC}), w = row_c - slot * PC;
                const int pixel = pixel_of[slot];
                ok[i] = pixel >= 0;
                at[i] = row < rows ? slot * stride + w * 2 * APL : -1;
                channels[i] = p.C - w * kWordBits;
                const float *src = p.x + (size_t)(uint32_t)(ok[i] ? pixel : 0) * p.C + w * kWordBits;
                if (INPUT == kNhwcWords) {
                    const floatx4 f = *reinterpret_cast<const floatx4 *>(src + r * 4);
#pragma unroll
                    for (int e = 0; e < 4; e++) v[i][e] = f[e];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int ch = r + 16 * e;
                        v[i][e] = src[ch < channels[i] ? ch : channels[i] - 1];
                    }
                }
                t[i] = own_image ? t_image : th_of[slot];
            }
#pragma unroll
            for (int i = 0; i < LOADS; i++) {
                uint32_t out[4];
                if (INPUT == kNhwcWords) {
                    uint32_t sign, nz;
                    compare4<MODE>(floatx4{v[i][0], v[i][1], v[i][2], v[i][3]}, t[i], sign, nz);
                    pack_row<MODE>(sign, nz, r, out);
                } else {
                    pack_row_strided<MODE>(v[i], t[i], r, channels[i], out);
                }
                if (r == 0 && at[i] >= 0) {
                    uint32_t *dst = act + at[i];
                    if (FIELDS) {
                        *reinterpret_cast<uintx2 *>(dst) = ok[i] ? uintx2{out[0], out[1]} : uintx2{0, 0};
                        *reinterpret_cast<uintx2 *>(dst + 2) = ok[i] ? uintx2{out[2], out[3]} : uintx2{0, 0};
                    } else if (APL == 2) {
                        *reinterpret_cast<uintx2 *>(dst) = ok[i] ? uintx2{out[0], out[2]} : uintx2{0, 0};
                        *reinterpret_cast<uintx2 *>(dst + 2) = ok[i] ? uintx2{out[1], out[3]} : uintx2{0, 0};
                    } else {
                        dst[0] = ok[i] ? out[0] : 0u;
                        dst[1] = ok[i] ? out[1] : 0u;
                    }
                }
            }
        }
    }
    if constexpr (WLDS) __builtin_amdgcn_s_waitcnt(0);  // this wave's granules have landed
    __syncthreads();
    if (f0 >= p.KN) return;  // no barrier past this point

    // ---- multiply ----------------------------------------------------------------------------------------------------
    const uint32_t inv_tc = (256u + (uint32_t)tc - 1) / (uint32_t)tc;  // i / tc for i below 16
    const int li = (int)((uint32_t)r * inv_tc >> 8), ci = r - li * tc;
    const uint32_t *mine = act + (r < tl * tc ? (li * rs * pw + ci * cs) * stride : 0) + (q & 1) * APL;
    f32x4v acc = {0.f, 0.f, 0.f, 0.f};
    int nonzero = 0;  // BTN: bits set in the nonzero plane of this lane's part of its filter
    for (int c = 0; c < chunks; c++) {
        uint32_t a[PAIRS][APL];
#pragma unroll
        for (int j = 0; j < PAIRS; j++) {
            const uint32_t *src = mine + place_of[2 * (c * PAIRS + j) + (q >> 1)];
            if (APL == 2) {
                const uintx2 v = *reinterpret_cast<const uintx2 *>(src);
                a[j][0] = v[0];
                a[j][APL - 1] = v[1];
            } else {
                a[j][0] = src[0];
            }
        }
        uint32_t now[PAIRS][BPL];
#pragma unroll
        for (int j = 0; j < PAIRS; j++) {
            if constexpr (WLDS) {
                const int pair = c * PAIRS + j, k = BPL == 1 ? pair : 2 * pair + (q >> 1);
                const uint32_t *src = weights + ((k < granules ? k : 0) * 64 + wave * 16 + r) * 4 + (BPL == 1 ? q : (q & 1) * kHalf);
#pragma unroll
                for (int pl = 0; pl < BPL; pl++) now[j][pl] = src[kPlane * pl];
            } else {
#pragma unroll
                for (int pl = 0; pl < BPL; pl++) now[j][pl] = raw[j % (WLDS ? 1 : PAIRS)][pl];
            }
        }
        if constexpr (!WLDS)
            if (c + 1 < chunks) request_weights((c + 1) * PAIRS);
#pragma unroll
        for (int j = 0; j < PAIRS; j++) {
            // (words past K: zeros on both sides, +64 each for binary x binary, which the bias counts)
            const bool live = 2 * (c * PAIRS + j) + (q >> 1) < G;
            const i32x8 af = expand_operand<TYPE, 0>(live ? a[j][0] : 0u, live ? a[j][APL - 1] : 0u, consts);
            const uint32_t b0 = live ? now[j][0] : 0u, b1 = live ? now[j][BPL - 1] : 0u;
            const i32x8 bf = expand_operand<TYPE, 1>(b0, b1, consts);
            if (TYPE == 2) nonzero += __builtin_popcount(b1);
            acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(af, bf, acc, 4, 4, 0, 0, 0, 0);
        }
    }

    // ---- store: element i of lane (q, r) is pixel 4q + i of the block, filter r of the tile ---------------------------------
    const int padded = chunks * PAIRS * 2;  // words of K multiplied
    const int f = f0 + r;
    // BTN btn[f] - popcount(b1 of f), BNN NUM - 64 per word (TAB_GEMM.cu:116, 144)
    float bias = TYPE == 3 ? (float)(KH * KW * p.C - 64 * padded) : 0.f;
    if (TYPE == 2) {
        int total = nonzero + __shfl_xor(nonzero, 16, 64);
        total += __shfl_xor(total, 32, 64);
        bias = (float)((f < p.KN ? p.btn[f] : 0) - total);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int px = 4 * q + i;
        const int pl = (int)((uint32_t)px * inv_tc >> 8), pcol = px - pl * tc;
        const int line = line0 + pl, col = col0 + pcol;
        if (f < p.KN && px < tl * tc && line < lines && col < p.OW)
            p.y[(((size_t)n0 * p.OH + line) * p.OW + col) * p.KN + f] = acc[i] * kSumScale<TYPE> + bias;
    }
}

int small_act_bits(int type) { return type < 2 || type > 3 ? 2 : 1; }
int small_weight_bits(int type) { return type == 1 || type == 3 ? 1 : 2; }

int small_input(const float *x, bool nchw, int C)
{
    return nchw ? kNchw : (C % kWordBits == 0 && (uintptr_t)x % 16 == 0 ? kNhwcWords : kNhwcRagged);
}

// Lines and columns of a block of 16 outputs: whole lines where they are short, else even parts of one line.
void block_of(int OW, int &tl, int &tc)
{
    if (OW >= 16) {
        const int blocks = (OW + 15) / 16;
        tl = 1;
        tc = (OW + blocks - 1) / blocks;
    } else {
        tl = 16 / OW;
        tc = OW;
    }
}

struct SmallPlan {
    int tl, tc, pw, ph, slots, stride, lines_blocks, column_blocks, images, filter_groups;
    int words, pairs;  // words of K, pairs of them per turn
    bool weights_in_lds;
    long workgroups;
    size_t lds;
};

SmallPlan plan_small(int abits, int wbits, int N, int C, int KN, int KH, int KW, int s1, int s2, int OH, int OW)
{
    SmallPlan s;
    block_of(OW, s.tl, s.tc);
    const bool own_image = OH >= s.tl;
    s.pw = (s.tc - 1) * slot_step(true, s2, KW) + KW;
    s.ph = (s.tl - 1) * slot_step(own_image, s1, KH) + KH;
    s.slots = s.pw * s.ph;
    const int PC = (C + kWordBits - 1) / kWordBits;
    s.stride = PC * 2 * abits + abits;
    const int G = KH * KW * PC;
    s.words = G;
    s.weights_in_lds = G > 10 && (wbits == 2 || G % 2 == 0);
    s.pairs = G <= 2 ? 1 : (G <= 10 ? 5 : (s.weights_in_lds ? 6 : 9));
    const size_t words = ((size_t)(G + 1) / 2 + s.pairs - 1) / s.pairs * s.pairs * 2;
    s.lds = (((size_t)s.slots * (s.stride + 2) + words + 3) & ~(size_t)3) * 4 + (s.weights_in_lds ? (size_t)64 * G * wbits * 8 : 0);
    const long lines = own_image ? OH : (long)N * OH;
    s.lines_blocks = (int)((lines + s.tl - 1) / s.tl);
    s.column_blocks = (OW + s.tc - 1) / s.tc;
    s.images = own_image ? N : 1;
    s.filter_groups = (KN + 63) / 64;
    s.workgroups = (long)s.lines_blocks * s.column_blocks * s.images * s.filter_groups;
    return s;
}

template <int TYPE, int INPUT>
hipError_t launch_small(const SmallConvArgs &a, const SmallPlan &s, hipStream_t stream)
{
    const dim3 grid((unsigned)(s.lines_blocks * s.column_blocks), (unsigned)s.images, (unsigned)s.filter_groups), block(kConvThreads);
    if (s.weights_in_lds) conv_small<TYPE, INPUT, 6, true><<<grid, block, s.lds, stream>>>(a);
    else if (s.pairs == 1) conv_small<TYPE, INPUT, 1, false><<<grid, block, s.lds, stream>>>(a);
    else if (s.pairs == 5) conv_small<TYPE, INPUT, 5, false><<<grid, block, s.lds, stream>>>(a);
    else conv_small<TYPE, INPUT, 9, false><<<grid, block, s.lds, stream>>>(a);
    return hipGetLastError();
}

// What a launch's duration is made of: a wave's passes over the patch, its pairs of words of K, and how many workgroups a CU gets
// beyond the first, which run at the rate of waves that share a SIMD.  A two-plane activation costs half as much again to pack,
// channels that are no whole words nearly twice.  Against the measured duration in graph replays (conv_small_timings.txt) the
// prediction is off by 7 % in the median on 306 NHWC calls (5 % too low on average) and by 19 %, too low, on 64 NCHW ones.
struct SmallCost {
    float passes, pairs, more;
    float us() const { return 3.7f + 0.075f * passes + 0.062f * pairs + more * (0.033f * passes + 0.044f * pairs + 0.32f); }
};

SmallCost small_cost(const SmallPlan &s, int abits, int wbits, int PC, int input)
{
    SmallCost c;
    c.passes = (float)((s.slots * PC + 63) / 64 * 4) * (abits == 2 ? 1.5f : 1.f);
    if (input == kNhwcRagged) c.passes *= 1.8f;
    if (input == kNchw) c.passes = (float)((s.slots + 63) / 64 * PC) * (abits == 2 ? 4.f : 3.f);
    c.pairs = (float)((((s.words + 1) / 2) + s.pairs - 1) / s.pairs * s.pairs) * 0.5f * (float)(abits + wbits);
    const float cus = (float)device_compute_units();
    c.more = (float)s.workgroups > cus ? (float)s.workgroups / cus - 1.f : 0.f;
    return c;
}

}  // namespace

// True when conv_small takes the call.  Two launches cost the host 5 us and the GPU 5 us or more at any size; called one after
// the other from Python, calls on NHWC take 8.4-8.7 us in two launches and 5.3-6.3 in this one where it is taken.  The limit lies
// between what suits such callers (420 measured calls of random geometry, time as a share of always two launches: 82 % at 5.5 us,
// 78 % at 6.3, 77 % from 6.6 on; with the better choice of each 76 %) and graph replays, where a launch costs the host nothing
// (94, 95, 96 and from 8 us on 100 %; 93 %).  tab_amd/tuning/check_conv_small_cost.py prints this from the timings beside it.
// Of the 1x1 layers it is left those that conv1x1_fused does not take, within one workgroup a CU.
bool conv_small_supported(int type, const float *x, bool nchw, int N, int H, int W, int C, int KN, int KH, int KW, int p1, int p2, int s1,
                          int s2, int OH, int OW)
{
    constexpr float kMostUs = 6.3f;
    float cost[4];
    return conv_small_cost(type, x, nchw, N, H, W, C, KN, KH, KW, p1, p2, s1, s2, OH, OW, cost) && cost[0] <= kMostUs;
}

bool conv_small_cost(int type, const float *x, bool nchw, int N, int H, int W, int C, int KN, int KH, int KW, int p1, int p2, int s1, int s2,
                     int OH, int OW, float (&cost)[4])
{
    // (type 5: the two words of every 64 channels exist)
    if (type < 0 || type > 5 || (type > 3 && nchw) || (type == 5 && (C + 31) / 32 % 2 != 0) || KH > 255 || KW > 255 || s1 > 65535 || s2 > 65535 || p1 > 65535 || p2 > 65535 || N > 65535) return false;
    if ((long)N * H * W * C > (4L << 20) || (long)N * OH * OW > 65535) return false;  // no need to plan for these
    const int PC = (C + kWordBits - 1) / kWordBits, abits = small_act_bits(type), wbits = small_weight_bits(type);
    const SmallPlan s = plan_small(abits, wbits, N, C, KN, KH, KW, s1, s2, OH, OW);
    if (s.lds > 64 * 1024 || (long)s.slots * PC >= 65536 || (long)s.lines_blocks * s.column_blocks >= 65536 || s.filter_groups > 65535 ||
        (size_t)KN * s.words * 16 >= kNoFilter)
        return false;
    if (KH * KW == 1 && s.workgroups > device_compute_units()) return false;
    const SmallCost c = small_cost(s, abits, wbits, PC, small_input(x, nchw, C));
    cost[0] = c.us();
    cost[1] = c.passes;
    cost[2] = c.pairs;
    cost[3] = c.more;
    return true;
}

// A workgroup's outputs lie in one image (then its waves add up an image's partial sums together).
bool conv_small_in_one_image(int OH, int OW)
{
    int tl, tc;
    block_of(OW, tl, tc);
    return OH >= tl;
}

bool conv_small_own_thresholds(const float *x, int H, int W, int C, int KH, int KW, int p1, int p2)
{
    // (an image of more than 4096 channels may be summed in several slices)
    return H == 1 && W == 1 && KH == 1 && KW == 1 && p1 == 0 && p2 == 0 && C <= 4096 && small_input(x, false, C) == kNhwcWords &&
           threshold_splits(1, C) == 1;
}

hipError_t launch_conv_small(int type, const float *x, bool nchw, const Thresholds &ths, const uint64_t *qw, const int32_t *btn, float *y,
                             int N, int H, int W, int C, int KN, int KH, int KW, int p1, int p2, int s1, int s2, int OH, int OW,
                             hipStream_t stream)
{
    const SmallPlan s = plan_small(small_act_bits(type), small_weight_bits(type), N, C, KN, KH, KW, s1, s2, OH, OW);
    const int PC = (C + kWordBits - 1) / kWordBits;
    SmallConvArgs a;
    a.x = x; a.ths = ths; a.qw = qw; a.btn = btn; a.y = y;
    a.N = N; a.H = H; a.W = W; a.C = C; a.KN = KN; a.OH = OH; a.OW = OW;
    a.s12 = (uint32_t)s1 | (uint32_t)s2 << 16;
    a.p12 = (uint32_t)p1 | (uint32_t)p2 << 16;
    a.kernel = (uint32_t)KH | (uint32_t)KW << 8 | (uint32_t)s.tl << 16 | (uint32_t)s.tc << 24;
    a.magic_pw = make_fastdiv((uint32_t)s.pw).magic;
    a.magic_pc = make_fastdiv((uint32_t)PC).magic;
    a.magic_blocks = make_fastdiv((uint32_t)s.column_blocks).magic;
    const int input = small_input(x, nchw, C);
    auto by_input = [&](auto t) {
        constexpr int TYPE = decltype(t)::value;
        if constexpr (TYPE <= 3)
            if (input == kNchw) return launch_small<TYPE, kNchw>(a, s, stream);
        if (input == kNhwcWords) return launch_small<TYPE, kNhwcWords>(a, s, stream);
        return launch_small<TYPE, kNhwcRagged>(a, s, stream);
    };
    switch (type) {
    case 0: return by_input(std::integral_constant<int, 0>());
    case 1: return by_input(std::integral_constant<int, 1>());
    case 2: return by_input(std::integral_constant<int, 2>());
    case 3: return by_input(std::integral_constant<int, 3>());
    case 4: return by_input(std::integral_constant<int, 4>());
    case 5: return by_input(std::integral_constant<int, 5>());
    default: return hipErrorInvalidValue;
    }
}

}  // namespace tab
