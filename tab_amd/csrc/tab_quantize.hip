// Quantizer / bit-packer for gfx950 (wave64): fp32 NHWC -> packed int64 bit planes.
//
// Semantics follow the reference kernels TerOnlyKernel (TAB_GEMM.cu:163-208) and
// BinOnlyKernel (TAB_GEMM.cu:211-247) with the per-item threshold ths[n] of the CPU path
// (TAB_CPU.cpp:67,72), plus BTN_Weight (TAB_GEMM.cu:150-160) for every item.
//
// The tensor is a sequence of "rows" of 64 consecutive channels; row r becomes packed
// word r (C % 64 == 0) so the whole op is one streaming pass: 256 B in, 8 or 16 B out.
#include "tab_conv_stage.h"
#include "tab_pack.h"
#include "tab_quantize_rows.h"
#include "tab_patch_weights.h"

namespace tab {
namespace {

constexpr int kThreads = 256;
constexpr int kWavesPerBlock = kThreads / 64;
constexpr int kRowsPerWave = 4 * kLoadsPerLane; // each wave-wide float4 load covers 4 rows
// LDS that the streaming launches of quantize_rows64 ask for and do not use: seven workgroups on a CU, where registers would let eight.
// Their reads then follow each other more closely in memory: 822 MB of one plane 136.6 -> 134.1 us, of two 148.0 -> 145.8; six are as fast
// there, but 54 MB, 1636 workgroups, are a second round for them (10.4 -> 11.1).
constexpr int kStreamLds = 22 << 10;

constexpr long kSmallLaunchBlocks = 512;        // at or below this many 128-row workgroups a launch is latency-bound

__device__ __forceinline__ int wave_sum(int v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

// The counts of items 0 .. items - 1 start at zero (for one plane they stay there, TAB_GEMM.cu:283).  Every quantizer
// writes them on the side, since a launch of its own for them costs 1.2-4.8 us before the quantizer: a lane takes the
// counts with the numbers of `n` rows (or pixels) of its own, of which there are at least as many as items.  At the end of
// the kernel, so that nothing waits for the argument.  Null: none wanted.
__device__ __forceinline__ void zero_counts(int32_t *btn, long items, long first, int n = 1)
{
    if (btn == nullptr) return;
    for (int i = 0; i < n; i++)
        if (first + i < items) btn[first + i] = 0;
}

// Counts of nonzero values made by the quantizer itself (template parameter COUNT, two planes): each item is cut into
// `slices` workgroups, a workgroup takes the slice's units (what it quantizes in one go) `slices` apart and stores their
// count, in btn where an item is one slice, else in a workspace from where count_finish adds the slices up.  Reading the packed
// output back for the counts instead took a launch of 4.8-9.6 us behind every two-plane quantizer, a third of the whole for
// tensors of 10-20 MB.
struct Counts {
    int32_t *out;  // [items * slices]
    int slices;
};

// The sum of `count` over the workgroup, stored by one thread.  scratch: a dword per wave, free to overwrite.
template <int WAVES>
__device__ __forceinline__ void store_count(int count, int32_t *out, int32_t *scratch)
{
    count = wave_sum(count);
    if (WAVES == 1) {
        if (threadIdx.x == 0) *out = count;
        return;
    }
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = count;
    __syncthreads();
    if (threadIdx.x == 0) {
        int total = 0;
#pragma unroll
        for (int w = 0; w < WAVES; w++) total += scratch[w];
        *out = total;
    }
}

// One workgroup per item; four counts in flight a thread (one wave with a count at a time took 5 us for 700).
__global__ __launch_bounds__(kThreads) void count_finish(const int32_t *__restrict__ counts, int32_t *__restrict__ btn, int slices)
{
    __shared__ int32_t scratch[kWavesPerBlock];
    const int32_t *src = counts + (long)blockIdx.x * slices;
    int count = 0;
    for (int i = threadIdx.x; i < slices; i += 4 * kThreads) {
        int32_t v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = src[i + u * kThreads < slices ? i + u * kThreads : i];
#pragma unroll
        for (int u = 0; u < 4; u++) count += i + u * kThreads < slices ? v[u] : 0;
    }
    store_count<kWavesPerBlock>(count, btn + blockIdx.x, scratch);
}

// The streaming path (tab_quantize_rows.h).
template <int BITS, int LOADS = kLoadsPerLane, bool OWN = false>
__global__ __launch_bounds__(kThreads) void quantize_rows64(const floatx4 *__restrict__ x, const Thresholds ths, uint32_t *__restrict__ q, long rows,
                                                            long rows_per_item, Div32 div_item, int32_t *btn, long items)
{
    quantize_rows_block<BITS, LOADS, OWN>(WholeRows{}, x, ths, q, rows, rows_per_item, div_item, OWN ? in_eighths(blockIdx.x, ths.eighth) : blockIdx.x);
    const long row = (long)blockIdx.x * (4 * LOADS * kWavesPerBlock) + (threadIdx.x >> 6) * (4 * LOADS) + (threadIdx.x & 63);
    if ((threadIdx.x & 63) < 4 * LOADS) zero_counts(btn, items, row);
}

// Beside a convolution's weights, which the first workgroups lay out (kernels of their own: with the code for the weights in every
// quantizer the short ones took 2-4 % longer).
template <int BITS, int LOADS = kLoadsPerLane, bool OWN = false>
__global__ __launch_bounds__(kThreads) void quantize_rows64_weights(const floatx4 *__restrict__ x, const Thresholds ths, uint32_t *__restrict__ q,
                                                                    long rows, long rows_per_item, Div32 div_item, const WeightJob job)
{
    uint32_t block = blockIdx.x;
    if (pack_weights<kThreads>(job, block)) return;
    quantize_rows_block<BITS, LOADS, OWN>(WholeRows{}, x, ths, q, rows, rows_per_item, div_item, OWN ? in_eighths(block, ths.eighth) : block);
}

// The same for any channel count and any alignment of x.  Bound like quantize_rows64 by reading x, and by the lanes that a pixel's last
// row leaves without channels.  A tile of pixels sent through LDS, which took these tensors before, waited for its whole run and went
// over the pixels of a wave word after word (one plane / two, before -> now, us): C=100 2 MB 4.3 / 4.7 -> 2.4 / 2.5, 8 MB 4.6 / 5.2 -> 3.0 / 3.3, 60
// MB 13.0 / 14.9 -> 11.3 / 12.7, 300 MB 54.6 / 57.7 -> 49.6 / 54.5 (6.0 TB/s); C=494 8 MB 7.1 / 8.4 -> 2.9 / 3.1; C=1000 2 MB 8.2 / 9.8 -> 2.4 / 2.5,
// 300 MB 121 / 147 -> 49 / 53.  32 rows a workgroup or 128 as for whole rows (C=100, 8 MB 3.0 / 4.0, 20 MB 5.8 / 5.8, 60 MB 12.4 / 11.3).
// Format 5 is the one bound by its instructions: with the addresses of its words from the wave's first and its fields spread two operations at a time 120 MB
// of C=33 take 30.8 us, 36.1 without, 33.6 by tiles.
template <int BITS, int LOADS = kLoadsPerLane, bool OWN = false>
__global__ __launch_bounds__(kThreads) void quantize_rows_ragged(const floatx4 *__restrict__ x, const Thresholds ths, uint32_t *__restrict__ q, long rows,
                                                                 long rows_per_item, Div32 div_item, int32_t *btn, long items, const RaggedRows ragged)
{
    quantize_rows_block<BITS, LOADS, OWN>(ragged, x, ths, q, rows, rows_per_item, div_item, OWN ? in_eighths(blockIdx.x, ths.eighth) : blockIdx.x);
    const long row = (long)blockIdx.x * (4 * LOADS * kWavesPerBlock) + (threadIdx.x >> 6) * (4 * LOADS) + (threadIdx.x & 63);
    if ((threadIdx.x & 63) < 4 * LOADS) zero_counts(btn, items, row);
}

template <int BITS, int LOADS = kLoadsPerLane, bool OWN = false>
__global__ __launch_bounds__(kThreads) void quantize_rows_ragged_weights(const floatx4 *__restrict__ x, const Thresholds ths, uint32_t *__restrict__ q,
                                                                         long rows, long rows_per_item, Div32 div_item, const RaggedRows ragged,
                                                                         const WeightJob job)
{
    uint32_t block = blockIdx.x;
    if (pack_weights<kThreads>(job, block)) return;
    quantize_rows_block<BITS, LOADS, OWN>(ragged, x, ths, q, rows, rows_per_item, div_item, OWN ? in_eighths(block, ths.eighth) : block);
}

// The row quantizer for a 1x1 convolution with stride and no padding, which reads only the
// pixels (oh*s1, ow*s2): one wave per 4*LOADS consecutive words of one output line (n, oh); the packed
// result is the compact [N][OH][OW][PC] activation, i.e. what the conv reads with stride 1.
// grid = (ceil(OW*PC / (4*LOADS)), N*OH), one wave per workgroup; OW*PC < 65536 (fastdiv range).
template <int BITS, int LOADS = kLoadsPerLane>
__global__ __launch_bounds__(64) void quantize_rows64_strided(const floatx4 *__restrict__ x, const Thresholds ths,
                                                              uint32_t *__restrict__ q, int H, int W, int PC, int OH,
                                                              int OW, int s1, int s2, FastDiv div_pc)
{
    const int lane = threadIdx.x;
    const int sub = lane >> 4, l = lane & 15;
    const int n = blockIdx.y / OH, oh = blockIdx.y - n * OH;  // uniform
    const int line_words = OW * PC;
    const long in_line = ((long)n * H + (long)oh * s1) * W;   // first input pixel of the line
    const long out_line = (long)blockIdx.y * line_words;
    const int j0 = blockIdx.x * (4 * LOADS);

    floatx4 v[LOADS];
#pragma unroll
    for (int u = 0; u < LOADS; u++) {
        const int j = min(j0 + u * 4 + sub, line_words - 1);  // words past the line read its last word again (not stored)
        const int ow = (int)fastdiv((uint32_t)j, div_pc), pc = j - ow * PC;
        const long r = (in_line + (long)ow * s2) * PC + pc;
        v[u] = LOADS == 2 ? x[r * 16 + l] : __builtin_nontemporal_load(&x[r * 16 + l]);
    }
    const float t = wave_threshold(ths, n);
#pragma unroll
    for (int u = 0; u < LOADS; u++) {
        const int j = j0 + u * 4 + sub;
        const long r = out_line + j;
        uint32_t sign, nz, out[4];
        compare4<BITS>(v[u], t, sign, nz);
        pack_row<BITS>(sign, nz, l, out);
        if (BITS != 1) {
            if (j < line_words && l == 0) *reinterpret_cast<uintx4 *>(q + r * 4) = uintx4{out[0], out[1], out[2], out[3]};
        } else {
            if (j < line_words && l == 0) *reinterpret_cast<uintx2 *>(q + r * 2) = uintx2{out[0], out[1]};
        }
    }
}

// Two planes with counts (see Counts): a slice is one unit, 4 * LOADS rows of every wave.
template <int LOADS, bool NT, class Rows>
__device__ __forceinline__ void quantize_rows_counted(const Rows kind, const floatx4 *__restrict__ x, const Thresholds &ths, uint32_t *__restrict__ q,
                                                      long rows_per_item, const Counts &counts, int32_t *scratch)
{
    constexpr int UNIT = 4 * LOADS * kWavesPerBlock;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sub = lane >> 4, l = lane & 15;
    const int item = (int)(blockIdx.x / (uint32_t)counts.slices), slice = (int)blockIdx.x - item * counts.slices;
    int count = 0;
    const long at = (long)slice * UNIT + wave * (4 * LOADS);  // of the item's rows
    if (at < rows_per_item) {
        const long first = item * rows_per_item + at;
        const uint32_t live = (uint32_t)(rows_per_item - at < 4 * LOADS ? rows_per_item - at : 4 * LOADS);
        RowLoads<LOADS> held;
        load_rows<NT>(kind, x, first, live, sub, l, held);
        const float t = given_threshold(ths, item);
#pragma unroll
        for (int u = 0; u < LOADS; u++) {
            const uint32_t r = u * 4 + sub;
            uint32_t sign, nz, out[4];
            compare4<2>(held.v[u], t, sign, nz);
            if (std::is_same<Rows, RaggedRows>::value) {
                sign &= held.exist[u];
                nz &= held.exist[u];
            }
            count += r < live ? __builtin_popcount(nz) : 0;
            pack_row<2>(sign, nz, l, out);
            if (r < live && l == 0) *reinterpret_cast<uintx4 *>(q + (first + r) * 4) = uintx4{out[0], out[1], out[2], out[3]};
        }
    }
    store_count<kWavesPerBlock>(count, counts.out + blockIdx.x, scratch);
}

template <int LOADS, bool NT>
__global__ __launch_bounds__(kThreads) void quantize_rows64_count(const floatx4 *__restrict__ x, const Thresholds ths, uint32_t *__restrict__ q,
                                                                  long rows_per_item, const Counts counts)
{
    __shared__ int32_t scratch[kWavesPerBlock];
    quantize_rows_counted<LOADS, NT>(WholeRows{}, x, ths, q, rows_per_item, counts, scratch);
}

template <int LOADS, bool NT>
__global__ __launch_bounds__(kThreads) void quantize_rows_ragged_count(const floatx4 *__restrict__ x, const Thresholds ths, uint32_t *__restrict__ q,
                                                                       long rows_per_item, const Counts counts, const RaggedRows ragged)
{
    __shared__ int32_t scratch[kWavesPerBlock];
    quantize_rows_counted<LOADS, NT>(ragged, x, ths, q, rows_per_item, counts, scratch);
}

// A convolution's weights alone.
__global__ __launch_bounds__(kThreads) void patch_weights(const WeightJob job)
{
    uint32_t block = blockIdx.x;
    pack_weights<kThreads>(job, block);
}

// Up to 32 channels, any alignment of x, every format (MODE as in compare4), where a row of 16 lanes a pixel would be mostly empty: a
// workgroup takes a tile of consecutive pixels,
// whose channels are one contiguous run of x, sends the run to LDS in granules of 16 bytes, and its waves then read the words
// out of it: LP lanes a word (the smallest power of two that holds it; 64 / LP pixels a read), so
// that one compare makes the bits of a whole read as a wave mask (LSB first; onebit[i] = 1 << i, TAB_GEMM.cu:252-258).  Lane
// i keeps the word of the wave's pixel i.  Unused high bits of a tail word stay 0
// (TAB_GEMM.cu:203-206).
// Bound by reading x and by the waits of a tile for its run: the 16-byte loads do not care where pixels begin, and a word costs
// six to twelve instructions.  Against 4-byte loads a lane and row, ORed together over the lanes of a word (one plane / two, us):
// 64x112x112x32 31 / 33 -> 18.0 / 18.6, 64x224x224x3 19.3 / 25.0 -> 13.3 / 16.8; 60 MB against rows of 16 lanes (quantize_rows_ragged):
// C=5 68 / 85 -> 16.5 / 20.7, C=27 15.2 / 18.3 -> 11.8 / 13.2.
// Formats 4 and 5 belong to the CPU-only conv types, whose layouts follow from the reference's GEMMs (it has no quantizer for
// them: TAB_Conv calls Parallel_Binarize_NCHW and Parallel_Ternarize_RTN, TAB_CPU.cpp:522,527, which no file defines):
// 4, DoReFa 2-bit (DRFGEMM_baseline, TAB_CPU.cpp:345-354): [pixel][ceil(C/64)][2], plane 0 the weight-2 bit and plane 1 the
//    weight-1 bit of level = (v >= 0.5t) + (v >= 1.5t) + (v >= 2.5t);
// 5, RTN (RTNGEMM_baseline, TAB_CPU.cpp:364-379; 32 channels per word, 520-521): [pixel][ceil(C/32)], channel c in word c/32
//    as the field (bit 2*(c%32) = nonzero, bit 2*(c%32)+1 = sign) of the ternarizer's value.
// One tile: `live` pixels from p0 on.  Returns how many of the values this lane stored are nonzero (MODE 2).
template <int MODE, int LP>
__device__ __forceinline__ int quantize_one_tile(const float *__restrict__ x, const Thresholds &ths, uint64_t *__restrict__ q, long p0, int live,
                                                 long pixels_per_item, Div32 div_item, int C, int tile_pixels)
{
    static_assert(LP <= 32, "a word of 32 bits or less");
    constexpr int G = 64 / LP;  // rows per read
    constexpr int U = 2;        // reads in flight
    extern __shared__ __attribute__((aligned(16))) uint32_t tile[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int count = 0;

    // ---- the run of x, from the 16-byte boundary at or below its start to its last float ----------------------------------
    const uintptr_t start = (uintptr_t)(x + p0 * C);
    const int skew = (int)(start & 15) / 4;  // floats
    const int floats = live * C + skew;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(start & ~(uintptr_t)15), 0, floats * 4, kBufferFlags);
    for (int i = wave * 64; i * 4 < floats; i += kThreads) load16_to_lds(rsrc, tile + i * 4, (uint32_t)(i + lane) * 16u);

    // ---- thresholds: one for the tile, or a table behind the run ---------------------------------------------------------------
    auto item_of = [&](long pixel) { return div_item.mul ? (long)div32((uint32_t)pixel, div_item) : pixel / pixels_per_item; };
    const long item_first = item_of(p0);
    const bool one_item = item_of(p0 + live - 1) == item_first;
    float *const th = reinterpret_cast<float *>(tile + (tile_pixels * C + 3 + 3) / 4 * 4 + 256);
    const float t_first = wave_threshold(ths, item_first);
    if (!one_item)
        for (int i0 = wave * 64; i0 < live; i0 += kThreads) {
            const long item = item_of(p0 + min(i0 + lane, live - 1));
            const long first = item_of(p0 + i0), last = item_of(p0 + min(i0 + 63, live - 1));
            const float t = MODE == 2 && ths.splits > 0 ? span_threshold(ths, item, first, last, request_threshold(ths, first)) : given_threshold(ths, item);
            if (i0 + lane < live) th[i0 + lane] = t;
        }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();

    // ---- words: the wave's pixels of the tile, 64 at a time; a read takes G of them -------------------------------------------------
    const int share = ((live + 3) / 4 + G - 1) / G * G;
    const int end = min(live, (wave + 1) * share);
    const float *const run = reinterpret_cast<const float *>(tile) + skew;
    const int ch = lane % LP;
    const uint64_t exist = __ballot(ch < C);
    for (int px0 = wave * share; px0 < end; px0 += 64) {
        const float *src = run + px0 * C + (lane / LP) * C + min(ch, C - 1);
        const int reads = (min(end - px0, 64) + G - 1) / G;
        uint32_t out0 = 0, out1 = 0;  // the planes' low halves of pixel px0 + lane; the high ones are zero
        for (int j0 = 0; j0 < reads; j0 += U) {
            float v[U], t[U];
#pragma unroll
            for (int u = 0; u < U; u++) {  // (reads past the tile's last pixel: that of the first, kept by no lane)
                const bool past = px0 + (j0 + u) * G + lane / LP >= live;
                v[u] = src[past ? 0 : (j0 + u) * G * C];
                t[u] = one_item ? t_first : th[past ? 0 : px0 + (j0 + u) * G + lane / LP];
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                uint64_t m0, m1 = 0;
                if (MODE == 1) {
                    m0 = __ballot(v[u] < t[u]) & exist;
                } else if (MODE == 4) {
                    const uint64_t l1 = __ballot(v[u] >= 0.5f * t[u]), l2 = __ballot(v[u] >= 1.5f * t[u]), l3 = __ballot(v[u] >= 2.5f * t[u]);
                    // level = number of bounds reached, whatever their order (t may be negative)
                    m0 = ((l1 & l2) | (l1 & l3) | (l2 & l3)) & exist;
                    m1 = (l1 ^ l2 ^ l3) & exist;
                } else {
                    const uint64_t pos = __ballot(v[u] > t[u]);
                    m0 = __ballot(v[u] < -t[u]) & ~pos & exist;
                    m1 = (pos & exist) | m0;
                }
                // lane j * G + g keeps the LP bits of the read's pixel g
                const bool mine = lane / G == j0 + u;
                const int shift = LP * (lane % G);
                constexpr uint32_t bits = LP >= 32 ? ~0u : (1u << (LP & 31)) - 1;
                out0 = mine ? (uint32_t)(m0 >> shift) & bits : out0;
                if (MODE != 1) out1 = mine ? (uint32_t)(m1 >> shift) & bits : out1;
            }
        }
        if (px0 + lane < end) {
            const size_t pixel = (size_t)p0 + px0 + lane;
            if (MODE == 1) {
                *reinterpret_cast<uintx2 *>(q + pixel) = uintx2{out0, 0};
            } else if (MODE == 5) {
                q[pixel] = spread_bits(out1) | spread_bits(out0) << 1;  // one word of 32 fields
            } else {
                *reinterpret_cast<uintx4 *>(q + 2 * pixel) = uintx4{out0, 0, out1, 0};
                if (MODE == 2) count += __builtin_popcount(out1);
            }
        }
    }
    return count;
}

template <int MODE, int LP>
__global__ __launch_bounds__(kThreads) void quantize_tile(const float *__restrict__ x, const Thresholds ths, uint64_t *__restrict__ q,
                                                          long pixels, long pixels_per_item, Div32 div_item, int C, int tile_pixels,
                                                          int32_t *btn, long items)
{
    const long p0 = (long)in_eighths(blockIdx.x, ths.eighth) * tile_pixels;
    const int live = pixels - p0 < tile_pixels ? (int)(pixels - p0) : tile_pixels;  // pixels of the tile that exist
    quantize_one_tile<MODE, LP>(x, ths, q, p0, live, pixels_per_item, div_item, C, tile_pixels);
    for (int i = threadIdx.x; i < live; i += kThreads) zero_counts(btn, items, p0 + i);
}

// Without counts, beside a convolution's weights.
template <int MODE, int LP>
__global__ __launch_bounds__(kThreads) void quantize_tile_weights(const float *__restrict__ x, const Thresholds ths, uint64_t *__restrict__ q,
                                                                  long pixels, long pixels_per_item, Div32 div_item, int C, int tile_pixels,
                                                                  const WeightJob job)
{
    uint32_t block = blockIdx.x;
    if (pack_weights<kThreads>(job, block)) return;
    const long p0 = (long)in_eighths(block, ths.eighth) * tile_pixels;
    const int live = pixels - p0 < tile_pixels ? (int)(pixels - p0) : tile_pixels;  // pixels of the tile that exist
    quantize_one_tile<MODE, LP>(x, ths, q, p0, live, pixels_per_item, div_item, C, tile_pixels);
}

// The same with counts (see Counts); a unit is a tile of whole pixels.
template <int LP>
__global__ __launch_bounds__(kThreads) void quantize_tile_count(const float *__restrict__ x, const Thresholds ths, uint64_t *__restrict__ q,
                                                                long pixels_per_item, Div32 div_item, int C, int tile_pixels, const Counts counts)
{
    __shared__ int32_t scratch[kWavesPerBlock];
    const int item = (int)(blockIdx.x / (uint32_t)counts.slices), slice = (int)blockIdx.x - item * counts.slices;
    int count = 0;
    for (long at = (long)slice * tile_pixels; at < pixels_per_item; at += (long)counts.slices * tile_pixels) {
        const int live = pixels_per_item - at < tile_pixels ? (int)(pixels_per_item - at) : tile_pixels;
        if (at >= (long)counts.slices * tile_pixels) __syncthreads();  // the waves have read the tile before
        count += quantize_one_tile<2, LP>(x, ths, q, item * pixels_per_item + at, live, pixels_per_item, div_item, C, tile_pixels);
    }
    store_count<kWavesPerBlock>(count, counts.out + blockIdx.x, scratch);
}

// The same quantizers on an NCHW tensor, the layout the reference's CPU quantizers read
// (Parallel_Ternarize_NCHWB_to_NHWCB / Parallel_Binarize_NCHW_to_NHWC, TAB_CPU.cpp:20-206), into the same NHWC
// packed output.  A thread owns a run of VEC consecutive pixels of one image and a part of a word's channels: each load is
// VEC floats of one channel plane (consecutive threads read consecutive pixels of the plane, so every load instruction is
// contiguous), and each compare shifts its bit into the words the thread holds in registers: no cross-lane step at all.
// An image of H*W pixels is ceil(H*W / VEC) runs; where VEC does not divide H*W the last one is moved back to end with the
// image and overlaps the one before it (the same words are then written twice).  Planes of odd sizes so take the same 16-byte
// loads, which need 4-byte alignment only, as even ones: with one pixel a thread 55x55 planes were read at 4 TB/s.
template <int VEC, bool EVEN = false>
struct PixelRun {
    typedef float Vec __attribute__((ext_vector_type(VEC)));
    typedef Vec VecAnywhere __attribute__((aligned(4)));
    long n, s, pixel;  // image, first pixel in the image, first pixel counted through all images
    int repeated;      // pixels at the run's start that the run before it has too (the per-image numbering only)

    // run `i` counted through all images; past the last one: the last one again, with the same results.  by_image divides by
    // the pixels of an image (EVEN) or its runs; mul == 0 says that they reach 2^31 and the division takes 64 bits, which every
    // wave waits for before it can request a pixel
    __device__ __forceinline__ PixelRun(long i, int N, long HW, Div32 by_image) : repeated(0)
    {
        if (EVEN) {
            const long total = N * HW;
            pixel = i * VEC < total ? i * VEC : total - VEC;
            n = by_image.mul ? (long)div32((uint32_t)pixel, by_image) : pixel / HW;
            s = pixel - n * HW;
        } else {
            const long per_image = (HW + VEC - 1) / VEC;
            const long runs = N * per_image;
            if (i >= runs) i = runs - 1;
            n = by_image.mul ? (long)div32((uint32_t)i, by_image) : i / per_image;
            s = (i - n * per_image) * VEC;
            if (s > HW - VEC) s = HW - VEC;
            pixel = n * HW + s;
        }
    }
    // run `i` of image `image`
    __device__ __forceinline__ PixelRun(long i, long image, long HW, std::true_type)
    {
        n = image;
        s = i * VEC < HW - VEC ? i * VEC : HW - VEC;
        pixel = n * HW + s;
        repeated = i * VEC - s < VEC ? (int)(i * VEC - s) : VEC;
    }
    template <bool NT = false>
    __device__ __forceinline__ void load(float (&v)[VEC], const float *src) const
    {
        if constexpr (VEC == 1) {
            v[0] = *src;
        } else {
            const VecAnywhere *at = reinterpret_cast<const VecAnywhere *>(src);
            const Vec w = NT ? __builtin_nontemporal_load(at) : *at;
#pragma unroll
            for (int e = 0; e < VEC; e++) v[e] = w[e];
        }
    }
    // the thread's threshold in two steps (every lane active): the partial sums of the wave's first image are requested before the pixels.
    // OWN: it may have to be added up (layers of two planes); ONE: the workgroup has one image
    template <bool OWN>
    __device__ __forceinline__ floatx4 request(const Thresholds &ths) const
    {
        return OWN && ths.splits > 0 ? request_threshold(ths, (long)__builtin_amdgcn_readfirstlane((int)n)) : floatx4{};
    }
    template <bool OWN, bool ONE>
    __device__ __forceinline__ float threshold(const Thresholds &ths, const floatx4 requested) const
    {
        if (ONE) return given_threshold(ths, n);
        const long n_first = (long)__builtin_amdgcn_readfirstlane((int)n), n_last = (long)__builtin_amdgcn_readlane((int)n, 63);
        if (OWN && ths.splits > 0) return span_threshold(ths, n, n_first, n_last, requested);
        return n_last == n_first ? given_threshold(ths, n_first) : given_threshold(ths, n);
    }
    // pixels [first, last) of a wave's lanes from..to, which follow each other without a gap
    __device__ __forceinline__ long first(int from = 0) const { return lane_pixel(from); }
    __device__ __forceinline__ long last(int to = 63) const { return lane_pixel(to) + VEC; }
    __device__ __forceinline__ long lane_pixel(int lane) const
    {
        const uint32_t low = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)pixel, lane);
        const uint32_t high = (uint32_t)__builtin_amdgcn_readlane((int)((uint64_t)pixel >> 32), lane);
        return (long)((uint64_t)high << 32 | low);
    }
};

//
// A wave packs 16 channels of 64 runs, all of whose loads it requests at once; the up to four waves of a workgroup that
// share a word (SPLIT: C > 32 four, C > 16 two) meet in LDS, from where the word is stored, pixels in order over the lanes.
// With a thread to a whole word, 64 loads and the 200 to 700 instructions of their bits in a row were what a tensor too small
// to fill the chip waited for, and two loads in three were short of the parallelism a large one needs: N=32 64 x 56 x 56
// (two planes) 6.1 -> 4.4 us, N=128 64 x 112 x 112 79.9 -> 72.4 (6.0 TB/s), N=64 3 x 112 x 112 16.6 -> 6.7.
// grid = ceil(runs / (64 * 4 / SPLIT)) * PC workgroups, the word index fastest: the workgroups that write the PC words of the
// same pixels run side by side, so their 8- or 16-byte stores meet in L2 as whole lines.  Where last words have waves of their own (LAST), plane_units
// units in the order of plane_unit: those of four or two groups of runs, word after word, then one for the last words of all of these groups.
// The lane's nonzero values are counted for COUNT (see Counts).
template <int BITS, int VEC, int SPLIT, bool NT, bool COUNT = false>
__device__ __forceinline__ int quantize_nchw_unit(const float *__restrict__ x, const Thresholds &ths, uint64_t *__restrict__ q, const PixelRun<VEC> &run,
                                                  int C, long HW, int PC, int pc)
{
    constexpr int kPart = 16;                       // channels a wave packs of its pixels
    constexpr int GROUPS = kWavesPerBlock / SPLIT;  // of 64 pixel runs, per workgroup
    constexpr int SLOTS = 64 * VEC;
    // Loads are requested in the order in which their bits are shifted in: from the last channel down the bits come out in
    // place (4.2 -> 3.95 us at 26 MB); runs of four, which overlap cache lines of the planes' ends, are read faster upwards
    // (24 x 75 x 61 x 47: 7.1 -> 6.7 us).
    constexpr bool UP = VEC == 4;
    __shared__ alignas(16) uint16_t parts[GROUPS][SPLIT][BITS][SLOTS];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int part = wave % SPLIT, group = wave / SPLIT;
    const int c0 = pc * kWordBits + part * kPart;
    const int channels = C - c0 < kPart ? C - c0 : kPart;  // zero or less: no such part
    uint32_t less[VEC], more[VEC];
#pragma unroll
    for (int e = 0; e < VEC; e++) less[e] = more[e] = 0;
    if (channels > 0) {
        const float *src = x + (run.n * C + c0) * HW + run.s;
        const floatx4 requested = run.template request<BITS == 2 && !COUNT>(ths);
        float v[kPart][VEC];
        if (channels == kPart) {
#pragma unroll
            for (int i = 0; i < kPart; i++) {
                const int u = UP ? i : kPart - 1 - i;
                run.template load<NT>(v[u], src + u * HW);
            }
        } else {  // what is left of C: nothing is read twice (a clamped channel number would, past the cache if NT)
#pragma unroll
            for (int u = 0; u < kPart; u++) {
#pragma unroll
                for (int e = 0; e < VEC; e++) v[u][e] = 0.f;
                if (u < channels) run.template load<NT>(v[u], src + u * HW);
            }
        }
        // the threshold is added up while the channels are in flight
        const float t = run.template threshold<BITS == 2 && !COUNT, COUNT>(ths, requested);
        const float low = BITS == 2 ? -t : t;
        if constexpr (VEC == 4) {
#pragma unroll
            for (int u = 0; u < kPart; u++) {
                shift_in_less4(less, v[u], low);
                if (BITS == 2) shift_in_more4(more, v[u], t);
            }
        } else {
#pragma unroll
            for (int u = kPart - 1; u > 0; u -= 4) {
                shift_in_less4(less[0], v[u][0], v[u - 1][0], v[u - 2][0], v[u - 3][0], low);
                if (BITS == 2) shift_in_more4(more[0], v[u][0], v[u - 1][0], v[u - 2][0], v[u - 3][0], t);
            }
        }
        const uint32_t exist = 0xffffu >> (kPart - channels);
#pragma unroll
        for (int e = 0; e < VEC; e++) {
            if (UP) {  // the first channel went in first and stands highest
                less[e] = __brev(less[e]) >> (32 - kPart);
                more[e] = __brev(more[e]) >> (32 - kPart);
            }
            less[e] &= exist;
            more[e] &= exist;
        }
    }
    typedef uint16_t Bits __attribute__((ext_vector_type(VEC)));
    Bits sign, nz;
#pragma unroll
    for (int e = 0; e < VEC; e++) {
        sign[e] = (uint16_t)(BITS == 2 ? less[e] & ~more[e] : less[e]);
        nz[e] = (uint16_t)(less[e] | more[e]);
    }
    *reinterpret_cast<Bits *>(&parts[group][part][0][lane * VEC]) = sign;
    if (BITS == 2) *reinterpret_cast<Bits *>(&parts[group][part][BITS - 1][lane * VEC]) = nz;
    __syncthreads();
#pragma unroll
    for (int s0 = 0; s0 < SLOTS; s0 += 64 * SPLIT) {
        if (s0 + part * 64 >= SLOTS) break;
        const int slot = s0 + part * 64 + lane;
        const long pixel = (VEC == 1 ? run.pixel : run.first() + __shfl((int)(run.pixel - run.first()), slot / VEC, 64)) + slot % VEC;
        uint64_t word[BITS];
#pragma unroll
        for (int b = 0; b < BITS; b++) {
            word[b] = 0;
#pragma unroll
            for (int p = 0; p < SPLIT; p++) word[b] |= (uint64_t)parts[group][p][b][slot] << (kPart * p);
        }
        uint64_t *dst = q + (pixel * PC + pc) * BITS;
#pragma unroll
        for (int b = 0; b < BITS; b++) dst[b] = word[b];
    }
    int count = 0;
#pragma unroll
    for (int e = 0; e < VEC; e++) count += e >= run.repeated ? __builtin_popcount((uint32_t)nz[e]) : 0;
    return count;
}

// Waves that a last word of few channels takes in place of four; 0: as many as the others.
__host__ __device__ __forceinline__ int last_word_waves(int C, int PC)
{
    const int channels = C - (PC - 1) * kWordBits;
    return PC == 1 || channels > 32 ? 0 : (channels <= 16 ? 1 : 2);
}

// Which word of which run the wave of a workgroup's unit `block` packs, and how many waves share it.  With four waves on a last word of up to 32
// channels two or three of them would have none and hold a place on the CU for as long as the others' loads take; and with PC even every
// second CU would get such words only.  So a workgroup takes the last words of four (or two) groups of runs, behind the other words of those
// (LAST).  us, one plane: 24 61x47 of 75 channels 7.4 -> 6.4, 128 28x28 of 75 8.9 -> 7.5, 64 56x56 of 200 34.0 -> 32.6.
struct PlaneUnit {
    long run;  // of the wave's first lane
    int pc, split;
};
template <int SPLIT, bool LAST>
__device__ __forceinline__ PlaneUnit plane_unit(uint32_t block, int C, int PC, int wave)
{
    if (LAST) {
        const int last = last_word_waves(C, PC);
        const uint32_t groups = 4 / last, others = PC - 1, units = groups * others + 1, first = block / units * groups, in = block % units;
        if (in == units - 1) return {(long)(first + wave / last) * 64, PC - 1, last};
        return {(long)(first + in / others) * 64, (int)(in % others), SPLIT};
    }
    return {((long)(block / (uint32_t)PC) * (kWavesPerBlock / SPLIT) + wave / SPLIT) * 64, (int)(block % (uint32_t)PC), SPLIT};
}
// Units of `groups` groups of 64 runs with the last words apart (last: their waves), if those are no more than without, groups * PC: few groups
// fill a unit of four groups' last words badly, and the workspace of counts has room for that many.
inline long plane_units(long groups, int PC, int &last)
{
    if (last) {
        const long of_last = 4 / last, units = (groups + of_last - 1) / of_last * (of_last * (PC - 1) + 1);
        if (units <= groups * PC) return units;
        last = 0;
    }
    return groups * PC;
}

template <int BITS, int VEC, int SPLIT, bool NT, bool LAST, bool COUNT = false>
__device__ __forceinline__ int quantize_nchw_unit_of(const float *__restrict__ x, const Thresholds &ths, uint64_t *__restrict__ q, const PixelRun<VEC> &run,
                                                     const PlaneUnit unit, int C, long HW, int PC)
{
    if (LAST && unit.split == 1) return quantize_nchw_unit<BITS, VEC, 1, NT, COUNT>(x, ths, q, run, C, HW, PC, unit.pc);
    if (LAST && unit.split == 2) return quantize_nchw_unit<BITS, VEC, 2, NT, COUNT>(x, ths, q, run, C, HW, PC, unit.pc);
    return quantize_nchw_unit<BITS, VEC, SPLIT, NT, COUNT>(x, ths, q, run, C, HW, PC, unit.pc);
}

template <int BITS, int VEC, int SPLIT, bool NT, bool LAST>
__device__ __forceinline__ void quantize_nchw_block(const float *__restrict__ x, const Thresholds &ths, uint64_t *__restrict__ q, int N, int C, long HW, int PC,
                                                    Div32 by_image, uint32_t block, int32_t *btn)
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const PlaneUnit unit = plane_unit<SPLIT, LAST>(block, C, PC, wave);
    const PixelRun<VEC> run(unit.run + (threadIdx.x & 63), N, HW, by_image);
    quantize_nchw_unit_of<BITS, VEC, SPLIT, NT, LAST>(x, ths, q, run, unit, C, HW, PC);
    if (wave % SPLIT == 0) zero_counts(btn, N, run.pixel, VEC);
}

template <int BITS, int VEC, int SPLIT, bool NT = false, bool LAST = false>
__global__ __launch_bounds__(kThreads) void quantize_nchw(const float *__restrict__ x, const Thresholds ths,
                                                          uint64_t *__restrict__ q, int N, int C, long HW, int PC, Div32 by_image, int32_t *btn)
{
    quantize_nchw_block<BITS, VEC, SPLIT, NT, LAST>(x, ths, q, N, C, HW, PC, by_image, in_eighths(blockIdx.x, ths.eighth), btn);
}

// Beside a convolution's weights.
template <int BITS, int VEC, int SPLIT, bool NT = false, bool LAST = false>
__global__ __launch_bounds__(kThreads) void quantize_nchw_weights(const float *__restrict__ x, const Thresholds ths, uint64_t *__restrict__ q, int N,
                                                                  int C, long HW, int PC, Div32 by_image, const WeightJob job)
{
    uint32_t block = blockIdx.x;
    if (pack_weights<kThreads>(job, block)) return;
    quantize_nchw_block<BITS, VEC, SPLIT, NT, LAST>(x, ths, q, N, C, HW, PC, by_image, in_eighths(block, ths.eighth), nullptr);
}

// The same with counts: a unit is what plane_unit gives a workgroup, 64 * 4 / SPLIT runs and one word, or the last words of several groups of runs.
template <int VEC, int SPLIT, bool NT = false, bool LAST = false>
__global__ __launch_bounds__(kThreads) void quantize_nchw_count(const float *__restrict__ x, const Thresholds ths, uint64_t *__restrict__ q, int C,
                                                                long HW, int PC, int units, const Counts counts)
{
    __shared__ int32_t scratch[kWavesPerBlock];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int item = (int)(blockIdx.x / (uint32_t)counts.slices), slice = (int)blockIdx.x - item * counts.slices;
    int count = 0;
    for (int unit = slice; unit < units; unit += counts.slices) {
        if (unit >= counts.slices) __syncthreads();  // the waves have read the words before
        const PlaneUnit of = plane_unit<SPLIT, LAST>((uint32_t)unit, C, PC, wave);
        const PixelRun<VEC> run(of.run + (threadIdx.x & 63), item, HW, std::true_type());
        count += quantize_nchw_unit_of<2, VEC, SPLIT, NT, LAST, true>(x, ths, q, run, of, C, HW, PC);
    }
    store_count<kWavesPerBlock>(count, counts.out + blockIdx.x, scratch);
}


// The NCHW quantizer for PC a multiple of U = 2 or 4 and at least one wave of work per SIMD: a thread packs U
// neighbouring words of its four pixels, one after the other, and the wave then turns its 256 pixels x U words
// (x 2 planes) around in LDS, so that a store instruction writes whole runs of the output - U * BITS words per pixel,
// the entire kilobyte when PC == U - instead of one 8-byte word per lane at the stride of a pixel.  Measured on
// 256 x 256 x 56 x 56: 137 us (one plane) / 151 us (two); with quantize_nchw 166 / 187.  Planes of odd sizes
// (256 x 256 x 55 x 55: 159 -> 146 us, 177 -> 153): EVEN keeps the flat numbering of runs for the others, whose 3 us of 137
// are the registers that it does without.
// One wave per workgroup (with four, the 784 workgroups of that tensor load the CUs 4 : 3), 4 KB of LDS, gone through
// in WPP / 2 rounds of 64 / rounds lanes each.  grid = ceil(runs / 64) * (PC / U), the word group fastest.
// Bits are made by the form and in as many registers as measured best: SHIFT for U = 2.
// COUNT: a wave is a slice of one unit (see Counts).
// WEIGHTS: a convolution's weights beside (then without counts).
template <int BITS, int U, bool EVEN, bool COUNT = false, bool WEIGHTS = false>
__global__ __launch_bounds__(64, BITS == 1 ? (U == 4 ? 4 : 7) : (U == 4 ? 1 : 4)) void quantize_nchw_gather(const float *__restrict__ x, const Thresholds ths,
                                                                 uint64_t *__restrict__ q, int N, int C, long HW, int PC, Div32 by_image,
                                                                 typename std::conditional<WEIGHTS, WeightJob, int32_t *>::type extra)
{
    static_assert(!COUNT || (BITS == 2 && !EVEN), "counts of two planes; runs of one image are numbered for any plane size");
    constexpr int VEC = 4, kInFlight = 8;
    constexpr int WPP = U * BITS;      // words a thread packs per pixel, contiguous in q
    constexpr int ROUNDS = WPP / 2;    // 64 / ROUNDS lanes x 4 pixels x WPP words = 512 words a round
    constexpr int LPR = 64 / ROUNDS;
    constexpr bool SHIFT = U == 2;
    static_assert(U == 2 || U == 4, "one word per thread is quantize_nchw");
    __shared__ __attribute__((aligned(16))) uint64_t stage[512];
    uint32_t block = blockIdx.x;
    if constexpr (WEIGHTS)
        if (pack_weights<64>(extra, block)) return;
    int32_t *btn = nullptr;
    if constexpr (!WEIGHTS) btn = extra;
    if constexpr (!COUNT) block = in_eighths(block, ths.eighth);
    const int groups = PC / U;
    // COUNT: N is the number of slices of an image
    const int image = COUNT ? (int)(block / (uint32_t)N) : 0;
    const int unit = (int)block - image * N * COUNT;
    const int pc0 = (unit % groups) * U;
    const int lane = threadIdx.x;
    const PixelRun<VEC, EVEN> run = COUNT ? PixelRun<VEC, EVEN>((long)(unit / groups) * 64 + lane, image, HW, std::true_type())
                                          : PixelRun<VEC, EVEN>((long)(unit / groups) * 64 + lane, N, HW, by_image);
    // The U words are U * 64 consecutive channels: batches of kInFlight channels, the next batch's loads issued before
    // the compares of this one (two register buffers), so the memory pipe never waits for the packing.
    const int cbase = pc0 * kWordBits;
    const float *src = x + run.n * C * HW + run.s;
    auto load = [&](float (&v)[kInFlight][VEC], const int b) {
#pragma unroll
        for (int i = 0; i < kInFlight; i++) {
            const int k = SHIFT ? kInFlight - 1 - i : i;  // in the order of use
            int c = cbase + b * kInFlight + k;
            c = c < C ? c : C - 1;  // past the last channel (tail word, prefetch after the last batch): masked in pack() or unused
            run.template load<true>(v[k], src + (long)c * HW);
        }
    };
    uint64_t words[VEC][WPP];
    uint64_t sign[VEC], nz[VEC];
    float t;
    auto pack = [&](const float (&v)[kInFlight][VEC], const int b) {
        uint32_t s[VEC], z[VEC];
        if constexpr (SHIFT) {
            const int left = C - cbase - b * kInFlight;
            const uint32_t exist = left >= kInFlight ? (1u << kInFlight) - 1 : left > 0 ? (1u << left) - 1 : 0u;
            uint32_t less[VEC] = {0, 0, 0, 0}, more[VEC] = {0, 0, 0, 0};
#pragma unroll
            for (int k = kInFlight - 1; k >= 0; k--) {
                if (BITS == 1) {
                    shift_in_less4(less, v[k], t);
                } else {
#pragma unroll
                    for (int e = 0; e < VEC; e++) {
                        less[e] |= v[k][e] < -t ? 1u << k : 0u;
                        more[e] |= t < v[k][e] ? 1u << k : 0u;
                    }
                }
            }
#pragma unroll
            for (int e = 0; e < VEC; e++) {
                s[e] = (less[e] & ~more[e]) & exist;
                z[e] = (less[e] | more[e]) & exist;
            }
        } else {
#pragma unroll
            for (int e = 0; e < VEC; e++) s[e] = z[e] = 0;
#pragma unroll
            for (int k = 0; k < kInFlight; k++) {
                const uint32_t bit = cbase + b * kInFlight + k < C ? 1u << k : 0u;
#pragma unroll
                for (int e = 0; e < VEC; e++) {
                    if (BITS == 2) {
                        const bool pos = v[k][e] > t;
                        const bool neg = !pos && (v[k][e] < -t);
                        if (pos || neg) z[e] |= bit;
                        if (neg) s[e] |= bit;
                    } else {
                        if (v[k][e] < t) s[e] |= bit;
                    }
                }
            }
        }
        const int shift = (b * kInFlight) % kWordBits;
#pragma unroll
        for (int e = 0; e < VEC; e++) {
            sign[e] |= (uint64_t)s[e] << shift;
            if (BITS == 2) nz[e] |= (uint64_t)z[e] << shift;
        }
    };
    constexpr int kBatches = kWordBits / kInFlight;  // per word
    float v0[kInFlight][VEC], v1[kInFlight][VEC];
    const floatx4 requested = run.template request<BITS == 2 && !COUNT>(ths);
    load(v0, 0);
    t = run.template threshold<BITS == 2 && !COUNT, COUNT>(ths, requested);
#pragma unroll
    for (int u = 0; u < U; u++) {
#pragma unroll
        for (int e = 0; e < VEC; e++) sign[e] = nz[e] = 0;
#pragma unroll 1
        for (int b = u * kBatches; b < (u + 1) * kBatches; b += 2) {
            load(v1, b + 1);
            pack(v0, b);
            load(v0, b + 2);  // after the last batch too (a valid channel, unused): guarding it costs more than the 8 loads
            pack(v1, b + 1);
        }
#pragma unroll
        for (int e = 0; e < VEC; e++) {
            words[e][u * BITS] = sign[e];
            if (BITS == 2) words[e][u * BITS + 1] = nz[e];
        }
    }
#pragma unroll
    for (int r = 0; r < ROUNDS; r++) {
        const long first = run.first(r * LPR);
        __builtin_amdgcn_wave_barrier();
        if (lane / LPR == r) {
            ulonglong2 *dst = reinterpret_cast<ulonglong2 *>(stage + (run.pixel - first) * WPP);
#pragma unroll
            for (int e = 0; e < VEC; e++)
#pragma unroll
                for (int j = 0; j < WPP; j += 2)
                    dst[(e * WPP + j) / 2] = make_ulonglong2(words[e][j], words[e][j + 1]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const long last = run.last(r * LPR + LPR - 1);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int w = (i * 64 + lane) * 2;  // two words a lane: 1 KB a store instruction
            const long pixel = first + w / WPP;
            const ulonglong2 pair = *reinterpret_cast<const ulonglong2 *>(stage + w);
            // an even word index (PC * BITS, pc0 * BITS and w % WPP are even) into a 16-byte aligned q
            if (pixel < last) *reinterpret_cast<ulonglong2 *>(q + (pixel * PC + pc0) * BITS + w % WPP) = pair;
        }
    }
    if (COUNT) {
        int count = 0;
#pragma unroll
        for (int e = 0; e < VEC; e++)
#pragma unroll
            for (int u = 0; u < U; u++) count += e >= run.repeated ? __popcll(words[e][u * BITS + BITS - 1]) : 0;
        store_count<1>(count, btn + blockIdx.x, nullptr);
    } else {
        zero_counts(btn, N, run.pixel, VEC);
    }
}

// btn[n] = sum over item n of popcount(nonzero-plane word) (BTN_Weight, TAB_GEMM.cu:150-160,
// for every n).  q is the ternary output [items][words_per_item][2]; one workgroup per
// (item, split) reads its words as 16-byte (sign, nonzero) pairs.  With one split the result
// is stored directly; with several the partial sums are added atomically into btn, which the
// quantizer zeroed.
// Bound by reading the packed output back (from the caches, it was just written): four loads in flight a lane and a
// full CU of waves, in workgroups of 1024 because every workgroup of a split item is one more atomic on the few cache
// lines of btn.
constexpr int kCountThreads = 1024;
constexpr int kCountLoads = 4;

__global__ __launch_bounds__(kCountThreads) void btn_popcount(const ulonglong2 *__restrict__ q,
                                                              int32_t *__restrict__ btn,
                                                              long words_per_item, int splits, int threads)
{
    __shared__ int partial[kCountThreads / 64];
    const long item = blockIdx.x / splits;
    const int split = blockIdx.x % splits;
    const long per_split = (words_per_item + splits - 1) / splits;
    const long w0 = split * per_split;
    long w1 = w0 + per_split;
    if (w1 > words_per_item) w1 = words_per_item;
    const ulonglong2 *src = q + item * words_per_item;
    int count = 0;
    long w = w0 + threadIdx.x;
    const long step = threads;  // the workgroup's size, as an argument: blockDim would add 256 bytes of hidden ones
    for (; w + (kCountLoads - 1) * step < w1; w += kCountLoads * step) {
        ulonglong2 v[kCountLoads];
#pragma unroll
        for (int u = 0; u < kCountLoads; u++) v[u] = src[w + u * step];
#pragma unroll
        for (int u = 0; u < kCountLoads; u++) count += __popcll(v[u].y);
    }
    for (; w < w1; w += step) count += __popcll(src[w].y);
    count = wave_sum(count);
    if ((threadIdx.x & 63) == 0) partial[threadIdx.x >> 6] = count;
    __syncthreads();
    if (threadIdx.x == 0) {
        int total = 0;
        for (int i = 0; i < threads >> 6; i++) total += partial[i];
        if (splits == 1)
            btn[item] = total;
        else if (total)
            atomicAdd(&btn[item], total);
    }
}

// ---- thresholds: ths[n] = scale * mean(|x[n]|) ------------------------------------------------
// The step right before Quantize in the reference's demo flow (the caller computes it in
// torch).  Two fixed-order stages so that the result does not depend on scheduling: `splits`
// workgroups per item each reduce a contiguous slice to one fp32 partial (per-thread serial
// sums of float4, then a tree over lanes and waves), then one thread per item adds the
// partials in index order in fp64.
// An item of one slice is finished here: `out` gets its threshold, not its sum.
__global__ __launch_bounds__(kThreads) void abs_sum_partial(const float *__restrict__ x, float *__restrict__ out,
                                                            long per_item, int splits, double scale_over_count, int eighth, int kept)
{
    constexpr int kLoads = 4;  // in flight per lane
    __shared__ float wave_part[kWavesPerBlock];
    const uint32_t block = in_eighths(blockIdx.x, eighth);
    const bool keep = (int)(blockIdx.x >> 3) >= kept;  // uniform
    const long item = block / (uint32_t)splits;
    const int split = (int)(block % (uint32_t)splits);
    const long slice = ((per_item + splits - 1) / splits + 3) & ~3L;  // multiple of 4 elements
    const long begin = split * slice;
    long end = begin + slice;
    if (end > per_item) end = per_item;
    const float *src = x + item * per_item;
    float sum = 0.f;
    if (((uintptr_t)(src + begin) & 15) == 0) {
        const long n4 = begin < end ? (end - begin) / 4 : 0;
        const floatx4 *src4 = reinterpret_cast<const floatx4 *>(src + begin);
        auto add = [&](const floatx4 v) {
            sum += (__builtin_fabsf(v[0]) + __builtin_fabsf(v[1])) + (__builtin_fabsf(v[2]) + __builtin_fabsf(v[3]));
        };
        long i = threadIdx.x;
        auto stream = [&](auto load) {
            for (; i + (kLoads - 1) * kThreads < n4; i += kLoads * kThreads) {
                floatx4 v[kLoads];
#pragma unroll
                for (int u = 0; u < kLoads; u++) v[u] = load(&src4[i + u * kThreads]);
#pragma unroll
                for (int u = 0; u < kLoads; u++) add(v[u]);
            }
            for (; i < n4; i += kThreads) add(load(&src4[i]));
        };
        if (keep) stream([](const floatx4 *p) { return *p; });
        else stream([](const floatx4 *p) { return __builtin_nontemporal_load(p); });
        for (i = begin + n4 * 4 + threadIdx.x; i < end; i += kThreads) sum += __builtin_fabsf(src[i]);
    } else {
        for (long i = begin + threadIdx.x; i < end; i += kThreads) sum += __builtin_fabsf(src[i]);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off, 64);
    if ((threadIdx.x & 63) == 0) wave_part[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        float total = 0.f;
#pragma unroll
        for (int w = 0; w < kWavesPerBlock; w++) total += wave_part[w];
        out[block] = splits == 1 ? (float)((double)total * scale_over_count) : total;
    }
}

// One wave per item.  (One thread per item, adding its partial sums one dependent load after the other, took 5.8 us for 32
// items of 64 slices.)
__global__ __launch_bounds__(64) void abs_mean_finish(const Thresholds source, float *__restrict__ ths)
{
    const float t = wave_threshold(source, blockIdx.x);
    if (threadIdx.x == 0) ths[blockIdx.x] = t;
}

}  // namespace

int threshold_splits(long items, long per_item)
{
    int splits = 1;
    while (splits < 1024 && items * splits < 2048 && per_item / (splits * 2) >= 8L * kThreads) splits *= 2;
    return splits;
}

hipError_t launch_abs_sums(const float *x, long items, long per_item, float scale, float *partial, Thresholds *source,
                           hipStream_t stream)
{
    const int splits = threshold_splits(items, per_item);
    source->values = partial;
    source->scale = (double)scale / (double)per_item;
    source->splits = splits == 1 ? 0 : splits;
    // The quantizer that follows reads x again, backwards in eighths: what it begins with, 24 MB, is read through the L2s here, the rest
    // past them (plain loads stream 8-11 % slower from 400 MB on).  Two passes over 25.7 MB (NCHW, N=32 56x56x64): 7.0 + 7.0 -> 5.6 +
    // 5.6 us; over 103 MB (N=64 56x56x128): 9.5 + 22.6 -> 8.8 + 17.2.
    source->eighth = -1;
    const long blocks = items * splits, share = blocks / 8, bytes = items * per_item * 4;
    const long kept = bytes <= (24L << 20) ? 0 : share - (long)((double)share * (24L << 20) / (double)bytes);
    abs_sum_partial<<<dim3((unsigned)blocks), dim3(kThreads), 0, stream>>>(x, partial, per_item, splits, source->scale, blocks < 64 ? 0 : (int)share,
                                                                         (int)kept);
    return hipGetLastError();
}

hipError_t launch_threshold_values(const Thresholds &source, long items, float *ths, hipStream_t stream)
{
    abs_mean_finish<<<dim3((unsigned)items), dim3(64), 0, stream>>>(source, ths);
    return hipGetLastError();
}

hipError_t launch_threshold(const float *x, long items, long per_item, float scale, float *ths, float *partial,
                            hipStream_t stream)
{
    Thresholds source;
    if (threshold_splits(items, per_item) == 1) return launch_abs_sums(x, items, per_item, scale, ths, &source, stream);
    const hipError_t e = launch_abs_sums(x, items, per_item, scale, partial, &source, stream);
    return e != hipSuccess ? e : launch_threshold_values(source, items, ths, stream);
}

// Workgroups per item of btn_popcount: enough to fill the chip twice over, none with less than a load a thread.
int count_splits(long items, long words_per_item)
{
    int splits = 1;
    while (splits < 64 && items * splits < 512 && words_per_item / (splits * 2) >= kCountThreads) splits *= 2;
    return splits;
}

void launch_btn_popcount(const uint64_t *qx, int32_t *btn, long items, long words_per_item, int splits, hipStream_t stream)
{
    // an item of few words (a filter) takes as many whole waves as it has words for
    const long per_split = (words_per_item + splits - 1) / splits;
    const int threads = per_split >= kCountThreads ? kCountThreads : (int)((per_split + 63) / 64) * 64;
    btn_popcount<<<dim3((unsigned)(items * splits)), dim3(threads), 0, stream>>>(reinterpret_cast<const ulonglong2 *>(qx), btn,
                                                                               words_per_item, splits, threads);
}

// Where the counts of a two-plane quantizer go: an item of this many units is one slice (a unit takes some 0.7 us, count_finish
// 2.4), others are slices of one unit each, whose counts need `workspace`; null: none there, the packed output is read back.
struct CountTarget {
    int32_t *btn, *workspace;
};
constexpr long kOneSliceUnits = 3;

void finish_counts(const CountTarget &target, long items, int slices, hipStream_t stream)
{
    if (slices > 1) count_finish<<<dim3((unsigned)items), dim3(kThreads), 0, stream>>>(target.workspace, target.btn, slices);
}

template <int MODE, int LP>
void launch_quantize_tile_of(const float *x, const Thresholds &ths, long pixels, long pixels_per_item, long items, int C, uint64_t *q,
                             int32_t *btn, const CountTarget *counted, const WeightJob *weights, hipStream_t stream)
{
    // 12 KB of x a tile, measured from 4 to 48 KB on C = 3 ... 32: what a few workgroups a CU keep in flight against the
    // wait of each for its whole tile.
    long tile_pixels = 12 * 1024 / (4L * C) / 16 * 16;
    const bool one_slice = counted && pixels_per_item <= kOneSliceUnits * tile_pixels;
    // a tensor of few tiles: smaller ones, down to a read of every wave
    while (!one_slice && tile_pixels >= 8 && pixels / tile_pixels < 512 && tile_pixels / 2 >= 4 * (64 / LP)) tile_pixels = tile_pixels / 8 * 4;
    const size_t lds = ((size_t)(tile_pixels * C + 6) / 4 * 4 + 256 + tile_pixels) * 4;
    const Div32 div_item = pixels < 0x7fffffffL ? make_div32((uint32_t)pixels_per_item) : Div32{0, 0};
    if constexpr (MODE == 2) {
        if (counted) {
            const long slices = one_slice ? 1 : (pixels_per_item + tile_pixels - 1) / tile_pixels;
            quantize_tile_count<LP><<<dim3((unsigned)(items * slices)), dim3(kThreads), lds, stream>>>(
                x, ths, q, pixels_per_item, div_item, C, (int)tile_pixels, Counts{slices == 1 ? counted->btn : counted->workspace, (int)slices});
            finish_counts(*counted, items, (int)slices, stream);
            return;
        }
    }
    const unsigned tiles = (unsigned)((pixels + tile_pixels - 1) / tile_pixels);
    if constexpr (MODE != 5) {  // (type 5 has no kernel that reads its weights in another order)
        if (weights) {
            quantize_tile_weights<MODE, LP><<<dim3(tiles + weights->blocks), dim3(kThreads), lds, stream>>>(
                x, ordered(ths, tiles), q, pixels, pixels_per_item, div_item, C, (int)tile_pixels, *weights);
            return;
        }
    }
    quantize_tile<MODE, LP><<<dim3(tiles), dim3(kThreads), lds, stream>>>(x, ordered(ths, tiles), q, pixels, pixels_per_item, div_item, C, (int)tile_pixels, btn, items);
}

// Up to 32 channels with the fewest lanes a word that hold it.
template <int MODE>
void launch_quantize_tile(const float *x, const Thresholds &ths, long pixels, long pixels_per_item, long items, int C, uint64_t *q,
                          int32_t *btn, const CountTarget *counted, const WeightJob *weights, hipStream_t stream)
{
    if (C <= 4) launch_quantize_tile_of<MODE, 4>(x, ths, pixels, pixels_per_item, items, C, q, btn, counted, weights, stream);
    else if (C <= 8) launch_quantize_tile_of<MODE, 8>(x, ths, pixels, pixels_per_item, items, C, q, btn, counted, weights, stream);
    else if (C <= 16) launch_quantize_tile_of<MODE, 16>(x, ths, pixels, pixels_per_item, items, C, q, btn, counted, weights, stream);
    else launch_quantize_tile_of<MODE, 32>(x, ths, pixels, pixels_per_item, items, C, q, btn, counted, weights, stream);
}

// Counts of every two-plane quantizer in slices: workspace ints at most (a unit holds at least four words).
size_t quantize_count_workspace(int bitwidth, long items, long pixels_per_item, int C)
{
    const long PC = (C + kWordBits - 1) / kWordBits;
    if (bitwidth != 2 || (pixels_per_item * PC <= 64 && PC <= kOneSliceUnits)) return 0;  // one slice in every form
    return (size_t)items * (pixels_per_item * PC / 4 + PC + 1) * sizeof(int32_t);
}

// Which path packs an NHWC tensor: a pixel of up to 32 channels leaves half of a row's 16 lanes and more without work, and tiles are as soon
// or sooner at every size (tile / rows, one plane, us: C=32 0.6 MB 2.5 / 2.5, 9.6 MB 3.8 / 4.2; C=16 1.2 MB 2.8 / 2.8, 9.6 MB 3.8 / 4.9; C=5 1.2
// MB 3.0 / 3.8, 60 MB 16.5 / 51); from 33 on rows are (C=33 2 MB 3.4 / 2.4, 150 MB 30.9 / 27.6).
enum class Path { whole, ragged, tile };
Path quantize_path(const float *x, int C)
{
    if (C % kWordBits == 0 && (uintptr_t)x % 16 == 0) return Path::whole;
    return C > 32 ? Path::ragged : Path::tile;
}

// Rows of 64 channels without counts.  A launch too small to fill the chip with 128 rows a workgroup takes 32, two loads a lane (3.1 MB
// of fp32: 5.5 -> 4.2 us).
template <int FORMAT>
hipError_t launch_rows(Path path, const float *x, const Thresholds &ths, long pixels, long pixels_per_item, long items, int C, uint64_t *qx,
                       int32_t *zeroed, const WeightJob *weights, hipStream_t stream)
{
    constexpr bool SUMS = FORMAT == 2;      // thresholds as partial sums
    constexpr bool BESIDE = FORMAT != 5;    // (type 5 has no kernel that reads its weights in another order)
    const long PC = (C + kWordBits - 1) / kWordBits, rows = pixels * PC, rows_per_item = pixels_per_item * PC;
    const Div32 div_item = rows < 0x7fffffffL ? make_div32((uint32_t)rows_per_item) : Div32{0, 0};
    const bool few = rows <= kSmallLaunchBlocks * 128, own = SUMS && ths.splits > 0;
    const long blocks = (rows + (few ? 31 : 127)) / (few ? 32 : 128);
    const Thresholds t = ordered(ths, blocks);
    const dim3 grid((unsigned)(blocks + (weights ? weights->blocks : 0)));
    const int lds = few ? 0 : kStreamLds;
    const floatx4 *x4 = reinterpret_cast<const floatx4 *>(x);
    uint32_t *q32 = reinterpret_cast<uint32_t *>(qx);
    if (path == Path::whole) {
        if (BESIDE && weights) {
            auto kernel = few ? own ? quantize_rows64_weights<BESIDE ? FORMAT : 1, 2, SUMS> : quantize_rows64_weights<BESIDE ? FORMAT : 1, 2>
                              : own ? quantize_rows64_weights<BESIDE ? FORMAT : 1, 8, SUMS> : quantize_rows64_weights<BESIDE ? FORMAT : 1>;
            kernel<<<grid, dim3(kThreads), lds, stream>>>(x4, t, q32, rows, rows_per_item, div_item, *weights);
        } else {
            auto kernel = few ? own ? quantize_rows64<FORMAT, 2, SUMS> : quantize_rows64<FORMAT, 2> : own ? quantize_rows64<FORMAT, 8, SUMS> : quantize_rows64<FORMAT>;
            kernel<<<grid, dim3(kThreads), lds, stream>>>(x4, t, q32, rows, rows_per_item, div_item, zeroed, items);
        }
    } else {
        const RaggedRows ragged{C, make_div32((uint32_t)PC)};
        if (BESIDE && weights) {
            auto kernel = few ? own ? quantize_rows_ragged_weights<BESIDE ? FORMAT : 1, 2, SUMS> : quantize_rows_ragged_weights<BESIDE ? FORMAT : 1, 2>
                              : own ? quantize_rows_ragged_weights<BESIDE ? FORMAT : 1, 8, SUMS> : quantize_rows_ragged_weights<BESIDE ? FORMAT : 1>;
            kernel<<<grid, dim3(kThreads), lds, stream>>>(x4, t, q32, rows, rows_per_item, div_item, ragged, *weights);
        } else {
            auto kernel = few ? own ? quantize_rows_ragged<FORMAT, 2, SUMS> : quantize_rows_ragged<FORMAT, 2> : own ? quantize_rows_ragged<FORMAT, 8, SUMS> : quantize_rows_ragged<FORMAT>;
            kernel<<<grid, dim3(kThreads), lds, stream>>>(x4, t, q32, rows, rows_per_item, div_item, zeroed, items, ragged);
        }
    }
    return hipGetLastError();
}

// x: fp32 [items][pixels_per_item][C]; qx: [items*pixels_per_item][PC][bitwidth];
// btn: [items] or nullptr (then no counts are produced).
hipError_t launch_quantize(const float *x, const Thresholds &ths, int bitwidth, long pixels_per_item,
                           long items, int C, uint64_t *qx, int32_t *btn, int32_t *count_workspace, hipStream_t stream,
                           const WeightJob *weights)
{
    const int PC = (C + kWordBits - 1) / kWordBits;
    const long pixels = items * pixels_per_item;
    const long words_per_item = pixels_per_item * PC;
    const int splits = btn && bitwidth == 2 ? count_splits(items, words_per_item) : 1;
    // counts that are not stored whole by btn_popcount start at zero
    int32_t *zeroed = btn && (bitwidth != 2 || splits > 1) ? btn : nullptr;
    const Path path = quantize_path(x, C);
    const CountTarget target{btn, count_workspace};
    const bool counted = btn && bitwidth == 2 && items * (words_per_item / 4 + 1) < 0x7fffffffL &&
                         (count_workspace || (words_per_item <= 64 && PC <= kOneSliceUnits));
    // an item of several slices, or whose counts would be read back (words_per_item <= 128: one slice, no second launch)
    if (btn && bitwidth == 2 && words_per_item > (counted ? 128 : 0) && quantize_items_supported(false, false, items, pixels_per_item, C))
        return launch_quantize_items(x, ths, false, items, pixels_per_item, C, qx, btn, stream);
    if (counted && path != Path::tile) {
        const floatx4 *x4 = reinterpret_cast<const floatx4 *>(x);
        uint32_t *q32 = reinterpret_cast<uint32_t *>(qx);
        auto launch = [&](auto whole, auto ragged, long rows, int lds) {
            const long slices = (words_per_item + rows - 1) / rows;
            const dim3 grid((unsigned)(items * slices));
            const Counts counts{slices == 1 ? btn : count_workspace, (int)slices};
            if (path == Path::whole) whole<<<grid, dim3(kThreads), lds, stream>>>(x4, ths, q32, words_per_item, counts);
            else ragged<<<grid, dim3(kThreads), lds, stream>>>(x4, ths, q32, words_per_item, counts, RaggedRows{C, make_div32((uint32_t)PC)});
            finish_counts(target, items, (int)slices, stream);
        };
        // (units of 128 rows for streaming and 32 for launches too small to fill the chip, as above)
        if (words_per_item > 32 && words_per_item <= 128) launch(quantize_rows64_count<8, false>, quantize_rows_ragged_count<8, false>, 128, 0);
        else if (items * words_per_item <= kSmallLaunchBlocks * 128) launch(quantize_rows64_count<2, false>, quantize_rows_ragged_count<2, false>, 32, 0);
        else launch(quantize_rows64_count<8, true>, quantize_rows_ragged_count<8, true>, 128, kStreamLds);
        return hipGetLastError();
    }
    if (counted) {
        launch_quantize_tile<2>(x, ths, pixels, pixels_per_item, items, C, qx, nullptr, &target, nullptr, stream);
        return hipGetLastError();
    }
    hipError_t e = hipSuccess;
    if (path != Path::tile) {
        if (bitwidth == 2) e = launch_rows<2>(path, x, ths, pixels, pixels_per_item, items, C, qx, zeroed, weights, stream);
        else e = launch_rows<1>(path, x, ths, pixels, pixels_per_item, items, C, qx, zeroed, weights, stream);
    } else if (bitwidth == 2) {
        launch_quantize_tile<2>(x, ths, pixels, pixels_per_item, items, C, qx, zeroed, nullptr, weights, stream);
    } else {
        launch_quantize_tile<1>(x, ths, pixels, pixels_per_item, items, C, qx, zeroed, nullptr, weights, stream);
    }
    if (e != hipSuccess) return e;
    if (btn && bitwidth == 2) launch_btn_popcount(qx, btn, items, words_per_item, splits, stream);
    return hipGetLastError();
}

hipError_t launch_patch_weights(const WeightJob &job, hipStream_t stream)
{
    patch_weights<<<dim3(job.blocks), dim3(kThreads), 0, stream>>>(job);
    return hipGetLastError();
}

// Words of an NCHW tensor whose pixels have several: whether the form that gathers each wave's output into whole runs of them takes it (PC even,
// enough pixels for a wave on every SIMD), `unit` words a thread, and else how many waves a last word of at most 32 channels takes, apart from the
// others (0: as many as those).  1500 measured calls (quantize_last_words_timings.txt), gathered or all words alike / by this rule, us:
//   * A thread of the gathering form goes through such a last word as long as through the others.  With two words a thread (PC = 2, 6, 10 ..)
//     units are the sooner form then: one plane 46 80x80 of 80 24.6 / 20.0, 3287 7x7 of 348 61.2 / 51.1.  With four the form's whole lines are worth
//     more (120 56x56 of 209 62.5 in units, 58.5; 45 64x64 of 453 69.8, 62.6), unless planes are not whole fours, of which units read no less:
//     1263 of 205 pixels and 224 channels 55.4 / 51.2; at more than four words only where they are shorter than a wave.
//   * Last words apart are half of PC = 2's work: 5 % from 4 MB of one plane on, 10 % from 30, of two planes 2 % from 6 MB; a third to an
//     eighth, 2 % from 40 MB on, one plane only.  Below that a launch is as long as its longest wave, which such a unit makes 0.1 us later (2 47x61 of
//     261 4.04, 3.88), and four words of two planes are half a cache line a pixel, which the last word then reaches later.
// All of them: 0.977 of the forms' time that know no such words, the best form of each 0.969, 15 more than 3 % slower, the worst 9; units with the last
// words apart everywhere 0.990, 395 more than 3 % slower, the worst 44.
PlaneForm plane_form(int bitwidth, long N, long HW, int C)
{
    const int PC = (C + kWordBits - 1) / kWordBits, few = last_word_waves(C, PC), unit = PC % 4 == 0 ? 4 : PC % 2 == 0 ? 2 : 1;
    const long gather_waves = (N * ((HW + 3) / 4) + 63) / 64 * (PC / unit), values = N * HW * C;
    const bool units = few && (unit == 2 ? bitwidth == 1 || PC == 2 : bitwidth == 1 && HW % 4 != 0 && (PC == 4 || HW < 64));
    const bool apart = PC == 2 ? values >= (bitwidth == 1 ? 1L << 20 : 3L << 19) : bitwidth == 1 && PC <= 8 && values >= 10L << 20;
    return {HW >= 4 && unit > 1 && gather_waves >= 1024 && !units, unit, apart ? few : 0};
}

hipError_t launch_quantize_nchw(const float *x, const Thresholds &ths, int bitwidth, int N, int C, long HW, uint64_t *qx,
                                int32_t *btn, int32_t *count_workspace, hipStream_t stream, const WeightJob *weights)
{
    const int PC = (C + kWordBits - 1) / kWordBits;
    const long words_per_item = HW * PC;
    const int splits = btn && bitwidth == 2 ? count_splits(N, words_per_item) : 1;
    int32_t *zeroed = btn && (bitwidth != 2 || splits > 1) ? btn : nullptr;
    const long pixels = (long)N * HW;
    const long runs = N * ((HW + 3) / 4);
    const bool counted = btn && bitwidth == 2 && (count_workspace || (words_per_item <= 64 && PC <= kOneSliceUnits)) &&
                         N * (HW / 4 + 1) * PC < 0x7fffffffL;
    // an item of several slices (64 pixels and a word each at least), or whose counts would be read back
    if (btn && bitwidth == 2 && (!counted || (HW + 63) / 64 * PC > kOneSliceUnits) && quantize_items_supported(false, true, N, HW, C))
        return launch_quantize_items(x, ths, true, N, HW, C, qx, btn, stream);
    auto by_image = [&](long per_image) { return N * per_image < 0x7fffffffL ? make_div32((uint32_t)per_image) : Div32{0, 0}; };
    auto launch = [&](auto kernel, long blocks, int threads, long per_image) {
        kernel<<<dim3((unsigned)blocks), dim3(threads), 0, stream>>>(x, ordered(ths, blocks), qx, N, C, HW, PC, by_image(per_image), zeroed);
    };
    auto launch_weights = [&](auto kernel, long blocks, int threads, long per_image) {
        WeightJob job = *weights;
        job.blocks *= kThreads / threads;
        kernel<<<dim3((unsigned)blocks + job.blocks), dim3(threads), 0, stream>>>(x, ordered(ths, blocks), qx, N, C, HW, PC, by_image(per_image), job);
    };
    const PlaneForm words = plane_form(bitwidth, N, HW, C);
    const int unit = words.unit;
    int last = words.last;
    const long gather_waves = (runs + 63) / 64 * (PC / unit);
    if (gather_waves > 0x7fffffffL) return hipErrorInvalidValue;
    const long gather_slices = (runs / N + 63) / 64 * (PC / unit);
    if (words.gather && (uintptr_t)qx % 16 == 0 && !(counted && gather_slices > 1 && !count_workspace)) {
        if (counted) {
            const long slices = gather_slices;
            auto launch_counted = [&](auto kernel) {
                kernel<<<dim3((unsigned)(N * slices)), dim3(64), 0, stream>>>(x, ths, qx, (int)slices, C, HW, PC, Div32{0, 0}, slices == 1 ? btn : count_workspace);
            };
            launch_counted(unit == 4 ? quantize_nchw_gather<2, 4, false, true> : quantize_nchw_gather<2, 2, false, true>);
            finish_counts(CountTarget{btn, count_workspace}, N, (int)slices, stream);
            return hipGetLastError();
        }
        auto pick = [&](auto even, auto any, auto even_weights, auto any_weights) {
            const long per_image = HW % 4 ? (HW + 3) / 4 : HW;  // runs, or pixels
            if (weights) launch_weights(HW % 4 ? any_weights : even_weights, gather_waves, 64, per_image);
            else launch(HW % 4 ? any : even, gather_waves, 64, per_image);
        };
        if (unit == 4 && bitwidth == 2)
            pick(quantize_nchw_gather<2, 4, true>, quantize_nchw_gather<2, 4, false>, quantize_nchw_gather<2, 4, true, false, true>, quantize_nchw_gather<2, 4, false, false, true>);
        else if (unit == 4)
            pick(quantize_nchw_gather<1, 4, true>, quantize_nchw_gather<1, 4, false>, quantize_nchw_gather<1, 4, true, false, true>, quantize_nchw_gather<1, 4, false, false, true>);
        else if (bitwidth == 2)
            pick(quantize_nchw_gather<2, 2, true>, quantize_nchw_gather<2, 2, false>, quantize_nchw_gather<2, 2, true, false, true>, quantize_nchw_gather<2, 2, false, false, true>);
        else
            pick(quantize_nchw_gather<1, 2, true>, quantize_nchw_gather<1, 2, false>, quantize_nchw_gather<1, 2, true, false, true>, quantize_nchw_gather<1, 2, false, false, true>);
    } else {
        // waves per word: as many as it has parts of 16 channels
        const int split = C <= 16 ? 1 : C <= 32 ? 2 : 4;
        // One pixel a thread until four give two waves per SIMD (32 x 64 x 56 x 56: 4.4 us, with four 4.8; 53 MB of 57 x 57
        // planes: 14.1 us, with four 11.9).
        bool four = HW >= 4 && (runs + 63) / 64 * PC * split >= 2048;
        // Past the caches where the tensor is large next to them and a wave reads whole lines, i.e. its kilobyte of a plane
        // is not mostly a plane's end: 128 x 64 x 112 x 112 73.6 -> 67.6 us, but 128 x 512 x 28 x 28 38.9 -> 44.5.  Runs that straddle
        // lines fetch them twice then, from HBM if x is larger than the 256 MB cache: N=64 57x57x64 11.2 -> 10.2, 75x75 17.0 -> 16.5,
        // but N=40 151x151 (234 MB) 46.2 -> 48.3.
        const bool stream_past = four && split == 4 && pixels * C >= (8L << 20) && HW >= 2048 && (HW % 4 == 0 || pixels * C < (32L << 20));
        const int groups = kWavesPerBlock / split;
        // counted: units end with the image, and a last one that is mostly empty weighs more with four
        const long padded1 = (HW + 64 * groups - 1) / (64 * groups), padded4 = (HW + 256 * groups - 1) / (256 * groups) * 4;
        if (counted && HW % 4 == 0 && padded1 * 8 < padded4 * 7) four = false;
        if (counted) {
            const long units = plane_units(((four ? runs / N : HW) + 64 * groups - 1) / (64 * groups), PC, last);
            const int slices = units <= kOneSliceUnits ? 1 : (int)units;
            auto launch_counted = [&](auto kernel) {
                kernel<<<dim3((unsigned)(N * slices)), dim3(kThreads), 0, stream>>>(x, ths, qx, C, HW, PC, (int)units,
                                                                                   Counts{slices == 1 ? btn : count_workspace, slices});
            };
            if (stream_past) launch_counted(last ? quantize_nchw_count<4, 4, true, true> : quantize_nchw_count<4, 4, true>);
            else if (last) launch_counted(four ? quantize_nchw_count<4, 4, false, true> : quantize_nchw_count<1, 4, false, true>);
            else if (four) launch_counted(split == 4 ? quantize_nchw_count<4, 4> : split == 2 ? quantize_nchw_count<4, 2> : quantize_nchw_count<4, 1>);
            else launch_counted(split == 4 ? quantize_nchw_count<1, 4> : split == 2 ? quantize_nchw_count<1, 2> : quantize_nchw_count<1, 1>);
            finish_counts(CountTarget{btn, count_workspace}, N, slices, stream);
            return hipGetLastError();
        }
        const long blocks = plane_units(((four ? runs : pixels) + 64 * groups - 1) / (64 * groups), PC, last);
        if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
        auto form_of = [&](auto vec, auto parts, auto past, auto with_last) {
            constexpr int VEC = decltype(vec)::value, PARTS = decltype(parts)::value;
            constexpr bool PAST = decltype(past)::value, LAST = decltype(with_last)::value;
            if (weights) launch_weights(bitwidth == 2 ? quantize_nchw_weights<2, VEC, PARTS, PAST, LAST> : quantize_nchw_weights<1, VEC, PARTS, PAST, LAST>, blocks, kThreads, (HW + VEC - 1) / VEC);
            else launch(bitwidth == 2 ? quantize_nchw<2, VEC, PARTS, PAST, LAST> : quantize_nchw<1, VEC, PARTS, PAST, LAST>, blocks, kThreads, (HW + VEC - 1) / VEC);
        };
        auto form = [&](auto vec, auto parts, auto past) {
            if constexpr (decltype(parts)::value == 4) {
                if (last) return form_of(vec, parts, past, std::true_type());
            }
            form_of(vec, parts, past, std::false_type());
        };
        using std::integral_constant;
        auto parts = [&](auto vec) {
            if (split == 4) form(vec, integral_constant<int, 4>(), std::false_type());
            else if (split == 2) form(vec, integral_constant<int, 2>(), std::false_type());
            else form(vec, integral_constant<int, 1>(), std::false_type());
        };
        if (stream_past) form(integral_constant<int, 4>(), integral_constant<int, 4>(), std::true_type());
        else if (four) parts(integral_constant<int, 4>());
        else parts(integral_constant<int, 1>());
    }
    if (btn && bitwidth == 2) launch_btn_popcount(qx, btn, N, words_per_item, splits, stream);
    return hipGetLastError();
}

hipError_t launch_quantize_format(const float *x, const float *ths_values, int format, long pixels_per_item, long items, int C,
                                  uint64_t *qx, hipStream_t stream, const WeightJob *weights)
{
    const Thresholds ths = given_thresholds(ths_values);
    const long pixels = items * pixels_per_item;
    if (format != 4 && format != 5) return hipErrorInvalidValue;
    const Path path = quantize_path(x, C);
    if (path != Path::tile)  // a row is 16 bytes of either format
        return format == 4 ? launch_rows<4>(path, x, ths, pixels, pixels_per_item, items, C, qx, nullptr, weights, stream)
                           : launch_rows<5>(path, x, ths, pixels, pixels_per_item, items, C, qx, nullptr, nullptr, stream);
    if (format == 4) launch_quantize_tile<4>(x, ths, pixels, pixels_per_item, items, C, qx, nullptr, nullptr, weights, stream);
    else launch_quantize_tile<5>(x, ths, pixels, pixels_per_item, items, C, qx, nullptr, nullptr, weights, stream);
    return hipGetLastError();
}

bool quantize_strided_supported(const float *x, int H, int W, int C, int OH, int OW)
{
    const long PC = C / kWordBits;
    return C % kWordBits == 0 && (uintptr_t)x % 16 == 0 && OW * PC < 65536 && PC < 65536;
}

hipError_t launch_quantize_strided(const float *x, const Thresholds &ths, int bitwidth, int N, int H, int W, int C, int OH,
                                   int OW, int s1, int s2, uint64_t *qx, hipStream_t stream)
{
    const int PC = C / kWordBits;
    const dim3 block(64);
    const floatx4 *x4 = reinterpret_cast<const floatx4 *>(x);
    uint32_t *q32 = reinterpret_cast<uint32_t *>(qx);
    const long waves = (long)((OW * PC + kRowsPerWave - 1) / kRowsPerWave) * N * OH;
    if (waves <= kSmallLaunchBlocks * kWavesPerBlock) {  // latency-bound: four times the waves, two loads per lane each
        const dim3 grid((unsigned)((OW * PC + 7) / 8), (unsigned)(N * OH));
        if (bitwidth == 2)
            quantize_rows64_strided<2, 2><<<grid, block, 0, stream>>>(x4, ths, q32, H, W, PC, OH, OW, s1, s2, make_fastdiv(PC));
        else
            quantize_rows64_strided<1, 2><<<grid, block, 0, stream>>>(x4, ths, q32, H, W, PC, OH, OW, s1, s2, make_fastdiv(PC));
        return hipGetLastError();
    }
    const dim3 grid((unsigned)((OW * PC + kRowsPerWave - 1) / kRowsPerWave), (unsigned)(N * OH));
    if (bitwidth == 2)
        quantize_rows64_strided<2><<<grid, block, 0, stream>>>(x4, ths, q32, H, W, PC, OH, OW, s1, s2, make_fastdiv(PC));
    else
        quantize_rows64_strided<1><<<grid, block, 0, stream>>>(x4, ths, q32, H, W, PC, OH, OW, s1, s2, make_fastdiv(PC));
    return hipGetLastError();
}

}  // namespace tab
