// Ternary quantizer of small items, a workgroup of four or sixteen waves each: what needs the whole item - its threshold, the count of its nonzero
// values - is found in the same launch.
//
// With slices of an item in workgroups of their own, the sums of |x| or the counts take a launch before or behind the quantizer: 2.4 us on
// the GPU and 2.8 of the host, more than a small item's reading.  Here a workgroup reads its item once for the sum, all loads requested at
// once, and a second time, out of the L2, to pack it.  Bound by the latency of one CU's reads and their 64 bytes a cycle, hence the
// limits: items of 26 K values with their counts (24 K of ragged rows: 300 14x14x96 10.9 / 11.5), of 12 K with their thresholds, and not too many of
// them (quantize_items_supported).  Quantizer and counts in two launches / here, graph replays,
// us: 136 14x14x64 5.3 / 4.2 (NCHW 6.1 / 4.0), 256 7x7x512 9.4 / 8.1, 79 25x15x64 5.5 / 4.7, but 16 14x14x256 (49 K) 4.8 / 6.5; sums and quantizer:
// 91 rows of 576 4.6 / 3.7, 153 of 5376 5.4 / 4.3, 2000 of 2000 11.0 / 8.4, but 79 25x15x64 (23 K) 6.1 / 6.9.  Called one after the other such
// quantizers take 7.6 us in two launches, which is the host's time, and 5.0 in one; a ternary linear layer of 2048 inputs 11.4 in three, 8.5 in two.
#include "tab_pack.h"
#include "tab_patch_weights.h"
#include "tab_quantize_rows.h"

namespace tab {
namespace {

constexpr int kSumThreads = 256;  // of a slice of |x|, as in abs_sum_partial

// Waves that share 64 pixels of an item's channels (NCHW), sixteen channels each.
__host__ __device__ __forceinline__ int plane_parts_log(int C) { return C > 32 ? 2 : (C > 16 ? 1 : 0); }

// scale * the sum of |x|: slices and their sums as abs_sum_partial makes them, to the last bit the same, a slice to four waves.
template <int WAVES>
__device__ __forceinline__ float item_threshold(const float *__restrict__ src, long per_item, const Thresholds &ths, float *scratch)
{
    constexpr int kSumGroups = WAVES * 64 / kSumThreads, SLICES = WAVES == 4 ? 1 : 2, LOADS = 4;  // of a group in flight
    const int splits = ths.splits, thread = threadIdx.x % kSumThreads, lane = threadIdx.x & 63;
    const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / kSumThreads), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64) % (kSumThreads / 64);
    const long slice = ((per_item + splits - 1) / splits + 3) & ~3L;
    for (int s0 = group; s0 < splits; s0 += kSumGroups * SLICES) {
        float sum[SLICES];
        floatx4 v[SLICES][LOADS];
        auto add = [](const floatx4 w) { return (__builtin_fabsf(w[0]) + __builtin_fabsf(w[1])) + (__builtin_fabsf(w[2]) + __builtin_fabsf(w[3])); };
        auto begin_of = [&](int j) { return (s0 + j * kSumGroups) * slice; };
        auto end_of = [&](int j) { return begin_of(j) + slice < per_item ? begin_of(j) + slice : per_item; };
        const bool aligned = ((uintptr_t)src & 15) == 0;  // (a slice begins on a multiple of four)
#pragma unroll
        for (int j = 0; j < SLICES; j++) {
            sum[j] = 0.f;
            if (s0 + j * kSumGroups >= splits) break;  // uniform
            const long begin = begin_of(j), n4 = begin < end_of(j) ? (end_of(j) - begin) / 4 : 0;
#pragma unroll
            for (int k = 0; k < LOADS; k++) {
                v[j][k] = floatx4{0.f, 0.f, 0.f, 0.f};
                if (aligned && thread + k * kSumThreads < n4) v[j][k] = reinterpret_cast<const floatx4 *>(src + begin)[thread + k * kSumThreads];
            }
        }
#pragma unroll
        for (int j = 0; j < SLICES; j++) {
            if (s0 + j * kSumGroups >= splits) break;
            const long begin = begin_of(j), end = end_of(j), n4 = begin < end ? (end - begin) / 4 : 0;
            if (aligned) {
#pragma unroll
                for (int k = 0; k < LOADS; k++)
                    if (thread + k * kSumThreads < n4) sum[j] += add(v[j][k]);
                for (long i = thread + LOADS * kSumThreads; i < n4; i += kSumThreads) sum[j] += add(reinterpret_cast<const floatx4 *>(src + begin)[i]);
                for (long i = begin + n4 * 4 + thread; i < end; i += kSumThreads) sum[j] += __builtin_fabsf(src[i]);
            } else {
                for (long i = begin + thread; i < end; i += kSumThreads) sum[j] += __builtin_fabsf(src[i]);
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) sum[j] += __shfl_down(sum[j], off, 64);
            if (lane == 0) scratch[(s0 + j * kSumGroups) * (kSumThreads / 64) + wave] = sum[j];
        }
    }
    __syncthreads();
    auto total = [&](int s) {
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < kSumThreads / 64; w++) t += scratch[s * (kSumThreads / 64) + w];
        return t;
    };
    double sum = 0.0;
    for (int s = lane; s < splits; s += 64) sum += (double)total(s);
    const float t = (float)(wave_sum_f64(sum) * ths.scale);
    return __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(t)));
}

// x as [C][pixels]; 1 << PARTS_LOG waves share 64 pixels of a word
template <int PARTS_LOG> struct PlaneRows { static constexpr int kPartsLog = PARTS_LOG; };

template <class Rows> constexpr bool is_planes = false;
template <int PARTS_LOG> constexpr bool is_planes<PlaneRows<PARTS_LOG>> = true;

// OWN: ths has the number of slices and the scale of the thresholds to be found, else the thresholds.  btn: the counts, or null.
template <int WAVES, class Rows, bool OWN>
__device__ __forceinline__ void quantize_one_item(const Rows kind, const float *__restrict__ x, const Thresholds &ths, uint64_t *__restrict__ q, int32_t *btn,
                                                  int pixels, int C, int item)
{
    __shared__ alignas(16) uint32_t scratch[1024];  // sums of slices; words of planes; counts
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long per_item = (long)pixels * C;
    const float *const src = x + item * per_item;
    const float t = OWN ? item_threshold<WAVES>(src, per_item, ths, reinterpret_cast<float *>(scratch)) : given_threshold(ths, item);
    if (OWN) __syncthreads();
    const int PC = (C + kWordBits - 1) / kWordBits;
    int count = 0;
    if constexpr (is_planes<Rows>) {  // a lane takes sixteen channels of its pixel
        constexpr int PARTS = 1 << Rows::kPartsLog, GROUPS = WAVES / PARTS;
        uint16_t(*const halves)[2][64] = reinterpret_cast<uint16_t(*)[2][64]>(scratch);  // of a wave
        const int part = wave % PARTS, group = wave / PARTS;
        const int pixel_groups = (pixels + 63) / 64, tasks = pixel_groups * PC;
        uint64_t *const dst = q + (long)item * pixels * PC * 2;
        for (int task0 = 0; task0 < tasks; task0 += GROUPS) {
            const int task = task0 + group, pc = task % PC, pixel = task / PC * 64 + lane;
            const int c0 = pc * kWordBits + part * 16, channels = task < tasks ? (C - c0 < 16 ? C - c0 : 16) : 0;
            const float *const from = src + (long)c0 * pixels + (pixel < pixels ? pixel : pixels - 1);
            float v[16];
#pragma unroll
            for (int u = 0; u < 16; u++) {
                v[u] = 0.f;
                if (u < channels) v[u] = from[(long)u * pixels];
            }
            uint32_t less = 0, more = 0;
#pragma unroll
            for (int u = 15; u > 0; u -= 4) {
                shift_in_less4(less, v[u], v[u - 1], v[u - 2], v[u - 3], -t);
                shift_in_more4(more, v[u], v[u - 1], v[u - 2], v[u - 3], t);
            }
            const uint32_t exist = channels <= 0 ? 0u : 0xffffu >> (16 - channels);
            less &= exist;
            more &= exist;
            count += pixel < pixels ? __builtin_popcount(less | more) : 0;
            if (PARTS == 1) {
                if (task < tasks && pixel < pixels) *reinterpret_cast<uintx4 *>(dst + (long)pixel * 2) = uintx4{less & ~more, 0u, less | more, 0u};
                continue;
            }
            halves[wave][0][lane] = (uint16_t)(less & ~more);
            halves[wave][1][lane] = (uint16_t)(less | more);
            __syncthreads();
            if (part < 2 && task < tasks && pixel < pixels) {  // a wave a plane
                uint64_t word = 0;
#pragma unroll
                for (int p = 0; p < PARTS; p++) word |= (uint64_t)halves[wave - part + p][part][lane] << (16 * p);
                dst[((long)pixel * PC + pc) * 2 + part] = word;
            }
            if (task0 + GROUPS < tasks) __syncthreads();
        }
    } else {
        constexpr int LOADS = kLoadsPerLane;
        const int sub = lane >> 4, l = lane & 15, rows = pixels * PC;
        const long first = (long)item * rows;
        uint32_t *const dst = reinterpret_cast<uint32_t *>(q) + first * 4;
        for (int at = wave * (4 * LOADS); at < rows; at += WAVES * 4 * LOADS) {
            const uint32_t live = (uint32_t)(rows - at < 4 * LOADS ? rows - at : 4 * LOADS);
            RowLoads<LOADS> held;
            load_rows<false>(kind, reinterpret_cast<const floatx4 *>(x), first + at, live, sub, l, held);
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
                if (r < live && l == 0) *reinterpret_cast<uintx4 *>(dst + (at + r) * 4) = uintx4{out[0], out[1], out[2], out[3]};
            }
        }
    }
    if (btn == nullptr) return;
    __syncthreads();
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) count += __shfl_down(count, off, 64);
    if (lane == 0) scratch[wave] = (uint32_t)count;
    __syncthreads();
    if (threadIdx.x == 0) {
        int total = 0;
#pragma unroll
        for (int w = 0; w < WAVES; w++) total += (int)scratch[w];
        btn[item] = total;
    }
}

template <int WAVES, class Rows, bool OWN>
__global__ __launch_bounds__(64 * WAVES) void quantize_items(const float *__restrict__ x, const Thresholds ths, uint64_t *__restrict__ q, int32_t *btn,
                                                             int pixels, int C, const Rows kind)
{
    quantize_one_item<WAVES, Rows, OWN>(kind, x, ths, q, btn, pixels, C, (int)blockIdx.x);
}

// An item's values at most, words NHWC as 64 of them; NCHW pieces of 64 pixels and 16 channels, of which sixteen waves take a round.
constexpr long kCountedItem = 26 * 1024, kCountedRagged = 24 * 1024, kOwnItem = 12 * 1024, kCountedPieces = 32, kOwnPieces = 16;
constexpr long kFewWaves = 4096;  // values up to which an item takes four waves

inline long item_pieces(long pixels, int C) { return (pixels + 63) / 64 * ((C + kWordBits - 1) / kWordBits) << plane_parts_log(C); }
inline bool four_waves(bool nchw, long items, long pixels, int C)
{
    // (from more items than CUs on two of sixteen waves share a CU: 300 10x10x96 NCHW with thresholds 8.0 in two launches, 9.6)
    return pixels * C <= kFewWaves && (!nchw || item_pieces(pixels, C) <= (items > device_compute_units() ? 16 : 4));
}

}  // namespace

// Where this kernel is the sooner one, of the calls it can take: 1177 measured ones of 0.3 to 500 MB (quantize_items_timings.txt).
// The limits on the items are those of a workgroup's cost: four waves start 0.7 a nanosecond, whatever they read, and sixteen, two of which a CU
// holds, are as slow as what one CU reads as soon as there are several rounds of them; the two launches stream.  Two launches / here, us: own
// thresholds 16384 rows of 8192 values 160 / 242, 46875 of 128 46 / 71, 8000 7x7x128 67 / 111, counts 2200 7x7x300 29.6 / 42.6, 2200 NCHW 14x14x128
// 43.5 / 50.3.  These rules take 0.882 of the two launches' time, the better of both ways 0.879 (all of them here: 0.967); of 702 choices four are more than
// 2 % slower, the worst 13.
bool quantize_items_supported(bool own, bool nchw, long items, long pixels, int C)
{
    if (pixels > kCountedItem / C || items >= 0x7fffffffL) return false;
    const long values = pixels * C, units = device_compute_units();
    const bool four = four_waves(nchw, items, pixels, C);
    if (nchw) {
        const long pieces = item_pieces(pixels, C);
        // (few channels leave the sums nothing to make up for: 46 21x21x27, thresholds and quantizer, 6.2 us in two launches, 7.1 in one)
        if (own)  // past a round, items that fill their lanes
            return C > 32 && values <= kOwnItem && pieces <= kOwnPieces &&
                   (items <= units || (four && (values >= 320 * pieces || (pieces <= 8 && items <= 4 * units))));
        if (four || pieces > kCountedPieces) return pieces <= kCountedPieces;
        if (pieces <= (items > units ? 12 : 8)) return false;  // waves would have nothing to do
        // Planes shorter than a wave: the other kernels take four pixels a thread only of planes of whole fours, and once x is
        // past the caches they read each cache line several times.  Other planes: as long as the other kernels have too few waves.
        if (pixels % 4 != 0 && pixels > 2 && pixels < 64) return true;
        return items * values <= 8L << 20 || (pixels <= 64 && items * values > 80L << 20);
    }
    // (up to 32 channels go by tiles: a row of 16 lanes a pixel would be mostly empty)
    const long rows = pixels * ((C + kWordBits - 1) / kWordBits);
    if (C <= 32 || rows * kWordBits > (own ? kOwnItem : C % kWordBits ? kCountedRagged : kCountedItem)) return false;
    if (!own) return C % kWordBits ? items <= units && (rows <= 256 || 4 * items > units) : items * values <= 24L << 20;
    if (!four) return items <= 2 * units && values % 4 == 0;  // (an item between two multiples of four values is summed a value a load)
    if (C % kWordBits == 0) return values >= 768 || items <= 6 * values;
    if (values < 1024) return 2 * items <= 5 * values;
    return items <= 32 * units || (values % 4 == 0 && values >= 1792);
}

hipError_t launch_quantize_items(const float *x, const Thresholds &ths, bool nchw, long items, long pixels, int C, uint64_t *qx, int32_t *btn, hipStream_t stream)
{
    // (1024 rows of 2048 values, thresholds and quantizer: four waves 4.8 us, sixteen 8.9, two launches 7.2)
    auto launch = [&](auto kind) {
        using Rows = decltype(kind);
        auto of = [&](auto waves) {
            constexpr int WAVES = decltype(waves)::value;
            auto kernel = ths.splits > 0 ? quantize_items<WAVES, Rows, true> : quantize_items<WAVES, Rows, false>;
            kernel<<<dim3((unsigned)items), dim3(64 * WAVES), 0, stream>>>(x, ths, qx, btn, (int)pixels, C, kind);
        };
        if (four_waves(nchw, items, pixels, C)) of(std::integral_constant<int, 4>());
        else of(std::integral_constant<int, 16>());
    };
    if (nchw && plane_parts_log(C) == 0) launch(PlaneRows<0>{});
    else if (nchw && plane_parts_log(C) == 1) launch(PlaneRows<1>{});
    else if (nchw) launch(PlaneRows<2>{});
    else if (C % kWordBits == 0 && (uintptr_t)x % 16 == 0) launch(WholeRows{});
    else launch(RaggedRows{C, make_div32((uint32_t)((C + kWordBits - 1) / kWordBits))});
    return hipGetLastError();
}

hipError_t launch_quantize_own(const float *x, float scale, bool nchw, long items, long pixels, int C, uint64_t *qx, hipStream_t stream)
{
    const long per_item = pixels * C;
    return launch_quantize_items(x, Thresholds{nullptr, (double)scale / (double)per_item, threshold_splits(items, per_item), 0}, nchw, items, pixels, C, qx, nullptr, stream);
}

}  // namespace tab
