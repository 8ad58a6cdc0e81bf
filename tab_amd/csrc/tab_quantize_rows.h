// The streaming quantizer, by the workgroup: the body of quantize_rows64 and quantize_rows_ragged and of their forms that lay a
// convolution's weights out beside them (tab_quantize.hip).
#pragma once
#include "tab_conv_stage.h"
#include "tab_pack.h"

namespace tab {
namespace {

typedef uint32_t PackedPair __attribute__((ext_vector_type(4), aligned(8)));  // two words, aligned to one

constexpr int kQuantizeWaves = 4;  // of a workgroup
constexpr int kLoadsPerLane = 8;   // float4 loads in flight per lane

// Rows of 64 channels, one packed element each.  WholeRows: C % 64 == 0 and X 16-byte aligned.  RaggedRows: any C, any X aligned to its
// floats; row pixel * PC + w holds channels 64 w ... of its pixel, fewer than 64 in the pixel's last one.
struct WholeRows {};
struct RaggedRows {
    int C;
    Div32 div_pc;
};

// What a lane holds of the wave's rows; of a ragged row also which of its four channels exist (bit e) and how many pixels it
// lies behind the one that the wave begins in.
template <int LOADS>
struct RowLoads {
    floatx4 v[LOADS];
    uint32_t exist[LOADS], pixel[LOADS];
    bool one_word[LOADS];  // of 32 channels: the last 32 of the row do not exist
    long first_pixel;
};

// Rows row0 ... row0 + live - 1; a row past the end reads the last one again (not stored): straight-line loads, no branch per load.
// A small tensor is likely to sit in the caches (it was just written, or is read again): plain loads; a large one (NT) streams past
// them: non-temporal loads (plain ones are 8-11 % slower at 400 MB and more).
template <bool NT, int LOADS>
__device__ __forceinline__ void load_rows(const WholeRows, const floatx4 *__restrict__ x, long row0, uint32_t live, int sub, int l, RowLoads<LOADS> &rows)
{
    const floatx4 *const src = x + row0 * 16;  // 32-bit offsets from a scalar address leave registers for one more wave per SIMD
#pragma unroll
    for (int u = 0; u < LOADS; u++) {
        const floatx4 *at = &src[min((uint32_t)(u * 4 + sub), live - 1) * 16 + l];
        rows.v[u] = NT ? __builtin_nontemporal_load(at) : *at;
    }
}

// The same 16-byte loads wherever a row begins; they need 4-byte alignment only, and what a row's last load takes of the next pixel is
// masked away.  The descriptor ends with the wave's last row: past it loads give zeros.
template <bool NT, int LOADS>
__device__ __forceinline__ void load_rows(const RaggedRows ragged, const floatx4 *__restrict__ x, long row0, uint32_t live, int sub, int l, RowLoads<LOADS> &rows)
{
    const uint32_t C = (uint32_t)ragged.C, PC = (C + 63u) >> 6;
    const long pixel0 = row0 < 0x7fffffffL ? (long)div32((uint32_t)row0, ragged.div_pc) : row0 / (long)PC;
    const uint32_t word0 = (uint32_t)(row0 - pixel0 * (long)PC);
    rows.first_pixel = pixel0;
    // bytes from the first row on; the wave's rows are less than 8 KB of x, so that 32 bits hold them whatever C is
    auto begins = [&](uint32_t pixel, uint32_t word) { return (pixel * C + (word - word0) * 64u) * 4u; };
    const uint32_t last = word0 + live - 1, last_pixel = div32(last, ragged.div_pc), last_word = last - last_pixel * PC;
    const uint32_t bytes = begins(last_pixel, last_word) + min(C - last_word * 64u, 64u) * 4u;
    const float *const src = reinterpret_cast<const float *>(x) + pixel0 * (long)C + (long)word0 * 64;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)src, 0, (int)bytes, kBufferFlags);
#pragma unroll
    for (int u = 0; u < LOADS; u++) {
        const uint32_t row = word0 + min((uint32_t)(u * 4 + sub), live - 1), pixel = div32(row, ragged.div_pc), word = row - pixel * PC;
        const int here = (int)(C - word * 64u) - 4 * l;
        rows.pixel[u] = pixel;
        rows.one_word[u] = C - word * 64u <= 32u;
        rows.exist[u] = here >= 4 ? 15u : here > 0 ? (1u << here) - 1u : 0u;
        const uint32_t offset = begins(pixel, word) + 16u * (uint32_t)l;
        const u32x4 w = NT ? __builtin_amdgcn_raw_buffer_load_b128(rsrc, offset, 0, kStreamingStore) : __builtin_amdgcn_raw_buffer_load_b128(rsrc, offset, 0, 0);
        rows.v[u] = floatx4{__uint_as_float(w[0]), __uint_as_float(w[1]), __uint_as_float(w[2]), __uint_as_float(w[3])};
    }
}

// Lane layout: a 16-lane DPP row reads one row of 64 channels as 16 float4 (256 B contiguous),
// a wave reads 4 consecutive rows per load (1 KB contiguous) and keeps kLoadsPerLane loads
// in flight; pack_row turns the compare bits of the row's lanes into its packed element.
// BITS = 1 or 2 (the reference's bit widths), or the format of conv type 4 or 5; LOADS = 8 (128 rows per
// workgroup) for streaming, 2 for launches too small to fill the chip.
// block: the workgroup's number among those that quantize.
// OWN: thresholds are partial sums to be added up (a form of its own: the code that is not run costs calls with given thresholds 2 to 4 %).
template <int BITS, int LOADS, bool OWN, class Rows>
__device__ __forceinline__ void quantize_rows_block(const Rows kind, const floatx4 *__restrict__ x, const Thresholds &ths, uint32_t *__restrict__ q, long rows,
                                                    long rows_per_item, Div32 div_item, uint32_t block)
{
    constexpr bool RAGGED = std::is_same<Rows, RaggedRows>::value;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // scalar: so are row0 and the item test below
    const int sub = lane >> 4;  // which of the 4 rows of a load
    const int l = lane & 15;    // float4 within the row
    const long row0 = ((long)block * kQuantizeWaves + wave) * (4 * LOADS);
    if (row0 >= rows) return;
    long row_last = row0 + (4 * LOADS) - 1;
    if (row_last > rows - 1) row_last = rows - 1;

    // The wave's items (scalar; div_item.mul == 0 says that rows reach 2^31 and the division takes 64 bits).  Partial sums are
    // requested before x, whose loads do not wait for the division otherwise.
    long item_first = 0, item_last = 0;
    auto find_items = [&] {
        item_first = div_item.mul ? (long)div32((uint32_t)row0, div_item) : row0 / rows_per_item;
        item_last = div_item.mul ? (long)div32((uint32_t)row_last, div_item) : row_last / rows_per_item;
    };
    floatx4 requested = {};
    if (OWN) {
        find_items();
        requested = request_threshold(ths, item_first);
    }
    uint32_t *const dst = q + row0 * (BITS != 1 ? 4 : 2);
    const uint32_t live = (uint32_t)(row_last - row0) + 1;
    RowLoads<LOADS> held;
    load_rows<LOADS != 2>(kind, x, row0, live, sub, l, held);
    if (!OWN) find_items();
    const float t_first = OWN ? finish_threshold(ths, item_first, requested) : given_threshold(ths, item_first);
    const float t_last = item_last == item_first ? t_first : OWN ? wave_threshold(ths, item_last) : given_threshold(ths, item_last);

    auto finish = [&](int u, float t) {
        const uint32_t r = u * 4 + sub;
        uint32_t sign, nz, out[4];
        compare4<BITS>(held.v[u], t, sign, nz);
        if (RAGGED) {  // channels that do not exist stay 0 (TAB_GEMM.cu:203-206)
            sign &= held.exist[u];
            nz &= held.exist[u];
        }
        pack_row<BITS, RAGGED>(sign, nz, l, out);  // lane 0 stores the whole element (8 or 16 bytes) at once
        if constexpr (RAGGED && BITS == 5) {
            // 32 channels a word: a row is two words, or one where the last 32 channels of the pixel do not exist
            const bool odd = ((uint32_t)kind.C & 63u) - 1u < 32u;  // 1 .. 32 channels in the last row
            uint32_t *const at = q + 2 * (2 * row0 - (odd ? held.first_pixel : 0)) + 2u * (2u * r - (odd ? held.pixel[u] : 0u));
            if (r < live && l == 0) {
                if (held.one_word[u]) *reinterpret_cast<uintx2 *>(at) = uintx2{out[0], out[1]};
                else *reinterpret_cast<PackedPair *>(at) = PackedPair{out[0], out[1], out[2], out[3]};
            }
        } else if (BITS != 1) {
            if (r < live && l == 0) *reinterpret_cast<uintx4 *>(dst + r * 4) = uintx4{out[0], out[1], out[2], out[3]};
        } else {
            if (r < live && l == 0) *reinterpret_cast<uintx2 *>(dst + r * 2) = uintx2{out[0], out[1]};
        }
    };
    // copies of the loop under scalar branches: the common one has no load but x in flight, so each load is
    // waited for on its own
    if (item_last == item_first) {
#pragma unroll
        for (int u = 0; u < LOADS; u++) finish(u, t_first);
    } else if (item_last == item_first + 1) {
        const uint32_t border = (uint32_t)(item_last * rows_per_item - row0);  // where the second begins
#pragma unroll
        for (int u = 0; u < LOADS; u++) finish(u, (uint32_t)(u * 4 + sub) < border ? t_first : t_last);
    } else if (!OWN) {  // items of fewer rows than the wave (partial sums are those of 64 rows and more)
        const uint32_t before = (uint32_t)(row0 - item_first * rows_per_item);  // rows of the first item in front of the wave
#pragma unroll
        for (int u = 0; u < LOADS; u++) {
            const uint32_t at = before + min((uint32_t)(u * 4 + sub), live - 1);
            finish(u, given_threshold(ths, item_first + at / (uint32_t)rows_per_item));
        }
    }
}

}  // namespace
}  // namespace tab
