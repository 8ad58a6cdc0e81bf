// The streaming quantizer of whole words, by the workgroup: the body of quantize_rows64 and of quantize_rows64_weights, which lays a
// convolution's weights out beside it (tab_quantize.hip).
#pragma once
#include "tab_pack.h"

namespace tab {
namespace {

constexpr int kQuantizeWaves = 4;  // of a workgroup
constexpr int kLoadsPerLane = 8;   // float4 loads in flight per lane

// Fast path, C % 64 == 0 and X 16-byte aligned.
// Lane layout: a 16-lane DPP row reads one 64-channel row as 16 float4 (256 B contiguous),
// a wave reads 4 consecutive rows per load (1 KB contiguous) and keeps kLoadsPerLane loads
// in flight; pack_row turns the compare bits of the row's lanes into its packed element.
// BITS = 1 or 2 (the reference's bit widths), or the format of conv type 4 or 5; LOADS = 8 (128 rows per
// workgroup) for streaming, 2 for launches too small to fill the chip.
// block: the workgroup's number among those that quantize.
// OWN: thresholds are partial sums to be added up (a form of its own: the code that is not run costs calls with given thresholds 2 to 4 %).
template <int BITS, int LOADS, bool OWN>
__device__ __forceinline__ void quantize_rows64_block(const floatx4 *__restrict__ x, const Thresholds &ths, uint32_t *__restrict__ q, long rows,
                                                      long rows_per_item, Div32 div_item, uint32_t block)
{
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
    // x and q from the wave's row on: 32-bit offsets from a scalar address leave registers for one more wave per SIMD
    const floatx4 *const src = x + row0 * 16;
    uint32_t *const dst = q + row0 * (BITS != 1 ? 4 : 2);
    const uint32_t live = (uint32_t)(row_last - row0) + 1;
    floatx4 v[LOADS];
#pragma unroll
    for (int u = 0; u < LOADS; u++) {
        // rows past the end read the last row again (not stored): straight-line loads, no branch per load
        const floatx4 *at = &src[min((uint32_t)(u * 4 + sub), live - 1) * 16 + l];
        // a small tensor is likely to sit in the caches (it was just written, or is read again): plain loads;
        // a large one streams past them: non-temporal loads (plain ones are 8-11 % slower at 400 MB and more)
        v[u] = LOADS == 2 ? *at : __builtin_nontemporal_load(at);
    }
    if (!OWN) find_items();
    const float t_first = OWN ? finish_threshold(ths, item_first, requested) : given_threshold(ths, item_first);
    const float t_last = item_last == item_first ? t_first : OWN ? wave_threshold(ths, item_last) : given_threshold(ths, item_last);

    auto finish = [&](int u, float t) {
        const uint32_t r = u * 4 + sub;
        uint32_t sign, nz, out[4];
        compare4<BITS>(v[u], t, sign, nz);
        pack_row<BITS>(sign, nz, l, out);  // lane 0 stores the whole element (8 or 16 bytes) at once
        if (BITS != 1) {
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
