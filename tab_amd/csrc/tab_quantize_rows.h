// The streaming quantizer of whole words, by the workgroup: quantize_rows64 (tab_quantize.hip) and the convolutions that quantize
// their successor's activation on the side (tab_conv_mfma_patch.h).
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
template <int BITS, int LOADS>
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

    floatx4 v[LOADS];
#pragma unroll
    for (int u = 0; u < LOADS; u++) {
        const long r = row0 + u * 4 + sub;
        // rows past the end read the last row again (not stored): straight-line loads, no branch per load
        const floatx4 *src = &x[(r < rows ? r : rows - 1) * 16 + l];
        // a small tensor is likely to sit in the caches (it was just written, or is read again): plain loads;
        // a large one streams past them: non-temporal loads (plain ones are 8-11 % slower at 400 MB and more)
        v[u] = LOADS == 2 ? *src : __builtin_nontemporal_load(src);
    }

    // The wave's items (scalar; div_item.mul == 0 says that rows reach 2^31 and the division takes 64 bits): with the
    // short division the threshold is in flight together with the loads of x instead of behind a long one.
    const long item_first = div_item.mul ? (long)div32((uint32_t)row0, div_item) : row0 / rows_per_item;
    const long item_last = div_item.mul ? (long)div32((uint32_t)row_last, div_item) : row_last / rows_per_item;
    const bool one_item = item_last == item_first;
    const float t_first = wave_threshold(ths, item_first);

    auto finish = [&](int u, float t) {
        const long r = row0 + u * 4 + sub;
        uint32_t sign, nz, out[4];
        compare4<BITS>(v[u], t, sign, nz);
        pack_row<BITS>(sign, nz, l, out);  // lane 0 stores the whole element (8 or 16 bytes) at once
        if (BITS != 1) {
            if (r < rows && l == 0) *reinterpret_cast<uintx4 *>(q + r * 4) = uintx4{out[0], out[1], out[2], out[3]};
        } else {
            if (r < rows && l == 0) *reinterpret_cast<uintx2 *>(q + r * 2) = uintx2{out[0], out[1]};
        }
    };
    // two copies of the loop under a scalar branch: the common one has no load but x in flight, so each load is
    // waited for on its own
    if (one_item) {
#pragma unroll
        for (int u = 0; u < LOADS; u++) finish(u, t_first);
    } else {
#pragma unroll
        for (int u = 0; u < LOADS; u++) {
            const long r = row0 + u * 4 + sub;
            finish(u, lane_threshold(ths, (r < rows ? r : rows - 1) / rows_per_item));
        }
    }
}

}  // namespace
}  // namespace tab
