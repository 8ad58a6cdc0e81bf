// Weights in the order in which the lanes of conv_mfma_patch read them.
#pragma once
#include "tab_common.h"

namespace tab {

// Pairs of words of a chunk, one for each half-wave: a tap's (kc even) or those of two neighbouring taps (kc = 1).
__host__ __device__ __forceinline__ int patch_pairs(int taps, int kc) { return kc == 1 ? (taps + 1) >> 1 : taps * (kc >> 1); }

namespace {

// [32 filters][chunk][pair of words][half-wave][filter]: a lane's item is its filter's word of the pair, zeros where there is none.
// A wave then loads 0.5 or 1 KB in one piece, where the rows of the packed weights lie KH * KW * PC words apart (32 cache
// lines an instruction, which bound every tile of less than 128 rows a wave: N=256 28x28x512->512 TNN, 128x64 tiles, 337 -> 252 us).
// The two planes of a word travel as the pair words of the operand (ternary_dword, level_dword in tab_conv_mfma.h), which leaves 6
// instructions of the 10 for the conv kernel.
// True for the workgroups of the job (uniform); `block` is the workgroup's number, made the one among the others.
// THREADS: of a workgroup; blockDim would add 256 bytes of hidden arguments to every quantizer, past the 120 from which a launch takes
// longer (ConvParams).
template <int THREADS>
__device__ __forceinline__ bool pack_weights(const WeightJob &job, uint32_t &block)
{
    if (block >= job.blocks) {
        block -= job.blocks;
        return false;
    }
    const int kc = (int)(job.kc_planes & 255u), planes = (int)(job.kc_planes >> 8);
    const int PC = (int)(job.pc_taps & 0xffffu), taps = (int)(job.pc_taps >> 16);
    const int pairs = patch_pairs(taps, kc), chunks = (PC + kc - 1) / kc;
    const uint32_t item = block * THREADS + threadIdx.x;
    const int lane = (int)(item & 63u), r = lane & 31, kb = lane >> 5;
    const uint32_t run = item >> 6, chunk_run = run / (uint32_t)pairs;
    const int j = (int)(run - chunk_run * (uint32_t)pairs), tile = (int)(chunk_run / (uint32_t)chunks), c = (int)chunk_run - tile * chunks;
    if (tile * 32 >= job.KN) return true;
    const int filter = tile * 32 + r;
    const int unit = 2 * j + kb, tap = kc == 4 ? unit >> 2 : (kc == 2 ? unit >> 1 : unit), word = c * kc + (unit & (kc - 1));
    const bool live = filter < job.KN && tap < taps && word < PC;
    const uint64_t *src = job.qw + (((size_t)filter * taps + tap) * PC + word) * planes;
    if (planes == 2) {
        uint64_t sign = 0, nz = 0;  // or the weight-2 and the weight-1 bits
        if (live) { sign = src[0]; nz = src[1]; }
        uint64_t out[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t hi = (uint32_t)(sign >> 32 * h), lo = (uint32_t)(nz >> 32 * h);
            const uint32_t even = ((lo ^ (hi << 1)) & 0x55555555u) ^ (hi << 1), odd = ((hi ^ (lo >> 1)) & 0xAAAAAAAAu) ^ (lo >> 1);
            out[h] = (uint64_t)even | (uint64_t)odd << 32;
        }
        job.out[2 * (size_t)item] = out[0];
        job.out[2 * (size_t)item + 1] = out[1];
    } else {
        job.out[item] = live ? src[0] : 0;
    }
    return true;
}

}  // namespace
}  // namespace tab
