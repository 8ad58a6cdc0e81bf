// Geometry of the convolution that keeps its input patch in LDS (tab_conv_mfma_patch.h), as the host counts it: what fits, and
// in how many chunks.
#pragma once
#include "tab_common.h"
#include "tab_patch_weights.h"

namespace tab {

template <int KC> constexpr int kPatchItems = KC == 4 ? 2 : 3;  // pixels of the patch a thread fetches at most, KC words of each
constexpr int kPatchLdsBytes = 64 * 1024;                       // of a workgroup
constexpr int kCuLdsBytes = 160 * 1024;
constexpr int kPatchThreads = 256;

// Bit planes of the weights.
inline int patch_weight_planes(int type) { return type == 0 || type == 2 || type == 4 ? 2 : 1; }

// Words of a chunk at most: waves of eight MFMA tiles have no registers for four.
constexpr int patch_most_words(int tiles_per_wave) { return tiles_per_wave >= 8 ? 2 : 4; }

// Pixels of the patch of `rows` consecutive output pixels at most, wherever they begin on a multiple of `rows` (a power of two);
// kPatchPixels + 1 for any number above it.  (32-bit arithmetic: this runs in every call.)
constexpr int kPatchPixels = kPatchItems<1> * kPatchThreads;
inline int patch_pixels(const ConvArgs &a, int rows)
{
    const int64_t wide = (int64_t)(a.OW - 1) * a.s2 + a.KW;
    if (wide > kPatchPixels || a.KH > kPatchPixels || a.s1 > kPatchPixels) return kPatchPixels + 1;
    const int PW = (int)wide;
    // output lines touched: the run may begin at any multiple of gcd(rows, OW) of a line
    const int low = a.OW & -a.OW, g = low < rows ? low : rows;
    const int lines_out = (a.OW - g + rows - 1) / a.OW + 1;
    const int crossings = a.OH >= lines_out ? (lines_out > 1 ? 1 : 0) : (lines_out - 1 + a.OH - 1) / a.OH;  // from an image's last line to the next one's first
    const int across = a.KH > a.s1 ? a.KH - a.s1 : 0;
    const int lines = (lines_out - 1) * a.s1 + crossings * across + a.KH;
    return lines > kPatchPixels || lines * PW > kPatchPixels ? kPatchPixels + 1 : lines * PW;
}

// What a patch takes: words of a chunk (0: it does not fit), pixels, bytes of LDS, workgroups that a CU's LDS holds (at most 4, which is
// all that registers leave), chunks, and pairs of words multiplied (patch_pairs of every chunk).
struct PatchFit { int kc, npix, lds_bytes, by_lds, chunks, pairs; };

// The patch of `rows` output pixels in the most words a chunk, up to `most`, that fit.
inline PatchFit patch_fit(const ConvArgs &a, int rows, int most)
{
    const int pixels = patch_pixels(a, rows);
    if (pixels > kPatchPixels || (int64_t)(a.OH - 1) * a.s1 + a.KH + pixels >= 65536) return PatchFit{};
    for (int kc = a.PC == 1 ? 1 : most; kc >= 1; kc >>= 1) {
        // of four words at most one is padding, and of three words none
        if ((kc == 4 && a.PC % 4 != 0 && a.PC % 4 != 3) || (kc == 2 && a.PC == 3)) continue;
        const int planes = pixels + (kc == 1 ? 1 : 0);
        const int bytes = planes * 32 * kc * (a.PC > kc ? 2 : 1);
        if (bytes > kPatchLdsBytes || (kc == 4 && pixels > kPatchItems<4> * kPatchThreads)) continue;
        const int lds_bytes = bytes < 4096 ? 4096 : bytes;
        const int chunks = kc == 4 ? (a.PC + 3) >> 2 : kc == 2 ? (a.PC + 1) >> 1 : a.PC;
        return PatchFit{kc, planes, lds_bytes, 2 + (lds_bytes * 3 <= kCuLdsBytes) + (lds_bytes * 4 <= kCuLdsBytes), chunks, chunks * patch_pairs(a.KH * a.KW, kc)};
    }
    return PatchFit{};
}

// The kernel's shapes: rows and filters of a workgroup's tile, MFMA tiles of a wave, workgroups a CU holds by their registers.
// What bounds the loop of a wide launch is the operands' way out of LDS, TM reads of 1 KB for TM * TN multiplications of a wave, and the
// patch, which each tile of the filters fetches and expands again: 64 rows x 256 filters, waves of 2 x 2 MFMA tiles, read half as much per
// multiplication as 128 x 128 with waves of 4 x 1 and a patch once for 256 filters (N=32 56x56x256->256 TNN 36.6 -> 33.1 us, conv kernel
// alone; N=256 14x14x256->512 stride 2 16.2 -> 13.7).  64 x 128 tiles, waves of 2 x 1, leave launches of few tiles a better last round than
// 128 x 64 (N=64 56x56x64->128 stride 2 8.9 -> 8.4).  128 x 128 with waves of 2 x 2 and 128 x 256 won nowhere by more than 3 %.
struct PatchTile { int rows, filters, wave_tiles, held; };
constexpr int kPatchShapes = 7;
constexpr PatchTile kPatchTile[kPatchShapes] = {{256, 128, 8, 2}, {128, 128, 4, 3}, {128, 64, 2, 4}, {64, 64, 1, 4}, {256, 64, 4, 3}, {64, 256, 4, 3}, {64, 128, 2, 4}};

// The first shape with the same patch.
struct PatchTwins { int of[kPatchShapes]; };
constexpr PatchTwins patch_twins()
{
    PatchTwins t = {};
    for (int i = 0; i < kPatchShapes; i++)
        for (int j = i; j >= 0; j--)
            if (kPatchTile[j].rows == kPatchTile[i].rows && patch_most_words(kPatchTile[j].wave_tiles) == patch_most_words(kPatchTile[i].wave_tiles)) t.of[i] = j;
    return t;
}
constexpr PatchTwins kPatchTwins = patch_twins();

// What the predicted durations (tab_conv_patch_model.h) are linear in; the fit script states the same.
constexpr int kPatchFeatures = 26, kTiledFeatures = 32;
constexpr int kPatchColumns = 8;  // kPatchShapes and a spare one: two vectors of four

// A call through shape i: the busiest CU holds n tiles in so many rounds, the mean one its load of them; its loop, its patches, its chunks and its output, the
// activation read by every tile of filters, the weights by every tile of rows.  Then what the
// convolution replayed on the same operands does not show: laying out the weights, and fetching them where they are in no L2 yet, pair
// after pair of words (N=64 7x7x512->512 TNN, 36 pairs: 11.0 us replayed, 15.1 behind its quantizer).  One word a pixel leaves little
// but output; and rows of Y that end inside a cache line are written in parts until they go through the caches.
// What the shapes share is worked out once, and four shapes' sums at a time: calls of two short launches wait for the host (N=16 28x28x128
// TNN 8.5 us of it a call), so the rule's time is theirs (with the tiled kernels' ranking 340 -> 210 ns, shapes one after the other before).
struct PatchCall {
    uint32_t M, KN, cus;
    float y_mb, ragged, one, one_y_mb, ragged_uncached, beyond, ragged_beyond;
    float weights_mb;  // of a pair of words
    float x_mb;        // the packed activation
};
inline float y_beyond_mb(float y_mb) { return y_mb > 256.f ? y_mb - 256.f : 0.f; }
inline PatchCall patch_call(const ConvArgs &a, int type, uint32_t cus)
{
    const float y_mb = (float)a.M * (float)a.KN * 4e-6f, ragged = a.KN % 32 ? y_mb : 0.f, beyond = y_beyond_mb(y_mb);
    return PatchCall{(uint32_t)a.M, (uint32_t)a.KN, cus, y_mb, ragged, a.PC == 1 ? 1.f : 0.f, a.PC == 1 ? y_mb : 0.f,
                     ragged_rows_cached(a.M, a.KN) ? 0.f : ragged, beyond, a.KN % 32 ? beyond : 0.f, (float)((a.KN + 31) / 32) * (patch_weight_planes(type) == 2 ? 1024e-6f : 512e-6f),
                     (float)((long)a.N * a.H * a.W) * (float)a.PC * (type == 0 || type == 1 || type == 4 ? 16e-6f : 8e-6f)};
}
// The durations in the shapes whose patch fits (kc > 0); infinity in the others.  Column by column: the sums of all shapes go on at once.
inline void patch_durations(const PatchCall &c, const PatchFit (&fits)[kPatchShapes], const float (&cost)[kPatchFeatures][kPatchColumns],
                            float (&us)[kPatchColumns])
{
    float n[kPatchColumns], rounds[kPatchColumns], all[kPatchColumns], chunks[kPatchColumns], pairs[kPatchColumns], words[kPatchColumns], down[kPatchColumns], across[kPatchColumns];
    n[kPatchShapes] = rounds[kPatchShapes] = all[kPatchShapes] = chunks[kPatchShapes] = pairs[kPatchShapes] = words[kPatchShapes] = down[kPatchShapes] = across[kPatchShapes] = 0.f;
    us[kPatchShapes] = 0.f;
#pragma unroll
    for (int i = 0; i < kPatchShapes; i++) {
        const PatchTile &tile = kPatchTile[i];
        const PatchFit &fit = fits[i];
        // M is below 2^31 and a filter's row of Y below 16 MB: fewer than 2^41 tiles
        const uint32_t row_tiles = (c.M + (uint32_t)tile.rows - 1) / (uint32_t)tile.rows, filter_tiles = (c.KN + (uint32_t)tile.filters - 1) / (uint32_t)tile.filters;
        const uint64_t tiles = (uint64_t)row_tiles * filter_tiles;
        down[i] = (float)row_tiles;
        across[i] = (float)filter_tiles;
        const uint64_t busiest = tiles < 1u << 31 ? ((uint32_t)tiles + c.cus - 1) / c.cus : (tiles + c.cus - 1) / c.cus;
        const int held = tile.held < fit.by_lds ? tile.held : fit.by_lds;
        n[i] = (float)busiest;
        rounds[i] = (float)(held == 3 ? (busiest + 2) / 3 : (busiest + (uint64_t)held - 1) >> (held >> 1));
        all[i] = (float)tiles;
        chunks[i] = (float)fit.chunks;
        pairs[i] = (float)fit.pairs;
        words[i] = (float)(fit.npix * fit.kc);
        us[i] = fit.kc ? 0.f : INFINITY;
    }
    using Four = float __attribute__((ext_vector_type(4)));
    for (int i = 0; i < kPatchColumns; i += 4) {
        auto four = [i](const float *p) { return Four{p[i], p[i + 1], p[i + 2], p[i + 3]}; };
        const Four vn = four(n), vrounds = four(rounds), vchunks = four(chunks), vpairs = four(pairs);
        const Four load = four(all) * (1.f / (float)c.cus), busy = __builtin_elementwise_min(load, Four{1.f, 1.f, 1.f, 1.f});
        const Four K = 2.f * vpairs, patch = four(words) * vchunks * 1e-3f;  // words multiplied; words expanded a tile
        auto of = [&](int k) { return four(cost[k]); };
        const Four sum = (of(0) + of(1) * busy + of(2) * (K * vn) + of(3) * (K * vrounds) + of(4) * vn + of(5) * vrounds) +
                         (of(6) * c.y_mb + of(7) * (c.y_mb * busy) + of(8) * (patch * vn) + of(9) * (patch * vrounds) + of(10) * (vchunks * vrounds) + of(11) * load) +
                         (of(12) * c.ragged + of(13) * (c.weights_mb * vpairs) + of(14) * (0.01f * vpairs) + of(15) * c.one + of(16) * c.one_y_mb +
                          of(17) * c.ragged_uncached) +
                         (of(18) * c.beyond + of(19) * c.ragged_beyond + of(20) * (c.weights_mb * vpairs / __builtin_elementwise_max(load, Four{1.f, 1.f, 1.f, 1.f}))) +
                         (of(21) * (K * load) + of(22) * (patch * load) + of(23) * (vchunks * load) + of(24) * (c.x_mb * four(across)) +
                          of(25) * (0.01f * c.weights_mb * vpairs * four(down)));
        for (int j = 0; j < 4; j++) us[i + j] += sum[j];
    }
}

// The call through the tiled kernel, of the shape that conv_mfma_shape picks, which predicts `us` for its convolution: that prediction was fitted to
// even words per pixel, whole lines of Y and launches like the benchmark's.  Each shape has its own measure of it; chunks of K are single pairs of
// words where a pixel's words are no multiple of four and K none of six (launch_mfma_shape), which long K feels (N=22 24x18x128->128 5x5 BTN
// tiled 15.5 us, patch 10.1).
constexpr int kTiledShapes[] = {0, 1, 2, 4, 5, 6, 8, 9, 10, 11};
inline void tiled_features(const ConvArgs &a, int type, int shape, float us, float (&f)[kTiledFeatures])
{
    const float G = (float)a.G, y_mb = (float)a.M * (float)a.KN * 4e-6f, beyond = y_beyond_mb(y_mb);
    const float products = (float)a.M * (float)((a.KN + 63) / 64 * 64) * G * 1e-9f;
    const bool odd = a.PC % 2 != 0, one = a.PC == 1, pairs = a.PC % 2 == 0 && a.PC % 4 != 0 && a.G % 6 != 0;
    const float ragged = a.KN % 32 ? y_mb : 0.f, ragged_beyond = a.KN % 32 ? beyond : 0.f;
    const bool cached = a.M * (long)a.KN >= (6L << 20);  // (ragged_rows_cached of 33 filters and more)
    const float uncached = cached ? 0.f : ragged;
    const float values[22] = {1.f, us, y_mb, products, odd ? products : 0.f, odd ? us : 0.f, 0.1f * G, odd ? 0.1f * G : 0.f,
                              (float)a.M * G * 1e-6f, ragged, (float)a.KN * G * (float)patch_weight_planes(type) * 8e-6f,
                              one ? 1.f : 0.f, one ? us : 0.f, one && cached ? ragged : 0.f, pairs ? us : 0.f, pairs ? 0.1f * G : 0.f,
                              beyond, ragged_beyond, one ? beyond : 0.f, one ? ragged_beyond : 0.f, uncached, uncached > 12.f && shape != 2 ? uncached - 12.f : 0.f};
    for (int k = 0; k < 22; k++) f[k] = values[k];
    for (int k = 22; k < kTiledFeatures; k++) f[k] = kTiledShapes[k - 22] == shape ? us : 0.f;
}

}  // namespace tab
