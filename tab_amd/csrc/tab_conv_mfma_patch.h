// Matrix-core conv kernel that keeps the input patch of a tile in LDS as ready FP4 operands.
//
// The im2row kernels read every input pixel once per filter tap and expand it to FP4 once per tap and wave: KH * KW times the
// loads and the vector work that the pixel needs.  Here the workgroup loads the pixels its output rows touch once, expands them
// once and leaves them in LDS in the layout the MFMA reads; a tap is then an LDS offset, an operand of the activation one
// ds_read_b128 and no vector instruction, and only the weights are expanded beside the MFMAs, straight from registers.  What an
// MFMA of a 4x2 wave costs in vector instructions in the loop falls from 5.3 (binary) - 7.5 (ternary) to 2.9 - 3.0, and instead of a
// barrier every four words of K there is one per chunk of the patch.  (Over a whole launch, patches and epilogues included: 4.1 in
// N=256 28x28x512->512 BNN, 8.8 in 2x2 waves of N=32 56x56x256->256 TNN.)
//
// The patch: the padded input of an image has PH = (OH-1)*s1 + KH lines of PW = (OW-1)*s2 + KW pixels; the lines of all images
// one after the other make one run of lines, of which the tile's BM consecutive output pixels touch a contiguous piece.  Output
// pixel (n, oh, ow) begins at pixel ((n*PH + oh*s1 - L0) * PW + ow*s2) of it, whatever the stride and however many images the
// tile spans, and tap (kh, kw) is kh*PW + kw pixels further on.
//
// Chunks: KC words of every pixel, 4, 2 or 1, the largest that fits LDS; more than one chunk takes two buffers, the next chunk's
// words on their way in registers during a chunk (words past the last one are zeros, which the BNN bias counts).
//
// LDS: a plane per (word of the chunk, half of the word), 16 bytes a pixel: 32 channels as one FP4 operand of a lane.
// Consecutive rows of a tile read consecutive 16-byte granules: no bank conflicts at stride 1.
//
// Order of k: tap by tap; the half-waves take alternate words, of a tap (KC = 2, 4) or of two neighbouring taps (KC = 1), and a step of
// the MFMA multiplies the low, the next one the high halves.  An odd number of taps leaves the upper half-wave without one at the end
// (KC = 1): it reads a pixel of FP4 zeros, the last of either plane.
#pragma once
#include "tab_conv_mfma.h"
#include "tab_conv_patch.h"
#include "tab_patch_weights.h"

namespace tab {
namespace {

template <int PL>
__device__ __forceinline__ Item<PL> load_item_at(__amdgpu_buffer_rsrc_t rsrc, uint32_t offset, uint32_t scalar_offset)
{
    Item<PL> it;
    if (PL == 2) {
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, offset, scalar_offset, 0);
        it.d[0] = v[0]; it.d[1] = v[1]; it.d[2] = v[2]; it.d[3] = v[3];
    } else {
        const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rsrc, offset, scalar_offset, 0);
        it.d[0] = v[0]; it.d[1] = v[1];
    }
    return it;
}

// Workgroups of the first round, four a CU of 256; those behind them find the weights in the L2.  On a part of the chip with fewer CUs more than the
// first round ask for lines, which are then at hand: a hint, on which no result depends.
constexpr uint32_t kFirstWorkgroups = 1024;

// ConvParams with other contents where this kernel has no use for the usual ones: G = pixels of the patch (the stride between
// planes), nchunks = KH, the magics of PC and KW = those of PW and PH.
template <int TYPE, int WM, int WN, int TM, int TN, int KC>
__global__ __launch_bounds__(kConvThreads) __attribute__((amdgpu_waves_per_eu(TM * TN >= 8 ? 2 : (TM * TN >= 4 ? 3 : 4))))
void conv_mfma_patch(const ConvParams k)
{
    static_assert(WM * WN * 64 == kConvThreads, "four waves");
    constexpr int APL = Planes<TYPE>::A, BPL = Planes<TYPE>::B;
    constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN;
    constexpr int NM = TM * TN;
    ConvArgs p = unpack_conv<TYPE, false, BM, BN>(k);
    const int npix = p.G, KH = p.nchunks;
    const int taps = KH * p.KW;
    const int PW = (p.OW - 1) * p.s2 + p.KW, PH = (p.OH - 1) * p.s1 + KH;
    const FastDiv div_pw = {p.div_pc.magic, (uint32_t)PW}, div_ph = {p.div_kw.magic, (uint32_t)PH};
    const int nchunks = (p.PC + KC - 1) / KC;
    p.G = taps * KC * nchunks;  // words of K multiplied
    const uint32_t plane = (uint32_t)npix * 16u;              // bytes between planes
    const uint32_t buffer = (uint32_t)(2 * KC) * plane;       // bytes between the two chunk buffers
    const uint32_t zero_pixel = (uint32_t)(npix - 1) * 16u;   // KC = 1: npix counts one pixel of zeros, the last

    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    char *const base = reinterpret_cast<char *>(lds);

    int tile_m, tile_n;
    if (!tile_of_workgroup(p, tile_m, tile_n)) return;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int r = lane & 31, kb = lane >> 5;
    const int wm = wave % WM, wn = wave / WM;
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int pixels = p.OH * p.OW;
    const ExpandConsts consts;

    // ---- the patch: the lines from the first output row's first tap to the last one's last ----
    const int n_first = (int)div32((uint32_t)m0, p.div_pixels);  // uniform
    const int oh_first = (int)div32((uint32_t)(m0 - n_first * pixels), p.div_ow);
    const int line0 = oh_first * p.s1;  // counted from image n_first's first padded line, as every line below
    const int m_last = m0 + BM <= p.M ? m0 + BM - 1 : p.M - 1;
    const int n_last = (int)div32((uint32_t)m_last, p.div_pixels);
    const int line_end = (n_last - n_first) * PH + (int)div32((uint32_t)(m_last - n_last * pixels), p.div_ow) * p.s1 + KH;
    const int live_pixels = (line_end - line0) * PW;
    const size_t image_words = (size_t)p.H * p.W * p.PC * APL;
    const size_t a_bytes = (size_t)(p.N - n_first) * image_words * 8;
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(p.qx + (size_t)n_first * image_words), 0,
        a_bytes > 0xffffffffull ? (int)0xffffffffu : (int)a_bytes, kBufferFlags);
    constexpr int ITEMS = kPatchItems<KC>;
    uint32_t item_off[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
        const int pix = tid + i * kConvThreads;
        const int line = (int)fastdiv((uint32_t)pix, div_pw), col = pix - line * PW;
        const int l = line0 + line;
        const int n = (int)fastdiv((uint32_t)l, div_ph);
        const int ih = l - n * PH - p.p1, iw = col - p.p2;
        const bool ok = pix < live_pixels && n_first + n < p.N && (unsigned)ih < (unsigned)p.H && (unsigned)iw < (unsigned)p.W;
        item_off[i] = ok ? (uint32_t)(((n * p.H + ih) * p.W + iw) * p.PC) * (uint32_t)(APL * 8) : kNoData;
    }
    // one chunk of every pixel of this thread, as loaded
    struct Words { uint32_t d[ITEMS][KC][2 * APL]; };
    auto load_patch = [&](Words &w, int chunk) {
        const uint32_t soff = (uint32_t)chunk * (uint32_t)(KC * APL * 8);
        const int there = p.PC - chunk * KC;  // words
        auto each = [&]() {
#pragma unroll
            for (int i = 0; i < ITEMS; i++)
#pragma unroll
                for (int c = 0; c < KC; c++) {
                    const Item<APL> it = load_item_at<APL>(a_rsrc, c < there ? item_off[i] : kNoData, soff + (uint32_t)(c * APL * 8));
#pragma unroll
                    for (int q = 0; q < 2 * APL; q++) w.d[i][c][q] = it.d[q];
                }
        };
        if constexpr (APL == 1 && KC > 1) {
            if (p.PC & 1) {
                each();
            } else {  // two words at once
#pragma unroll
                for (int i = 0; i < ITEMS; i++)
#pragma unroll
                    for (int c = 0; c < KC; c += 2) {
                        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, c < there ? item_off[i] : kNoData, soff + (uint32_t)(c * 8), 0);
                        w.d[i][c][0] = v[0]; w.d[i][c][1] = v[1]; w.d[i][c + 1][0] = v[2]; w.d[i][c + 1][1] = v[3];
                    }
            }
        } else {
            each();
        }
    };
    auto write_patch = [&](const Words &w, uint32_t buf) {
#pragma unroll
        for (int i = 0; i < ITEMS; i++) {
            const int pix = tid + i * kConvThreads;
            if (pix < live_pixels) {
                char *dst = base + buf + (uint32_t)pix * 16u;
#pragma unroll
                for (int c = 0; c < KC; c++)
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        const i32x8 e = expand_operand<TYPE, 0>(w.d[i][c][h], w.d[i][c][2 * (APL - 1) + h], consts);
                        *reinterpret_cast<u32x4 *>(dst + (uint32_t)(2 * c + h) * plane) =
                            u32x4{(uint32_t)e[0], (uint32_t)e[1], (uint32_t)e[2], (uint32_t)e[3]};
                    }
            }
        }
    };

    // ---- operands of the MFMAs ----
    uint32_t a_base[TM];  // byte offset of the lane's pixel of row tile mt in a plane
#pragma unroll
    for (int mt = 0; mt < TM; mt++) {
        const int m = m0 + wm * (32 * TM) + mt * 32 + r;
        const int mm = m < p.M ? m : m0;
        const int n = (int)div32((uint32_t)mm, p.div_pixels);
        const int rem = mm - n * pixels;
        const int oh = (int)div32((uint32_t)rem, p.div_ow), ow = rem - oh * p.OW;
        a_base[mt] = (uint32_t)(((n - n_first) * PH + oh * p.s1 - line0) * PW + ow * p.s2) * 16u;
        if (KC > 1) a_base[mt] += (uint32_t)kb * 2u * plane;  // the lane's word of a pair
    }
    // The weights as pack_patch_weights lays them out: per 32 filters, chunk and pair of words one run of 64 lanes.
    constexpr uint32_t PAIR_BYTES = 64 * 8 * BPL;
    const int pairs = patch_pairs(taps, KC);  // of a chunk
    const uint32_t tile_bytes = (uint32_t)(nchunks * pairs) * PAIR_BYTES;
    const int filter_tiles = (p.KN + 31) / 32;
    const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(reinterpret_cast<const char *>(p.qw) + (size_t)(n0 / 32) * tile_bytes), 0,
        (int)((uint32_t)(filter_tiles - n0 / 32 < WN * TN ? filter_tiles - n0 / 32 : WN * TN) * tile_bytes), kBufferFlags);
    uint32_t b_base[TN];
#pragma unroll
    for (int nt = 0; nt < TN; nt++) b_base[nt] = (uint32_t)(wn * TN + nt) * tile_bytes + (uint32_t)lane * (uint32_t)(8 * BPL);  // (past the last tile: zeros)
    struct BWords { uint32_t d[TN][2 * BPL]; };
    uint32_t b_at = 0;  // of the pair to fetch
    auto fetch_b = [&](BWords &b) {
#pragma unroll
        for (int nt = 0; nt < TN; nt++) {
            const Item<BPL> it = load_item_at<BPL>(b_rsrc, b_base[nt], b_at);
#pragma unroll
            for (int e = 0; e < 2 * BPL; e++) b.d[nt][e] = it.d[e];
        }
        b_at = b_at + PAIR_BYTES < tile_bytes ? b_at + PAIR_BYTES : b_at;  // (past the last pair: words nobody multiplies)
    };

    f32x16 acc[TM][TN];
    int b_nonzero[TN];
#pragma unroll
    for (int nt = 0; nt < TN; nt++) b_nonzero[nt] = 0;
#pragma unroll
    for (int mt = 0; mt < TM; mt++)
#pragma unroll
        for (int nt = 0; nt < TN; nt++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[mt][nt][e] = 0.f;
    i32x8 af[2][TM], bf[2][TN];
#pragma unroll
    for (int set = 0; set < 2; set++) {
#pragma unroll
        for (int mt = 0; mt < TM; mt++) af[set][mt] = i32x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int nt = 0; nt < TN; nt++) bf[set][nt] = i32x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
    // dword q % 4 of filter tile q / 4's operand, half h of the lane's word
    auto expand_piece = [&](const BWords &b, int q, int h, int set) {
        const int nt = q / 4, d = q % 4;
        if constexpr (BPL == 2) {
            const uint32_t pw = b.d[nt][2 * h + (d & 1)];
            if (TYPE == 4) bf[set][nt][d] = (int)((d < 2 ? pw : pw >> 2) & ~consts.pair);
            else bf[set][nt][d] = (int)((d < 2 ? pw << 2 : pw) & consts.pair);
            if (TYPE == 2 && d < 2) b_nonzero[nt] += __builtin_popcount(pw & consts.even);
        } else if constexpr (TYPE == 1) {
            bf[set][nt][d] = half_binary_dword(b.d[nt][h], d, consts);
        } else {
            bf[set][nt][d] = expand_operand<TYPE, 1>(b.d[nt][h], b.d[nt][h], consts)[d];
        }
    };
    uint32_t a_at[TM];  // byte offset of the lane's operand of row tile mt, low half, for the pair at hand
    auto read_a = [&](int h, int set) {
#pragma unroll
        for (int mt = 0; mt < TM; mt++) {
            const u32x4 v = *reinterpret_cast<const u32x4 *>(base + a_at[mt] + (h ? plane : 0u));
#pragma unroll
            for (int e = 0; e < 4; e++) af[set][mt][e] = (int)v[e];
        }
    };
    auto multiply = [&](int i, int set) {
        const int mt = i / TN, nt = i % TN;
        acc[mt][nt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(af[set][mt], bf[set][nt], acc[mt][nt], 4, 4, 0, 0, 0, 0);
    };

    // byte offset of the tap to come in a plane, and its column
    uint32_t tap_off = 0;
    int tap_kw = 0;
    const uint32_t next_line = (uint32_t)(PW - p.KW + 1) * 16u;
    auto next_tap = [&]() {
        const uint32_t off = tap_off;
        tap_kw++;
        tap_off += tap_kw == p.KW ? next_line : 16u;
        if (tap_kw == p.KW) tap_kw = 0;
        return off;
    };
    // the pair j of the chunk at `buf`
    uint32_t pair_off = 0;
    auto place_pair = [&](uint32_t buf, int j) {
        if (j == 0) { tap_off = 0; tap_kw = 0; }
        if (KC == 4 && (j & 1)) pair_off += 4u * plane;
        else pair_off = next_tap() + buf;
        if (KC > 1) {
#pragma unroll
            for (int mt = 0; mt < TM; mt++) a_at[mt] = a_base[mt] + pair_off;
        } else {  // the half-waves take a tap each; past the last one the pixel of zeros
            const bool single = 2 * j + 1 >= taps;
            const uint32_t off1 = next_tap() + buf;
#pragma unroll
            for (int mt = 0; mt < TM; mt++) a_at[mt] = kb ? (single ? buf + zero_pixel : a_base[mt] + off1) : a_base[mt] + pair_off;
        }
    };

    constexpr int PER = (4 * TN + NM - 1) / NM;  // dwords of the next operands expanded after each MFMA
    Words words;
    BWords cur, nxt, fly;
    load_patch(words, 0);
    fetch_b(cur);
    fetch_b(nxt);
    // The weights come from behind the L2 of whichever XCD wrote them, two pairs of words ahead of the MFMAs: the first workgroups of a launch
    // would wait for every pair.  While they wait for the patch, eight neighbours ask for a cache line of their filters each, an eighth of them.
    // Whole calls, us: N=64 14x14x256 levels 14.8 / 14.1 (64x128 tiles 14.6 / 13.8), N=32 20x20x192 5x5 TBN in 64x128 tiles 22.5 / 18.6, N=32
    // 14x14x512->512 20.5 / 18.0; 64 layers 3 % in 64x128 tiles, 2 in 128x64, none in 256x128.  All lines by every workgroup, or before the patch's
    // addresses, gained half of that.
    // (Waves of eight tiles have the time: N=256 28x28x512->512 BNN 225.0 without, 226.3 with.)
    const uint32_t touched = TM * TN >= 8 ? 0u : __builtin_amdgcn_raw_buffer_load_b32(
        b_rsrc, blockIdx.x < kFirstWorkgroups ? (uint32_t)(tid * 8 + (tile_m & 7)) * 128u : kNoData, 0, 0);
    if (KC == 1 && tid < 4)  // the pixel of zeros, in both planes of both buffers
        *reinterpret_cast<u32x4 *>(base + (nchunks > 1 ? (uint32_t)(tid >> 1) * buffer : 0u) + (uint32_t)(tid & 1) * plane + zero_pixel) = u32x4{0, 0, 0, 0};
    write_patch(words, 0);
    asm volatile("" ::"v"(touched));
    __syncthreads();
    place_pair(0, 0);
    read_a(0, 0);
#pragma unroll
    for (int q = 0; q < 4 * TN; q++) expand_piece(cur, q, 0, 0);
    uint32_t buf = 0, other = nchunks > 1 ? buffer : 0;
    for (int chunk = 0; chunk < nchunks; chunk++) {
        const bool more = chunk + 1 < nchunks;
        if (more) load_patch(words, chunk + 1);
        auto pair_step = [&](int j, auto last_constant) {
            constexpr bool LAST = decltype(last_constant)::value;
            fetch_b(fly);
            // the low halves, while the high halves' operands are made
            read_a(1, 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < NM; i++) {
                multiply(i, 0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = i * PER; q < (i + 1) * PER && q < 4 * TN; q++) expand_piece(cur, q, 1, 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (LAST) {
                if (more) write_patch(words, other);
                __syncthreads();  // (a barrier under the condition keeps the compiler from unrolling the steps: arrays in scratch memory)
                place_pair(more ? other : buf, 0);
            } else {
                place_pair(buf, j + 1);
            }
            read_a(0, 0);
            __builtin_amdgcn_sched_barrier(0);
            // the high halves, while the next pair's low halves are made
#pragma unroll
            for (int i = 0; i < NM; i++) {
                multiply(i, 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = i * PER; q < (i + 1) * PER && q < 4 * TN; q++) expand_piece(nxt, q, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            cur = nxt;
            nxt = fly;
        };
        for (int j = 0; j < pairs - 1; j++) pair_step(j, std::false_type());
        pair_step(pairs - 1, std::true_type());
        const uint32_t t = buf;
        buf = other;
        other = t;
    }
    if (TYPE == 2) {
        // the first operand past the last pair was counted with the others
#pragma unroll
        for (int nt = 0; nt < TN; nt++) b_nonzero[nt] -= __builtin_popcount(cur.d[nt][0] & consts.even) + __builtin_popcount(cur.d[nt][1] & consts.even);
    }
    scale_sums<TYPE>(acc);
    const int wave_m0 = m0 + wm * (32 * TM), wave_n0 = n0 + wn * (32 * TN);
    conv_mfma_epilogue<TYPE, TM, TN>(p, acc, b_nonzero, wave_m0, wave_n0, lane, p.G);
}

template <int TYPE, int WM, int WN, int TM, int TN, int KC>
hipError_t launch_patch_chunk(ConvArgs a, int npix, int lds_bytes, hipStream_t stream)
{
    constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN;
    a.tiles_m = (a.M + BM - 1) / BM;
    const long blocks = order_workgroups<Planes<TYPE>::A>(a, (a.KN + BN - 1) / BN);
    if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
    a.div_pc = make_fastdiv((uint32_t)((a.OW - 1) * a.s2 + a.KW));
    a.div_kw = make_fastdiv((uint32_t)((a.OH - 1) * a.s1 + a.KH));
    a.G = npix;
    a.nchunks = a.KH;
    conv_mfma_patch<TYPE, WM, WN, TM, TN, KC><<<dim3((unsigned)blocks), dim3(kConvThreads), lds_bytes, stream>>>(pack_conv<TYPE, false>(a));
    return hipGetLastError();
}

template <int TYPE, int WM, int WN, int TM, int TN>
hipError_t launch_patch(const ConvArgs &a, hipStream_t stream)
{
    if (a.qy != nullptr) return hipErrorInvalidValue;  // fp32 output only: packed output comes without room for the weights
    constexpr int MOST = patch_most_words(TM * TN);
    const PatchFit fit = patch_fit(a, 32 * WM * TM, MOST);
    switch (fit.kc) {
    case 4:
        if constexpr (MOST == 4) return launch_patch_chunk<TYPE, WM, WN, TM, TN, 4>(a, fit.npix, fit.lds_bytes, stream);
        return hipErrorInvalidValue;
    case 2: return launch_patch_chunk<TYPE, WM, WN, TM, TN, 2>(a, fit.npix, fit.lds_bytes, stream);
    case 1: return launch_patch_chunk<TYPE, WM, WN, TM, TN, 1>(a, fit.npix, fit.lds_bytes, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace
}  // namespace tab
