// Fused zero-pad + im2row + popcount GEMM for gfx950 (wave64), all four TAB types.
//
// Replaces PadKernel + Img2RowKernel (TAB_GEMM.cuh:73-115) and TNNGEMM/TBNGEMM/BTNGEMM/
// BNNGEMM (TAB_GEMM.cu:25-147): Y[m][kn] = f(sum over k of popcount(op(A[m][k], B[kn][k])))
// with A the im2row view of the packed activation, never materialised: padding and stride
// live in the address math, out-of-range taps read all-zero words (TAB_CPU.cpp:39,155).
//
// Work decomposition: a 256-thread workgroup owns a BM x BN tile of Y (BM = 16*TM output
// pixels, BN = 64*NG filters); thread (ty, tx) of the 16x16 grid owns rows ty*TM.. and the
// column quads g*64 + tx*4.. .  K is walked in chunks of `kcw` packed 64-bit words; each
// chunk of both operands is staged in LDS, split into 32-bit halves and stored k-major
// ([plane][q][row], q = 2*word + half) so that a thread fetches its TM rows / 4 columns of
// one k-slice with 128-bit LDS reads (A reads broadcast over the 16 tx lanes, B reads are
// 256 B contiguous per 16 lanes).  The inner loop is pure VALU: XOR/AND + v_bcnt_u32_b32
// with the count accumulated in the instruction's addend.
#include "tab_conv_patch.h"
#include "tab_conv_patch_model.h"
#include "tab_conv_shape_model.h"
#include "tab_conv_stage.h"
#include "tab_patch_weights.h"

#include <atomic>

namespace tab {
namespace {

constexpr int kThreads = kConvThreads;

// Inner-loop primitives.  Measured on MI355X (tab_amd/lib/valu_peak and register-level probes):
// a SIMD issues v_xor/v_and/v_bitop3 in 2 cycles and v_bcnt_u32_b32 in 4, but only when one
// scalar `s_nop 0` sits between the logic op and its v_bcnt (xor+bcnt back to back: 8.6 cycles
// per wave; xor, s_nop, bcnt: 6.4; a nop after the bcnt as well: 8.4 again), and only with an
// even number of waves per SIMD.  The compiler puts a nop of its own between any two asm
// statements, so each statement below covers four word pairs of one row: (logic, nop, bcnt) x 4.
// v_bcnt carries the accumulator as its addend.
#define TAB_XB(n) "v_xor_b32 %[t], %[a], %[b" #n "]\n\ts_nop 0\n\tv_bcnt_u32_b32 %[c" #n "], %[t], %[c" #n "]\n\t"
#define TAB_TB(n, m) \
    "v_bitop3_b32 %[t], %[a], %[b" #n "], %[" m "] bitop3:0x28\n\ts_nop 0\n\tv_bcnt_u32_b32 %[c" #n "], %[t], %[c" #n "]\n\t"
#define TAB_TNN(n)                                                                                            \
    "v_and_b32 %[u], %[a1], %[m" #n "]\n\ts_nop 0\n\tv_bcnt_u32_b32 %[z" #n "], %[u], %[z" #n "]\n\t"         \
    "v_bitop3_b32 %[t], %[a], %[b" #n "], %[u] bitop3:0x28\n\ts_nop 0\n\tv_bcnt_u32_b32 %[c" #n "], %[t], %[c" #n "]\n\t"

// c[j] += popcount(a ^ b[j]), j = 0..3                                        (BNN, TAB_GEMM.cu:142)
__device__ __forceinline__ void bnn_quad(int *c, uint32_t a, const uint32_t *b)
{
    uint32_t t;
    asm(TAB_XB(0) TAB_XB(1) TAB_XB(2) TAB_XB(3)
        : [c0] "+v"(c[0]), [c1] "+v"(c[1]), [c2] "+v"(c[2]), [c3] "+v"(c[3]), [t] "=&v"(t)
        : [a] "v"(a), [b0] "v"(b[0]), [b1] "v"(b[1]), [b2] "v"(b[2]), [b3] "v"(b[3]));
}
// c[j] += popcount((a ^ b[j]) & m), j = 0..3: one v_bitop3_b32 (truth table 0x28 for operands
// 0xF0, 0xCC, 0xAA) per pair                                             (TBN, TAB_GEMM.cu:81-84)
__device__ __forceinline__ void tbn_quad(int *c, uint32_t a, uint32_t m, const uint32_t *b)
{
    uint32_t t;
    asm(TAB_TB(0, "m") TAB_TB(1, "m") TAB_TB(2, "m") TAB_TB(3, "m")
        : [c0] "+v"(c[0]), [c1] "+v"(c[1]), [c2] "+v"(c[2]), [c3] "+v"(c[3]), [t] "=&v"(t)
        : [a] "v"(a), [m] "v"(m), [b0] "v"(b[0]), [b1] "v"(b[1]), [b2] "v"(b[2]), [b3] "v"(b[3]));
}
// c[j] += popcount((a ^ b[j]) & m[j]), j = 0..3                          (BTN, TAB_GEMM.cu:113-114)
__device__ __forceinline__ void btn_quad(int *c, uint32_t a, const uint32_t *b, const uint32_t *m)
{
    uint32_t t;
    asm(TAB_TB(0, "m0") TAB_TB(1, "m1") TAB_TB(2, "m2") TAB_TB(3, "m3")
        : [c0] "+v"(c[0]), [c1] "+v"(c[1]), [c2] "+v"(c[2]), [c3] "+v"(c[3]), [t] "=&v"(t)
        : [a] "v"(a), [b0] "v"(b[0]), [b1] "v"(b[1]), [b2] "v"(b[2]), [b3] "v"(b[3]), [m0] "v"(m[0]),
          [m1] "v"(m[1]), [m2] "v"(m[2]), [m3] "v"(m[3]));
}
// both = a1 & m[j]; z[j] += popcount(both); c[j] += popcount((a ^ b[j]) & both)   (TNN, TAB_GEMM.cu:48-51)
__device__ __forceinline__ void tnn_quad(int *z, int *c, uint32_t a, uint32_t a1, const uint32_t *b, const uint32_t *m)
{
    uint32_t t, u;
    asm(TAB_TNN(0) TAB_TNN(1) TAB_TNN(2) TAB_TNN(3)
        : [z0] "+v"(z[0]), [z1] "+v"(z[1]), [z2] "+v"(z[2]), [z3] "+v"(z[3]), [c0] "+v"(c[0]), [c1] "+v"(c[1]),
          [c2] "+v"(c[2]), [c3] "+v"(c[3]), [t] "=&v"(t), [u] "=&v"(u)
        : [a] "v"(a), [a1] "v"(a1), [b0] "v"(b[0]), [b1] "v"(b[1]), [b2] "v"(b[2]), [b3] "v"(b[3]), [m0] "v"(m[0]),
          [m1] "v"(m[1]), [m2] "v"(m[2]), [m3] "v"(m[3]));
}
// acc += popcount(x)
__device__ __forceinline__ void popcount_acc(int &acc, uint32_t x)
{
    asm("v_bcnt_u32_b32 %0, %1, %0" : "+v"(acc) : "v"(x));
}

// TM rows x 4*NG columns per thread; KCH = packed 64-bit words of K per chunk, at most;
// PIPE = operand fragments double-buffered in registers (costs APL*TM + BPL*4*NG VGPRs).
// 256 threads: one wave per SIMD (512-thread workgroups were measured slightly slower).
template <int TYPE, int TM, int NG, int KCH, bool PIPE>
__global__ __launch_bounds__(kThreads) void conv_popcount(const ConvParams k)
{
    constexpr int APL = Planes<TYPE>::A, BPL = Planes<TYPE>::B;
    constexpr int BM = 16 * TM, BN = 64 * NG, TN = 4 * NG;
    const ConvArgs p = unpack_conv<TYPE, false, BM, BN>(k);
    using Stager = TileStager<TYPE, BM, BN, KCH>;
    constexpr int kMaxQ = Stager::Q, A_DWORDS = Stager::A_DWORDS, B_DWORDS = Stager::B_DWORDS;
    static_assert(TM % 4 == 0 || TM == 2, "TM is read with 64- or 128-bit LDS loads");

    // + one spare k-slice of the wider operand: the pipelined loop reads one slice ahead
    __shared__ __attribute__((aligned(16))) uint32_t lds[2 * (A_DWORDS + B_DWORDS) + (BM > BN ? BM : BN)];

    const int tid = threadIdx.x;
    const int tx = tid & 15, ty = tid >> 4;
    // consecutive workgroups walk M first so neighbours share the weight tile in L2
    const int tile_n = (int)div32(blockIdx.x, p.div_tiles_m), tile_m = (int)blockIdx.x - tile_n * p.tiles_m;
    const int m0 = tile_m * BM, n0 = tile_n * BN;

    Stager st;
    st.init(p, tid, m0, n0);

    // ---- accumulators --------------------------------------------------------------------
    // acc: popcount of the "negative" word (TNN/TBN/BTN) or of a^b (BNN);
    // nzc: TNN popcount(a1 & b1) per output; TBN popcount(a1) per row (independent of kn).
    int acc[TM][TN];
    int nzc[TYPE == 0 ? TM : 1][TYPE == 0 ? TN : 1];
    int row_nz[TYPE == 1 ? TM : 1];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            acc[i][j] = 0;
            if (TYPE == 0) nzc[i][j] = 0;
        }
    if (TYPE == 1) {
#pragma unroll
        for (int i = 0; i < TM; i++) row_nz[i] = 0;
    }

    // One k-slice (32 bits of K) of this thread's operands.
    struct Frag {
        uint32_t a[APL][TM], b[BPL][TN];
    };
    auto read_frag = [&](Frag &f, const uint32_t *la, const uint32_t *lb, int q) {
#pragma unroll
        for (int pl = 0; pl < APL; pl++) {
            const uint32_t *src = la + (pl * kMaxQ + q) * BM + ty * TM;
            if (TM == 2) {
                const u32x2 v = *reinterpret_cast<const u32x2 *>(src);
                f.a[pl][0] = v[0]; f.a[pl][1] = v[1];
            } else {
#pragma unroll
                for (int i4 = 0; i4 < TM / 4; i4++) {
                    const u32x4 v = *reinterpret_cast<const u32x4 *>(src + 4 * i4);
#pragma unroll
                    for (int e = 0; e < 4; e++) f.a[pl][4 * i4 + e] = v[e];
                }
            }
        }
#pragma unroll
        for (int pl = 0; pl < BPL; pl++)
#pragma unroll
            for (int g = 0; g < NG; g++) {
                const u32x4 v = *reinterpret_cast<const u32x4 *>(lb + (pl * kMaxQ + q) * BN + g * 64 + tx * 4);
#pragma unroll
                for (int e = 0; e < 4; e++) f.b[pl][4 * g + e] = v[e];
            }
    };
    auto mac = [&](const Frag &f) {
        if (TYPE == 1) {
#pragma unroll
            for (int i = 0; i < TM; i++) popcount_acc(row_nz[i], f.a[APL - 1][i]);
        }
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j += 4) {
                if (TYPE == 0)
                    tnn_quad(&nzc[i][j], &acc[i][j], f.a[0][i], f.a[1][i], &f.b[0][j], &f.b[1][j]);
                else if (TYPE == 1)
                    tbn_quad(&acc[i][j], f.a[0][i], f.a[1][i], &f.b[0][j]);  // popcount(a1) is summed once per row above
                else if (TYPE == 2)
                    btn_quad(&acc[i][j], f.a[0][i], &f.b[0][j], &f.b[1][j]);
                else
                    bnn_quad(&acc[i][j], f.a[0][i], &f.b[0][j]);
            }
    };

    st.fetch(p, 0);
    st.stage(lds);
    __syncthreads();

    for (int chunk = 0; chunk < p.nchunks; chunk++) {
        const bool more = chunk + 1 < p.nchunks;
        if (more) st.fetch(p, chunk + 1);

        const uint32_t *la = lds + (chunk & 1) * (A_DWORDS + B_DWORDS), *lb = la + A_DWORDS;
        const int words_here = (p.G - chunk * p.kcw < p.kcw) ? p.G - chunk * p.kcw : p.kcw;
        const int nq = 2 * words_here;
        // Register double buffering: the LDS reads of k-slice q+1 are issued before the VALU
        // work of slice q, so a single wave per SIMD still keeps the VALU busy.  nq is even.
        // The read of slice nq after the last pair stays inside the LDS allocation (one spare
        // slice is reserved) and its value is never used.
        if (PIPE) {
            Frag f0, f1;
            // drain outstanding scalar loads first: they share the LDS counter and return out
            // of order, which would force full waits inside the loop
            __builtin_amdgcn_s_waitcnt(0xc07f);
            read_frag(f0, la, lb, 0);
            for (int q = 0; q < nq; q += 2) {
                read_frag(f1, la, lb, q + 1);
                __builtin_amdgcn_sched_barrier(0);
                mac(f0);
                __builtin_amdgcn_sched_barrier(0);
                read_frag(f0, la, lb, q + 2);
                __builtin_amdgcn_sched_barrier(0);
                mac(f1);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            for (int q = 0; q < nq; q++) {
                Frag f;
                read_frag(f, la, lb, q);
                mac(f);
            }
        }

        if (more) st.stage(lds + ((chunk + 1) & 1) * (A_DWORDS + B_DWORDS));
        __syncthreads();
    }

    // ---- epilogue: integer result -> fp32, Y[m*KN + kn] (TAB_GEMM.cu:53,86,116,144) --------
    const bool vec_ok = (p.KN & 3) == 0;
#pragma unroll
    for (int g = 0; g < NG; g++) {
        const int kn = n0 + g * 64 + tx * 4;
        int bias[4] = {0, 0, 0, 0};
        if (TYPE == 2) {
#pragma unroll
            for (int e = 0; e < 4; e++) bias[e] = (kn + e < p.KN) ? p.btn[kn + e] : 0;
        }
#pragma unroll
        for (int i = 0; i < TM; i++) {
            const int m = m0 + ty * TM + i;
            if (m >= p.M) continue;
            float out[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int j = 4 * g + e;
                int v;
                if (TYPE == 0) v = nzc[i][j] - 2 * acc[i][j];
                else if (TYPE == 1) v = row_nz[i] - 2 * acc[i][j];
                else if (TYPE == 2) v = bias[e] - 2 * acc[i][j];
                else v = p.num - 2 * acc[i][j];
                out[e] = (float)v;
            }
            float *dst = p.y + (size_t)m * p.KN + kn;
            if (vec_ok && kn + 3 < p.KN) {
                *reinterpret_cast<f32x4 *>(dst) = f32x4{out[0], out[1], out[2], out[3]};
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (kn + e < p.KN) dst[e] = out[e];
            }
        }
    }
}

// Extra (unused) dynamic LDS per workgroup that makes the number of resident workgroups per
// CU - one wave per SIMD each - even: the VALU pairing above only pays off with an even number
// of waves per SIMD (2 or 4; 3 measured as slow as no pairing at all).
struct Occupancy {
    int dyn_lds;        // bytes of padding LDS per workgroup
    int blocks_per_cu;  // resident workgroups per CU with that padding (0 = unknown)
};

template <typename Kernel>
Occupancy even_occupancy(Kernel kernel)
{
    for (int dyn = 0; dyn <= 48 * 1024; dyn += 2048) {
        int blocks = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kernel, kThreads, dyn) != hipSuccess) {
            (void)hipGetLastError();
            return {0, 0};
        }
        if (blocks <= 2 || (blocks & 1) == 0) return {dyn, blocks};
    }
    return {0, 0};
}

template <int TYPE, int TM, int NG, int KCH, bool PIPE = true>
hipError_t launch_tile(ConvArgs a, hipStream_t stream)
{
    constexpr int BM = 16 * TM, BN = 64 * NG;
    static const Occupancy occ = even_occupancy(conv_popcount<TYPE, TM, NG, KCH, PIPE>);
    // chunk length: at most KCH words, chunks of equal length
    a.nchunks = (a.G + KCH - 1) / KCH;
    a.kcw = (a.G + a.nchunks - 1) / a.nchunks;
    a.nchunks = (a.G + a.kcw - 1) / a.kcw;
    a.tiles_m = (a.M + BM - 1) / BM;
    a.div_tiles_m = make_div32((uint32_t)a.tiles_m);
    const long tiles_n = (a.KN + BN - 1) / BN;
    const long blocks = (long)a.tiles_m * tiles_n;
    if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
    conv_popcount<TYPE, TM, NG, KCH, PIPE><<<dim3((unsigned)blocks), dim3(kThreads), occ.dyn_lds, stream>>>(pack_conv<TYPE, false>(a));
    return hipGetLastError();
}

// Kernel choice of tab_set_conv_kernel, (tm << 8) | (ng + 1) in one atomic word so that a launch on another
// thread sees either the old or the new pair, never a mix; 0 = the automatic choice.
std::atomic<int> g_forced_kernel{0};
struct Forced { int tm, ng; };
inline Forced forced_kernel()
{
    const int v = g_forced_kernel.load(std::memory_order_relaxed);
    return {v >> 8, (v & 0xff) - 1};
}

// Tile shapes.  Every shape keeps <= 128 VGPRs, i.e. at least 4 workgroups (4 waves per SIMD)
// per CU; shapes with 128 accumulators at 2 waves per SIMD and 512-thread workgroups were
// measured 10-25 % slower.  Three shapes are used:
//   big    128x128 (128x64 for TNN, which keeps two counts per output), chunks of 4 words;
//          fragments register double-buffered only where that still fits 128 VGPRs (BNN)
//   medium 64x64, chunks of 4 words, double-buffered fragments, 8 workgroups per CU
//   small  32x64, chunks of 8 words
// Measured over the ResNet-18 / sweep shapes at N = 32..256: the medium tile wins everywhere
// except on the very largest launches (>= 3 rounds of big tiles over the whole chip), and the
// small tile wins once even medium tiles give the CUs fewer than two workgroups each.
template <int TYPE>
hipError_t launch_big(const ConvArgs &a, hipStream_t stream)
{
    if constexpr (TYPE == 0)
        return launch_tile<TYPE, 8, 1, 4, false>(a, stream);
    else if constexpr (TYPE == 3)
        return launch_tile<TYPE, 8, 2, 4, true>(a, stream);
    else
        return launch_tile<TYPE, 8, 2, 4, false>(a, stream);
}

template <int TYPE>
hipError_t launch_type(const ConvArgs &a, hipStream_t stream)
{
    constexpr int BIG_BN = (TYPE == 0) ? 64 : 128;
    const int force_tm = forced_kernel().tm;
    if (force_tm == 8) return launch_big<TYPE>(a, stream);
    if (force_tm == 4) return launch_tile<TYPE, 4, 1, 4, true>(a, stream);
    if (force_tm == 2) return launch_tile<TYPE, 2, 1, 8, true>(a, stream);
    auto tiles = [&](int bm, int bn) { return (long)((a.M + bm - 1) / bm) * ((a.KN + bn - 1) / bn); };
    if (a.KN > BIG_BN / 2 && tiles(128, BIG_BN) >= 3072) return launch_big<TYPE>(a, stream);
    if (tiles(64, 64) >= 512) return launch_tile<TYPE, 4, 1, 4, true>(a, stream);
    return launch_tile<TYPE, 2, 1, 8, true>(a, stream);
}

}  // namespace

void force_conv_tile(int tm, int ng)
{
    g_forced_kernel.store(tm == 0 ? 0 : ((tm << 8) | ((ng + 1) & 0xff)), std::memory_order_relaxed);
}

std::atomic<int> g_compute_units{0};
void set_compute_units(int units) { g_compute_units.store(units > 0 ? units : 0, std::memory_order_relaxed); }

int device_compute_units()
{
    const int forced = g_compute_units.load(std::memory_order_relaxed);
    if (forced > 0) return forced;
    static std::atomic<int> cached{0};
    int cus = cached.load(std::memory_order_relaxed);
    if (cus == 0) {
        int device = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&device) == hipSuccess && hipGetDeviceProperties(&prop, device) == hipSuccess && prop.multiProcessorCount > 0) {
            cus = prop.multiProcessorCount;
        } else {
            (void)hipGetLastError();
            cus = 256;
        }
        cached.store(cus, std::memory_order_relaxed);
    }
    return cus;
}

std::atomic<int> g_tail_round{0};
void set_tail_round(int workgroups) { g_tail_round.store(workgroups > 0 ? workgroups : 0, std::memory_order_relaxed); }
int tail_round()
{
    const int forced = g_tail_round.load(std::memory_order_relaxed);
    return forced > 0 ? forced : device_compute_units();
}

bool conv_kernel_forced() { return g_forced_kernel.load(std::memory_order_relaxed) != 0; }

// fp32 accumulators hold integers up to 2^24 exactly; a product is at most 1 (9 for the 2-bit levels of
// type 4, see conv_mfma_exact_levels) and there are 64 per word
bool conv_mfma_exact(const ConvArgs &a) { return (long)a.G * 64 <= (1L << 22); }
bool conv_mfma_exact_levels(const ConvArgs &a) { return (long)a.G * 64 * 9 < (1L << 24); }

hipError_t launch_conv_mfma(int type, const ConvArgs &args, int shape, hipStream_t stream)
{
    if (!conv_mfma_exact(args)) return hipErrorInvalidValue;
    switch (type) {
    case 0: return launch_conv_mfma_tnn(args, shape, stream);
    case 1: return launch_conv_mfma_tbn(args, shape, stream);
    case 2: return launch_conv_mfma_btn(args, shape, stream);
    case 3: return launch_conv_mfma_bnn(args, shape, stream);
    case 4: return conv_mfma_exact_levels(args) ? launch_conv_mfma_drf(args, shape, stream) : hipErrorInvalidValue;
    case 5: return launch_conv_mfma_rtn(args, shape, stream);
    default: return hipErrorInvalidValue;
    }
}

// Workgroup tile of the matrix-core kernel: the shape with the lowest predicted duration under a cost model fitted to
// the measured duration of every shape on 420 (type, layer) cases (tab_conv_shape_model.h: the ResNet-18 layers at
// N = 16 / 64 / 256, the VGG stack, the 28x28 sweep and layers of other geometries).  What the model's features say:
// the busiest CU decides (ceil(tiles / CUs) tiles of a shape land on it, and it is refilled when it holds no more), K
// scales the loop, the size of Y the epilogue (with a price of its own where K is at most nine words and the launch is
// little but epilogue), and a launch smaller than the chip is as long as one tile.  Features and coefficients are all
// non-negative, so a prediction is positive and monotone in K, tiles and Y for any geometry; on top of that no prediction
// is taken below what the matrix cores of the busiest CU need at their peak rate plus a launch.
// (Types 4 and 5 have coefficients of their own: with those of the types of as many planes, 0 and 3, their choices took 4.2 %
// more than the best shapes', N=256 7x7x512 of type 5 28.4 us for 22.3.)
// A shape whose filter tile is at least twice the 64-rounded filter count is no candidate.
// cost_us (optional): the predicted duration of the chosen shape.
// (Host time of every call of two launches, 8.5 us at N=16 28x28x128: the loop over a table's shapes is unrolled, so that tile counts are
// shifts, and counts are divided in 32 bits where they fit: 72-163 -> 34-87 ns.)
template <bool PACKED>
static int conv_mfma_ranked(int type, const ConvArgs &a, float *cost_us)
{
    const long kn64 = ((long)a.KN + 63) / 64 * 64;
    const uint32_t cus = (uint32_t)device_compute_units();
    const bool narrow = conv_mfma_narrow(a);
    const float y_mb = (float)a.M * (float)a.KN * 4e-6f;
    const float words = type == 5 ? 0.5f * (float)a.G : (float)a.G;  // of 64 elements
    int best = 2;
    float best_cost = 0.f;
    bool any = false;
#pragma unroll
    for (int i = 0; i < (PACKED ? kConvPackedShapes : kConvShapes); i++) {
        const int shape = PACKED ? kConvPackedIds[i] : kConvShapeIds[i];
        const int bm = PACKED ? kConvPackedTile[i][0] : kConvShapeTile[i][0], bn = PACKED ? kConvPackedTile[i][1] : kConvShapeTile[i][1];
        const int held = PACKED ? kConvPackedTile[i][2] : kConvShapeTile[i][2];
        const float *const coefficients = PACKED ? kConvPackedCost[type & 3][i] : kConvShapeCost[type][i];
        if (bn >= 2 * kn64) continue;
        if (shape == 7 && a.G > 9) continue;
        if (shape == 3 && a.qy != nullptr) continue;        // the packed epilogues need tiles 64 filters wide
        if (shape >= 8 && a.PC % 2 != 0) continue;          // the split-K shapes move whole pairs of words inside a tap
        const uint64_t tiles = (uint64_t)(((uint32_t)a.M + bm - 1) / bm) * (((uint32_t)a.KN + bn - 1) / bn);
        const uint64_t whole = tiles < 1u << 31 ? (uint32_t)tiles / cus : tiles / cus, rest = tiles - whole * cus;
        float cost = 0.f, floor_us;
        if (shape == 10 || shape == 11) {
            // the mixed launches: whole tiles on every CU, then 64x64 quarter tiles (four to a 128x128 tile, eight to a
            // 128x256 one); candidates where they have both and K words x bit planes of the two operands exceed 36 (below
            // that the launch is bound by writing Y, whatever the balance of its last round)
            const int pieces = bm / 64 * (bn / 64);
            const uint32_t quarters = (uint32_t)(pieces * (uint32_t)rest + cus - 1) / cus;
            const int planes = type == 0 || type == 4 ? 4 : (type == 3 || type == 5 ? 2 : 3);
            if (a.G * planes <= 36 || whole == 0 || quarters == 0) continue;  // (an odd number of words per pixel: excluded above)
            if (shape == 11 && a.PC % 4 != 0) continue;                       // the 128x256 tiles take four-word chunks inside a tap
            const float f[kConvShapeFeatures] = {(float)a.G * (float)whole, (float)a.G * (float)quarters, (float)quarters, (float)whole, y_mb, y_mb,
                                                 1.f, 1.f, 0.f};
            for (int k = 0; k < kConvShapeFeatures; k++) cost += coefficients[k] * f[k];
            floor_us = 1.f + (float)(4 * (uint64_t)pieces * whole + 4 * quarters) * words * (32.f / 4.f / 2400.f);
        } else {
            const uint64_t busiest = whole + (rest != 0);
            const float n = (float)busiest, rounds = (float)((busiest + (uint64_t)held - 1) / (uint64_t)held);
            const float busy = whole != 0 ? 1.f : (float)tiles / (float)cus;
            const float f[kConvShapeFeatures] = {(float)a.G * n, (float)a.G * rounds, rounds, n, y_mb, y_mb * busy, busy, 1.f,
                                                 a.G <= 9 ? y_mb : 0.f};
            for (int k = 0; k < kConvShapeFeatures; k++) cost += coefficients[k] * f[k];
            // the busiest CU's n tiles of (bm/32)(bn/32) MFMA tiles x words, 32 cycles each on four SIMDs at 2.4 GHz, and a launch
            floor_us = 1.f + n * (float)(bm / 32 * (bn / 32)) * words * (32.f / 4.f / 2400.f);
        }
        // in their forms of 32 filters: what is above a launch, by a quarter less (179 measured cases, conv_narrow_timings.txt:
        // the choices take 1.4 % more than the best shapes, at worst 18 %)
        if (narrow && (shape == 1 || shape == 8)) {
            if (cost > 3.f) cost = 3.f + 0.75f * (cost - 3.f);
            floor_us = 1.f + 0.5f * (floor_us - 1.f);
        }
        if (cost < floor_us) cost = floor_us;
        if (!any || cost < best_cost) {
            any = true;
            best = shape;
            best_cost = cost;
        }
    }
    if (cost_us) *cost_us = best_cost;
    return best;
}

int conv_mfma_shape(int type, const ConvArgs &a, float *cost_us)
{
    // Packed output has a ranking of its own: with the one of fp32 output, and the kernel with the weights in registers wherever K is at
    // most nine words and M at least 65536, 743 random layers took 6 % more than the best shapes' time; with this one 1.5 %.
    // (types 4 and 5 are ranked as with fp32 output: they were not measured)
    // Below 128 tiles of 64x64, where none of those layers lies, the ranking of fp32 output stays (one image of 41x41x192 through four
    // layers: 26.1 us with it, 26.7 with the other), and weights in registers for K of at most two words.
    if (a.qy == nullptr || type > 3) return conv_mfma_ranked<false>(type, a, cost_us);
    if ((long)((a.M + 63) / 64) * (((long)a.KN + 63) / 64) >= 128) return conv_mfma_ranked<true>(type, a, cost_us);
    if (a.G <= 2) {
        if (cost_us) *cost_us = 0.f;
        return 7;
    }
    return conv_mfma_ranked<false>(type, a, cost_us);
}

// The kernel that splits K over the waves of a workgroup (tab_conv_mfma_waves.h): its shape with the lowest predicted duration, and whether
// that is 2 % below what the tiled kernel is predicted to take and below 12 us (tab_conv_waves_model.h: linear forms with non-negative
// coefficients, fitted to the calls of 1900 random layers and of 800 of residual and other networks' sizes, those that choices slowed down by
// more than 5 % counted threefold).  32x32 tiles it takes wherever conv_mfma_shape ranks them first, in 0.74 of the time of the kernel that ranking
// was made with, in which four waves shared chunks of K in LDS.  Of the other layers, quantizer and convolution take 0.943 of the tiled kernels'
// time, the better of each 0.925; of 715 choices 11 are more than 2 % slower, the worst 4.5 % (held out of the fit by quarters 0.943, 30, 8.7 %).
// (Fitted to the random layers alone and without a price for pixels of whole cache lines, N=16 14x14x512 of type 5 came out 22 %, N=64
// 7x7x512->512 TNN 31 % slower.  Those pixels' loads read the same bytes of 32 lines, a half more time than others.)  Convolution behind its
// quantizer, tiled / this, us: N=4 7x7x512->512 BNN 4.7 / 3.1, N=16 5.8 / 4.2, N=16 14x14x256->256 TNN 6.2 / 5.4, 14x14x256->512 stride 2 BNN 4.6 / 3.4;
// N=32 56x56x64->64 7.3 / 9.3 and N=64 7x7x512->512 TNN 11.6 / 15.2 stay with the tiles.
struct WavesTile { int rows, filters, waves, held; };
constexpr int kWavesShapes = 4, kWavesFeatures = 11, kWavesTiledFeatures = 10;
constexpr WavesTile kWavesTile[kWavesShapes] = {{32, 32, 8, 4}, {32, 32, 4, 8}, {64, 32, 4, 4}, {32, 64, 4, 4}};
constexpr float kWavesLimitUs = 12.f, kWavesMargin = 0.98f;
}  // namespace tab
#include "tab_conv_waves_model.h"
namespace tab {

int conv_waves_shape(int type, const ConvArgs &a, float *cost_us)
{
    const uint32_t cus = (uint32_t)device_compute_units();
    const float G = (float)a.G, y_mb = (float)a.M * (float)a.KN * 4e-6f;
    const float weights_mb = (float)a.KN * G * (type == 0 || type == 2 || type == 4 ? 16e-6f : 8e-6f);
    const int words = a.PC % 2 == 0 && type != 0 && type != 4 ? 2 : 1;  // kWavesOneWord
    const float lines = a.PC * (type <= 1 || type == 4 ? 16 : 8) % 128 == 0 ? G : 0.f;  // a pixel is whole cache lines
    const int units = (a.G + 2 * words - 1) / (2 * words);
    int best = 0;
    float best_us = 0.f;
#pragma unroll
    for (int i = 0; i < kWavesShapes; i++) {
        const WavesTile tile = kWavesTile[i];
        const uint64_t tiles = (uint64_t)(((uint32_t)a.M + tile.rows - 1) / tile.rows) * (((uint32_t)a.KN + tile.filters - 1) / tile.filters);
        const uint64_t busiest = tiles < 1u << 31 ? ((uint32_t)tiles + cus - 1) / cus : (tiles + cus - 1) / cus;
        const float load = (float)tiles / (float)cus, n = (float)busiest, rounds = (float)((busiest + tile.held - 1) / tile.held);
        const float f[kWavesFeatures] = {1.f, (float)((units + tile.waves - 1) / tile.waves * words), load < 1.f ? load : 1.f, n, n * G, load, load * G,
                                         rounds, y_mb, weights_mb, n * lines};
        float us = 0.f;
        for (int k = 0; k < kWavesFeatures; k++) us += kWavesCost[type][i][k] * f[k];
        if (tiles * (uint64_t)(64 * tile.waves) > 0xffffffffull) us = INFINITY;  // the threads a launch may have
        if (i == 0 || us < best_us) {
            best = i;
            best_us = us;
        }
    }
    if (cost_us) *cost_us = best_us;
    return kWavesShape + best;
}

// That kernel's shape or `tiled`, which conv_mfma_shape picked at a price of `tiled_us`.
// gain_us (optional): what that kernel is predicted to take less.
static int conv_waves_or(int type, const ConvArgs &a, int tiled, float tiled_us, float *gain_us = nullptr)
{
    if (gain_us) *gain_us = 0.f;
    if (a.qy != nullptr) return tiled;
    if (tiled == 3) return conv_waves_shape(type, a, nullptr);
    if ((long)((a.M + 31) / 32) * ((a.KN + 31) / 32) > 48L * device_compute_units()) return tiled;  // (far above the limit)
    float us = 0.f;
    const int shape = conv_waves_shape(type, a, &us);
    const float G = 0.1f * (float)a.G, y_mb = (float)a.M * (float)a.KN * 4e-6f;
    const float weights_mb = (float)a.KN * (float)a.G * (type == 0 || type == 2 || type == 4 ? 16e-6f : 8e-6f);
    const bool odd = a.PC % 2 != 0, one = a.PC == 1;
    const float f[kWavesTiledFeatures] = {1.f, tiled_us, y_mb, odd ? tiled_us : 0.f, G, odd ? G : 0.f, weights_mb,
                                          a.KN % 32 ? y_mb : 0.f, one ? 1.f : 0.f, one ? tiled_us : 0.f};
    float limit = 0.f;
    for (int k = 0; k < kWavesTiledFeatures; k++) limit += kWavesTiledCost[type][k] * f[k];
    if (gain_us) *gain_us = limit - us;
    limit *= kWavesMargin;
    return us < (limit < kWavesLimitUs ? limit : kWavesLimitUs) ? shape : tiled;
}

float conv_waves_gain(int type, const ConvArgs &a)
{
    float us = 0.f, gain = 0.f;
    const int tiled = conv_mfma_shape(type, a, &us);
    return conv_waves_or(type, a, tiled, us, &gain) >= kWavesShape ? (tiled == 3 ? INFINITY : gain) : -INFINITY;
}

int conv_fp32_shape(int type, const ConvArgs &a)
{
    float us = 0.f;
    const int tiled = conv_mfma_shape(type, a, &us);
    return conv_waves_or(type, a, tiled, us);
}

// The kernel that keeps the input patch in LDS, against the tiled one that conv_mfma_shape picks: the shape with the lowest predicted
// duration, if that is 1.5 % and 0.1 us below what the call through the tiled kernel is predicted to take (tab_conv_patch_model.h; both are
// linear forms with non-negative coefficients, fitted to the whole calls of 11068 layers, among them long K on few tiles, rows of Y that end inside a cache line
// and launches of 30 to 400 us, where a fit to 3970 had gone wrong: N=24 104x104x7->348 BNN 119 us through the tiles it chose, 78 here).  Those calls take 0.944
// of the time without this kernel (in total 0.914; the better one of each 0.937 and 0.907; the earlier fit 0.949, 0.921); of 4459 choices 149 are more than 2 % slower,
// 34 more than 5 %, the worst 18 % (61 %), and 113 calls are more than 10 % above the best kernel (341).  On thirds held out of the fit 0.944, 164, 47, 18 %, 124;
// on 1500 layers measured after it 0.938 (the earlier fit 0.940, best 0.922), of 644 choices 18 more than 2 % slower, six 5 %, the worst 10 %.  (Fitted to
// convolutions replayed on the same operands, weights in the L2s, a tenth of such layers were more than 5 % slower, the worst 1.6 times.)
// Where the tiled kernel's place is the split-K kernel's (conv_waves_or), the patch is taken if it is predicted to gain as much.
// Long K on few tiles, more than 192 words for more than 256 filters or more than 448 on less than 1.4 to 2 tiles of 64x64 a CU, stays with the others: the
// weights come from behind the L2s once, and nothing hides them (N=4 54x64x888->128 7x7 TBN 73 us in tile 8, 114 here).
// Nor does more than 150 MB of Y in rows of more than 64 filters go by 64x64 tiles, which write 256 bytes of a row at a time: timed between other kernels
// they are as soon as the others, call after call they are not (N=172 30x32x64->512 BNN 69 us, 64x128 tiles 67; N=72 54x35x64->448 BTN 54.4, 128x64 45.8).
// Not for 1x1 kernels, which read every pixel for one tap only, nor for at most 32 filters, half of whose tiles would be work for nothing,
// nor for launches of fewer 64x64 tiles than compute units, which last as long as one tile's chain of waits (from half as many on, 129
// of 2709 layers gained more than 3 %, none that a fit could tell from the others).  Measured, whole calls, tiled / patch: N=64 14x14x256
// levels 16.2 / 13.2 us, N=256 28x28x512->512 BNN 247 / 223, N=32 56x56x256->256 TNN 59.6 / 52.7 (64x256 tiles).  Each shape is the
// best one of some launches.
static bool forced_patch(const Forced &forced) { return forced.tm == 9 && forced.ng >= kPatchShape && forced.ng < kWavesShape; }

bool conv_patch_considered(int type, long M, int KN, int KH, int KW)
{
    if (type > 4) return false;
    const Forced forced = forced_kernel();
    if (forced_patch(forced)) return true;  // the test hook
    return (forced.tm == 0 || (forced.tm == 9 && forced.ng < 0)) && KH * KW > 1 && KN > 32 &&
           (M + 63) / 64 * (((long)KN + 63) / 64) >= device_compute_units();
}

PatchPlan conv_patch_plan(int type, const ConvArgs &a)
{
    PatchPlan plan = {-1, 0, 0, 0, -1, 0};
    const Forced forced = forced_kernel();
    if (!conv_patch_considered(type, a.M, a.KN, a.KH, a.KW) || !conv_mfma_exact(a) || (type == 4 && !conv_mfma_exact_levels(a))) return plan;
    auto take = [&](int i, const PatchFit &fit) {
        const size_t tiles = ((size_t)a.KN + 31) / 32;
        plan = PatchPlan{kPatchShape + i, fit.kc, fit.npix, fit.lds_bytes, plan.tiled, tiles * (size_t)fit.pairs * 512 * patch_weight_planes(type)};
    };
    auto fit_of = [&](int i) { return patch_fit(a, kPatchTile[i].rows, patch_most_words(kPatchTile[i].wave_tiles)); };
    if (forced_patch(forced)) {  // the test hook
        const int i = forced.ng - kPatchShape;
        const PatchFit fit = i < kPatchShapes ? fit_of(i) : PatchFit{};
        if (fit.kc) take(i, fit);
        return plan;
    }
    if (a.qy != nullptr) return plan;
    float tiled_us = 0.f;
    plan.tiled = conv_mfma_shape(type, a, &tiled_us);
    if (plan.tiled == 3) {  // K split over waves then: of 19 such layers the patch was faster on none
        plan.tiled = conv_waves_shape(type, a, nullptr);
        return plan;
    }
    const long kn64 = ((long)a.KN + 63) / 64, cus = device_compute_units();
    float waves_gain_us = 0.f;
    const int tiled = plan.tiled;
    plan.tiled = conv_waves_or(type, a, tiled, tiled_us, &waves_gain_us);  // (also where the weights then find no room)
    if (a.G > 192 && (a.KN > 256 || a.G > 448) && ((long)a.M + 63) / 64 * kn64 * 512 < cus * (512 + a.G)) return plan;
    float t[kTiledFeatures];
    tiled_features(a, type, tiled, tiled_us, t);
    float limit = 0.f;
    for (int k = 0; k < kTiledFeatures; k++) limit += kTiledCost[type][k] * t[k];
    const float tiled_call_us = limit;
    limit = 0.985f * limit - 0.1f;
    const PatchCall call = patch_call(a, type, (uint32_t)cus);
    PatchFit fits[kPatchShapes];
    for (int i = 0; i < kPatchShapes; i++) fits[i] = kPatchTwins.of[i] < i ? fits[kPatchTwins.of[i]] : fit_of(i);
    float us[kPatchColumns];
    patch_durations(call, fits, kPatchCost[type], us);
    int best = -1;
    const bool wide = kn64 > 1 && call.y_mb > 150.f;  // (not in 64x64 tiles)
    for (int i = 0; i < kPatchShapes; i++)
        if (us[i] < limit && kPatchTile[i].filters < 128 * kn64 && !(wide && kPatchTile[i].wave_tiles == 1)) {
            limit = us[i];
            best = i;
        }
    if (best >= 0 && (plan.tiled < kWavesShape || waves_gain_us <= tiled_call_us - us[best])) take(best, fits[best]);
    return plan;
}

size_t patch_weight_bytes(int type, int C, int KN, int KH, int KW)
{
    if (type > 4 || KN <= 0) return 0;
    const size_t PC = (size_t)(C + kWordBits - 1) / kWordBits, taps = (size_t)KH * KW;
    // (of four words at most one is padding, of two taps one)
    return ((size_t)KN + 31) / 32 * (((taps + 1) * (PC + 1) + 1) / 2) * 512 * patch_weight_planes(type);
}

WeightJob patch_weight_job(int type, const ConvArgs &a, const PatchPlan &plan, uint64_t *out)
{
    const int planes = patch_weight_planes(type);
    const long items = (long)(plan.weight_bytes / 8 / planes);  // 64 lanes a run
    return WeightJob{a.qw, out, a.KN, (uint32_t)a.PC | (uint32_t)(a.KH * a.KW) << 16,
                     (uint32_t)((items + 255) / 256 + 7) / 8 * 8,  // whole groups of eight: the quantizer's workgroups stay on their XCDs
                     (uint32_t)plan.kc | (uint32_t)planes << 8};
}

hipError_t launch_conv(int type, const ConvArgs &args, hipStream_t stream)
{
    Forced forced = forced_kernel();
    if (forced_patch(forced)) forced.ng = -1;  // (the weights here are in their public order)
    const int force_tm = forced.tm, force_ng = forced.ng;
    if (args.qy != nullptr) {  // packed output exists in the matrix-core kernel's 64-wide shapes only
        if (!conv_mfma_exact(args)) return hipErrorInvalidValue;
        const int shape = (force_tm == 9 && force_ng >= 0 && force_ng != 3 && force_ng <= 11) ? force_ng : conv_mfma_shape(type, args);
        return launch_conv_mfma(type, args, shape, stream);
    }
    if (force_tm == 9) return launch_conv_mfma(type, args, force_ng < 0 ? conv_fp32_shape(type, args) : force_ng, stream);
    // default path: matrix cores; the popcount kernel takes over when K is too long for exact fp32
    // accumulation (and when a benchmark forces one of its tiles)
    if (force_tm == 0 && conv_mfma_exact(args)) return launch_conv_mfma(type, args, conv_fp32_shape(type, args), stream);
    // types 4 and 5 exist on the matrix cores only
    if (type > 3) return launch_conv_mfma(type, args, conv_fp32_shape(type, args), stream);
    switch (type) {
    case 0: return launch_type<0>(args, stream);
    case 1: return launch_type<1>(args, stream);
    case 2: return launch_type<2>(args, stream);
    case 3: return launch_type<3>(args, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace tab
