// C ABI of the library (declared in include/tab_amd.h): argument checks, workspace
// carving and kernel launches.  No allocation, no synchronisation, no host<->device copy.
#include "../../include/tab_amd.h"
#include "tab_common.h"

#include <cstdarg>
#include <cstdio>
#include <mutex>

// Packed-activation scratch of tab_conv2d_static, one copy per GPU the library is loaded on.  In host code this
// name is only a handle for hipGetSymbolAddress; the device address is looked up once per device (static_scratch
// below) and that pointer is what the kernels get.
static __device__ __align__(256) unsigned char scratch[TAB_STATIC_SCRATCH_BYTES];

namespace {

thread_local char g_last_error[512] = "";

int fail(int status, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_last_error, sizeof(g_last_error), fmt, ap);
    va_end(ap);
    return status;
}

int device_fail(hipError_t e, const char *what)
{
    return fail(TAB_ERR_DEVICE, "%s: %s", what, hipGetErrorString(e));
}

constexpr long kMaxIndex = 0x7fffffffL;  // kernels index rows/pixels with 32-bit ints

struct ConvShape {
    int PC, OH, OW, abits, wbits;
    long M, G;
};

// Shared validation of the conv geometry (TAB_GEMM.cu:354-379).
int check_conv(int type, int p1, int p2, int s1, int s2, int N, int H, int W, int C, int KN,
               int KH, int KW, ConvShape *s)
{
    if (type < 0 || type > 5)
        return fail(TAB_ERR_BAD_ARGUMENT, "type must be 0 (TNN), 1 (TBN), 2 (BTN), 3 (BNN), 4 (DRF) or 5 (RTN), got %d", type);
    if (N < 1 || H < 1 || W < 1 || C < 1 || KN < 1 || KH < 1 || KW < 1)
        return fail(TAB_ERR_BAD_ARGUMENT, "N, H, W, C, KN, KH, KW must be positive");
    if (p1 < 0 || p2 < 0 || s1 < 1 || s2 < 1)
        return fail(TAB_ERR_BAD_ARGUMENT, "padding must be >= 0 and stride >= 1");
    s->PC = type == TAB_RTN ? (C + 31) / 32 : tab_packed_channels(C);
    s->OH = tab_out_extent(H, p1, KH, s1);
    s->OW = tab_out_extent(W, p2, KW, s2);
    if (s->OH < 1 || s->OW < 1)
        return fail(TAB_ERR_BAD_SHAPE, "empty output: OH=%d OW=%d", s->OH, s->OW);
    s->abits = (type < 2 || type == TAB_DRF) ? 2 : 1;  // planes per word position, TAB_CPU.cpp:345-354 for type 4
    s->wbits = (type == 0 || type == 2 || type == TAB_DRF) ? 2 : 1;
    s->M = (long)N * s->OH * s->OW;
    s->G = (long)KH * KW * s->PC;
    if (s->M > kMaxIndex - 512 || s->G >= 65536 || s->PC >= 65536 || KW >= 65536 ||
        (long)N * H * W > kMaxIndex || (long)H * W * s->PC * 2 > kMaxIndex)
        return fail(TAB_ERR_BAD_SHAPE, "problem too large for 32-bit row indices (M=%ld, K words=%ld)", s->M, s->G);
    // type 4 multiplies levels up to 3: 9 * 64 * G has to stay below 2^24 for the fp32 accumulators
    if (type == TAB_DRF && s->G * 64 * 9 >= (1L << 24))
        return fail(TAB_ERR_BAD_SHAPE, "K of %ld words is too long for exact accumulation of type 4", s->G);
    // a workgroup addresses the images its (at most 256) output pixels touch with 32-bit byte offsets
    const long image_bytes = (long)H * W * s->PC * s->abits * 8;
    if (image_bytes * (256 / ((long)s->OH * s->OW) + 2) > 0xffffffffL)
        return fail(TAB_ERR_BAD_SHAPE, "packed image of %ld bytes is too large for 32-bit offsets", image_bytes);
    // a wave addresses its (at most 128) rows of Y with 32-bit byte offsets below 2 GiB
    if ((long)KN * 4 * 128 >= (1L << 31))
        return fail(TAB_ERR_BAD_SHAPE, "KN=%d is too large for 32-bit offsets into a tile of Y", KN);
    return TAB_OK;
}

}  // namespace

extern "C" {

const char *tab_status_string(int status)
{
    switch (status) {
    case TAB_OK: return "TAB_OK";
    case TAB_ERR_BAD_ARGUMENT: return "TAB_ERR_BAD_ARGUMENT";
    case TAB_ERR_BAD_SHAPE: return "TAB_ERR_BAD_SHAPE";
    case TAB_ERR_WORKSPACE: return "TAB_ERR_WORKSPACE";
    case TAB_ERR_DEVICE: return "TAB_ERR_DEVICE";
    default: return "TAB_ERR_UNKNOWN";
    }
}

const char *tab_last_error(void) { return g_last_error; }

const char *tab_version(void) { return "tab_amd 0.1 gfx950"; }

/* Test hook, absent from include/tab_amd.h: the kernels' multiply-shift division evaluated on the host (x < 2^31, 1 <= d < 2^31). */
uint32_t tab_internal_div32(uint32_t x, uint32_t d) { return tab::div32(x, tab::make_div32(d)); }

/* Test hook, absent from include/tab_amd.h: the matrix-core workgroup shape the library would pick for an M x KN output with
 * G = taps * PC words of K (packed: thresholded output), and the duration in microseconds its model predicts for it. */
int tab_internal_conv_shape(int type, int M, int KN, int G, int PC, int packed, float *cost_us)
{
    tab::ConvArgs a = {};
    a.M = M; a.KN = KN; a.G = G; a.PC = PC;
    a.qy = packed ? reinterpret_cast<uint32_t *>(&a) : nullptr;  // only tested against null
    return tab::conv_mfma_shape(type, a, cost_us);
}

/* Test hook, absent from include/tab_amd.h: the shape of a launch, the one above or, of fp32 output, one (19 .. 22) of the kernel that splits K
 * over the waves of a workgroup. */
int tab_internal_conv_launch_shape(int type, int M, int KN, int G, int PC, int packed)
{
    tab::ConvArgs a = {};
    a.M = M; a.KN = KN; a.G = G; a.PC = PC;
    a.qy = packed ? reinterpret_cast<uint32_t *>(&a) : nullptr;  // only tested against null
    return tab::conv_fp32_shape(type, a);
}

/* Test hook, absent from include/tab_amd.h: the shape (19 .. 22) of the kernel that splits K over waves for a launch that is to go there. */
int tab_internal_conv_waves_shape(int type, int M, int KN, int G, int PC)
{
    tab::ConvArgs a = {};
    a.M = M; a.KN = KN; a.G = G; a.PC = PC;
    return tab::conv_waves_shape(type, a, nullptr);
}

/* Test hook, absent from include/tab_amd.h: what the kernel that splits K over waves is predicted to gain over the tiled ones, in microseconds;
 * infinity where those of 32x32 rank first, -infinity where it is not taken. */
float tab_internal_conv_waves_gain(int type, int M, int KN, int G, int PC)
{
    tab::ConvArgs a = {};
    a.M = M; a.KN = KN; a.G = G; a.PC = PC;
    return tab::conv_waves_gain(type, a);
}

/* Test hook, absent from include/tab_amd.h: workgroups a CU of a packed layer of short K. */
int tab_internal_regs_on_cu(int G, int tiles, int tiles_n, int most, int cus) { return tab::regs_on_cu(G, tiles, tiles_n, most, cus); }

/* Test hook, absent from include/tab_amd.h: whether items of two planes take a workgroup each (own: with thresholds of their own, else with
 * counts). */
int tab_internal_quantize_items(int own, int nchw, long items, long pixels, int C) { return tab::quantize_items_supported(own, nchw, items, pixels, C); }

/* Test hook, absent from include/tab_amd.h: the form of an NCHW quantizer: -1 gathered words, else the waves of a last word apart, 0 of none. */
int tab_internal_plane_form(int bitwidth, long N, long HW, int C)
{
    const tab::PlaneForm form = tab::plane_form(bitwidth, N, HW, C);
    return form.gather ? -1 : form.last;
}

/* Test hook, absent from include/tab_amd.h: whether the one-launch kernel of the smallest calls can run a call, and its predicted
 * duration on the GPU in microseconds with the three numbers it comes from. */
int tab_internal_conv_small_cost(int type, const float *dev_X, int nchw, int N, int H, int W, int C, int KN, int KH, int KW, int padding1,
                                 int padding2, int stride1, int stride2, float *cost)
{
    float c[4];
    const int OH = tab_out_extent(H, padding1, KH, stride1), OW = tab_out_extent(W, padding2, KW, stride2);
    if (OH < 1 || OW < 1 || !tab::conv_small_cost(type, dev_X, nchw != 0, N, H, W, C, KN, KH, KW, padding1, padding2, stride1, stride2, OH, OW, c))
        return 0;
    for (int i = 0; i < 4; i++) cost[i] = c[i];
    return 1;
}

/* Test hook, absent from include/tab_amd.h: the number of workgroups the mixed launch (TAB_CONV_MATRIX tile 10) counts as one
 * round of the chip; 0 = the device's compute units.  Small values let small test shapes mix whole tiles and quarters. */
void tab_internal_set_tail_round(int workgroups) { tab::set_tail_round(workgroups); }

/* Test hook, absent from include/tab_amd.h: the compute units that the rules choosing a kernel count; 0 = the device's. */
void tab_internal_set_compute_units(int units) { tab::set_compute_units(units); }

/* Test hook, absent from include/tab_amd.h: convolutions from fp32 take this shape (12 .. 18) of the kernel that keeps the input
 * patch in LDS wherever its patch fits, or this one (19 .. 22) of the kernel that splits K over waves; tab_set_conv_kernel ends it. */
void tab_internal_force_patch(int shape) { tab::force_conv_tile(9, shape); }

int tab_set_conv_kernel(int kernel, int tile)
{
    static const int popcount_tm[4] = {7, 8, 4, 2};  // 7: the popcount kernel's own choice
    if (kernel == TAB_CONV_AUTO && tile == -1) tab::force_conv_tile(0, 0);
    else if (kernel == TAB_CONV_MATRIX && tile >= -1 && tile <= 11) tab::force_conv_tile(9, tile);
    else if (kernel == TAB_CONV_POPCOUNT && tile >= -1 && tile <= 2) tab::force_conv_tile(popcount_tm[tile + 1], 0);
    else return fail(TAB_ERR_BAD_ARGUMENT, "no conv kernel %d with tile %d", kernel, tile);
    return TAB_OK;
}

int tab_packed_channels(int C) { return (C + tab::kWordBits - 1) / tab::kWordBits; }

int tab_out_extent(int in, int pad, int k, int stride)
{
    if (stride < 1) return 0;
    return (in + 2 * pad - k + 1) / stride;
}

static int quantize_any(const float *dev_X, const float *dev_ths, bool nchw, int bitwidth, int N, int H, int W, int C, int64_t *dev_QX,
                        int32_t *dev_BTN, int32_t *count_workspace, void *stream)
{
    if (bitwidth != 1 && bitwidth != 2) return fail(TAB_ERR_BAD_ARGUMENT, "bitwidth must be 1 or 2, got %d", bitwidth);
    if (N < 1 || H < 1 || W < 1 || C < 1) return fail(TAB_ERR_BAD_ARGUMENT, "N, H, W, C must be positive");
    if (!dev_X || !dev_ths || !dev_QX) return fail(TAB_ERR_BAD_ARGUMENT, "null device pointer");  // dev_BTN may be NULL
    if (((uintptr_t)dev_X % 4) || ((uintptr_t)dev_QX % (8 * bitwidth)))
        return fail(TAB_ERR_BAD_ARGUMENT, "X must be aligned to its floats and QX to a whole packed element (%d bytes)", 8 * bitwidth);
    if (nchw && ((long)N * H * W + 255) / 256 * tab_packed_channels(C) > kMaxIndex)
        return fail(TAB_ERR_BAD_SHAPE, "tensor too large for one launch (N*H*W/256 * ceil(C/64) workgroups)");
    const tab::Thresholds ths = tab::given_thresholds(dev_ths);
    uint64_t *q = reinterpret_cast<uint64_t *>(dev_QX);
    const hipError_t e =
        nchw ? tab::launch_quantize_nchw(dev_X, ths, bitwidth, N, C, (long)H * W, q, dev_BTN, count_workspace, static_cast<hipStream_t>(stream))
             : tab::launch_quantize(dev_X, ths, bitwidth, (long)H * W, N, C, q, dev_BTN, count_workspace, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return device_fail(e, "quantize launch");
    return TAB_OK;
}

int tab_quantize(const float *dev_X, const float *dev_ths, int bitwidth, int N, int H, int W,
                 int C, int64_t *dev_QX, int32_t *dev_BTN, void *stream)
{
    return quantize_any(dev_X, dev_ths, false, bitwidth, N, H, W, C, dev_QX, dev_BTN, nullptr, stream);
}

int tab_quantize_nchw(const float *dev_X, const float *dev_ths, int bitwidth, int N, int C, int H, int W,
                      int64_t *dev_QX, int32_t *dev_BTN, void *stream)
{
    return quantize_any(dev_X, dev_ths, true, bitwidth, N, H, W, C, dev_QX, dev_BTN, nullptr, stream);
}

size_t tab_quantize_workspace_bytes(int bitwidth, int N, int H, int W, int C)
{
    if (N < 1 || H < 1 || W < 1 || C < 1) return 0;
    return tab::quantize_count_workspace(bitwidth, N, (long)H * W, C);
}

int tab_quantize_counted(const float *dev_X, const float *dev_ths, int nchw, int bitwidth, int N, int H, int W, int C, int64_t *dev_QX,
                         int32_t *dev_BTN, void *workspace, size_t workspace_bytes, void *stream)
{
    if (!dev_BTN) return fail(TAB_ERR_BAD_ARGUMENT, "null device pointer");
    const size_t need = tab_quantize_workspace_bytes(bitwidth, N, H, W, C);
    if (need && (!workspace || workspace_bytes < need || ((uintptr_t)workspace % 4)))
        return fail(TAB_ERR_WORKSPACE, "workspace must hold %zu bytes (got %zu)", need, workspace_bytes);
    return quantize_any(dev_X, dev_ths, nchw != 0, bitwidth, N, H, W, C, dev_QX, dev_BTN, need ? static_cast<int32_t *>(workspace) : nullptr, stream);
}

size_t tab_threshold_workspace_bytes(int N, long per_item)
{
    if (N < 1 || per_item < 1) return 0;
    return (size_t)N * tab::threshold_splits(N, per_item) * sizeof(float);
}

int tab_threshold(const float *dev_X, int N, long per_item, float scale, float *dev_ths, void *workspace,
                  size_t workspace_bytes, void *stream)
{
    if (N < 1 || per_item < 1) return fail(TAB_ERR_BAD_ARGUMENT, "N and per_item must be positive");
    if (!dev_X || !dev_ths) return fail(TAB_ERR_BAD_ARGUMENT, "null device pointer");
    const size_t need = tab_threshold_workspace_bytes(N, per_item);
    if (!workspace || workspace_bytes < need || ((uintptr_t)workspace % 4))
        return fail(TAB_ERR_WORKSPACE, "workspace must hold %zu bytes (got %zu)", need, workspace_bytes);
    hipError_t e = tab::launch_threshold(dev_X, N, per_item, scale, dev_ths, static_cast<float *>(workspace),
                                         static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return device_fail(e, "threshold launch");
    return TAB_OK;
}

int tab_operand_words(int type, int operand, int C)
{
    if (type < 0 || type > 5 || operand < 0 || operand > 1 || C < 1) return 0;
    if (type == TAB_RTN) return (C + 31) / 32;
    const bool two_planes = type == TAB_DRF || (operand == 0 ? type < 2 : (type == 0 || type == 2));
    return tab_packed_channels(C) * (two_planes ? 2 : 1);
}

size_t tab_conv2d_workspace_bytes(int type, int N, int H, int W, int C)
{
    if (type < 0 || type > 5 || N < 1 || H < 1 || W < 1 || C < 1) return 0;
    return (size_t)N * H * W * tab_operand_words(type, 0, C) * sizeof(int64_t);
}

/* Room for a convolution's weights in another kernel's order, aligned. */
static size_t spare_weight_bytes(int type, int C, int KN, int KH, int KW)
{
    const size_t bytes = KH > 1 || KW > 1 ? tab::patch_weight_bytes(type, C, KN, KH, KW) : 0;
    return bytes ? bytes + 16 : 0;
}

size_t tab_conv2d_workspace_bytes_full(int type, int N, int H, int W, int C, int KN, int KH, int KW)
{
    const size_t need = tab_conv2d_workspace_bytes(type, N, H, W, C);
    if (need == 0 || KN < 1 || KH < 1 || KW < 1) return 0;
    return need + spare_weight_bytes(type, C, KN, KH, KW);
}

int tab_quantize_format(const float *dev_X, const float *dev_ths, int type, int N, int H, int W, int C,
                        int64_t *dev_QX, void *stream)
{
    if (type != TAB_DRF && type != TAB_RTN) return fail(TAB_ERR_BAD_ARGUMENT, "type must be 4 (DRF) or 5 (RTN), got %d", type);
    if (N < 1 || H < 1 || W < 1 || C < 1) return fail(TAB_ERR_BAD_ARGUMENT, "N, H, W, C must be positive");
    if (!dev_X || !dev_ths || !dev_QX) return fail(TAB_ERR_BAD_ARGUMENT, "null device pointer");
    if (((uintptr_t)dev_X % 4) || ((uintptr_t)dev_QX % 16))
        return fail(TAB_ERR_BAD_ARGUMENT, "X must be aligned to its floats and QX to 16 bytes");
    hipError_t e = tab::launch_quantize_format(dev_X, dev_ths, type, (long)H * W, N, C, reinterpret_cast<uint64_t *>(dev_QX),
                                               static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return device_fail(e, "quantize launch");
    return TAB_OK;
}

/* Pointer checks shared by every conv entry point; they run before anything is launched. */
static int check_conv_pointers(const ConvShape &s, int type, const void *dev_QX, const void *dev_QW, const void *dev_btn,
                               const void *dev_Y, const void *dev_QY)
{
    if (!dev_QX || !dev_QW || (!dev_Y && !dev_QY)) return fail(TAB_ERR_BAD_ARGUMENT, "null device pointer");
    if (type == TAB_BTN && !dev_btn) return fail(TAB_ERR_BAD_ARGUMENT, "btn is required for type 2 (BTN)");
    if (((uintptr_t)dev_QX % (8 * s.abits)) || ((uintptr_t)dev_QW % (8 * s.wbits)) || ((uintptr_t)dev_Y % 16))
        return fail(TAB_ERR_BAD_ARGUMENT, "QX/QW must be aligned to a whole packed element and Y to 16 bytes");
    return TAB_OK;
}

/* The sizes of the kernels' arguments, which is what the rules that pick a kernel read. */
static tab::ConvArgs conv_sizes(const ConvShape &s, int padding1, int padding2, int stride1, int stride2, int N, int H, int W, int KN, int KH, int KW)
{
    tab::ConvArgs a;
    a.qx = nullptr; a.qw = nullptr; a.btn = nullptr;
    a.y = nullptr; a.qy = nullptr;
    a.out_ths = nullptr;
    a.out_th = 0.f;
    a.out_bits = 0;
    a.N = N; a.H = H; a.W = W; a.PC = s.PC;
    a.KN = KN; a.KH = KH; a.KW = KW;
    a.p1 = padding1; a.p2 = padding2; a.s1 = stride1; a.s2 = stride2;
    a.OH = s.OH; a.OW = s.OW;
    a.M = (int)s.M;
    a.G = (int)s.G;
    return a;
}

/* The kernels' arguments for fp32 output. */
static tab::ConvArgs conv_args(const ConvShape &s, int padding1, int padding2, int stride1, int stride2, int N, int H, int W, int C, int KN,
                               int KH, int KW, const void *dev_QX, const int64_t *dev_QW, const int32_t *dev_btn, float *dev_Y)
{
    tab::ConvArgs a = conv_sizes(s, padding1, padding2, stride1, stride2, N, H, W, KN, KH, KW);
    a.qx = static_cast<const uint64_t *>(dev_QX);
    a.qw = reinterpret_cast<const uint64_t *>(dev_QW);
    a.btn = dev_btn;
    a.y = dev_Y;
    a.kcw = 0; a.nchunks = 0; a.tiles_m = 0;
    a.num = KH * KW * C;
    a.div_pc = tab::make_fastdiv((uint32_t)s.PC);
    a.div_kw = tab::make_fastdiv((uint32_t)KW);
    a.div_pixels = tab::make_div32((uint32_t)(s.OH * s.OW));
    a.div_ow = tab::make_div32((uint32_t)s.OW);
    a.div_tiles_m = tab::make_div32(1);
    a.tiles_n = 0;
    a.xcd_share = 0; a.filter_tiles = 1; a.tail_big = 0; a.tail_chunks = 0;
    // A Y that fits the 256 MB last-level cache beside the operands but not the L2s is written through the caches
    // (the cache takes the stores faster than HBM: Y of 190-206 MB 1-11 % sooner); every other Y with non-temporal
    // stores: a smaller one leaves no dirty L2 to flush when the launch ends (7-25 % sooner), a larger one would only
    // push the operands out (Y of 411 MB: 7-28 % sooner).  At 103 MB the two policies measured within 3 %.
    // A Y of 24 MB or more whose rows are no whole cache lines goes through the caches (tab::ragged_rows_cached).
    const long y_bytes = s.M * (long)KN * 4;
    a.y_cached = (y_bytes >= (128L << 20) && y_bytes <= (240L << 20)) || tab::ragged_rows_cached(s.M, KN);
    a.div_filter_tiles = tab::make_div32(1);
    return a;
}

/* Shared body of the packed-activation entry points: Y as fp32 (dev_Y) or thresholded (dev_out_ths per image, or out_th
 * for all of them) and packed (dev_QY). */
static int conv_packed(const int64_t *dev_QX, const int64_t *dev_QW, const int32_t *dev_btn, int type, int padding1,
                       int padding2, int stride1, int stride2, int N, int H, int W, int C, int KN, int KH, int KW,
                       float *dev_Y, const float *dev_out_ths, float out_th, int out_bitwidth, int64_t *dev_QY, void *stream)
{
    ConvShape s;
    int rc = check_conv(type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, &s);
    if (rc != TAB_OK) return rc;
    rc = check_conv_pointers(s, type, dev_QX, dev_QW, dev_btn, dev_Y, dev_QY);
    if (rc != TAB_OK) return rc;
    if (dev_QY) {
        if (out_bitwidth != 1 && out_bitwidth != 2)
            return fail(TAB_ERR_BAD_ARGUMENT, "out_bitwidth must be 1 or 2, got %d", out_bitwidth);
        if ((uintptr_t)dev_QY % (8 * out_bitwidth)) return fail(TAB_ERR_BAD_ARGUMENT, "QY must be aligned to a whole packed element");
    }

    tab::ConvArgs a = conv_args(s, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, dev_QX, dev_QW, dev_btn, dev_Y);
    a.qy = reinterpret_cast<uint32_t *>(dev_QY);
    a.out_ths = dev_out_ths;
    a.out_th = out_th;
    a.out_bits = out_bitwidth;
    hipError_t e = tab::launch_conv(type, a, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return device_fail(e, "conv launch");
    return TAB_OK;
}

int tab_conv2d_packed(const int64_t *dev_QX, const int64_t *dev_QW, const int32_t *dev_btn,
                      int type, int padding1, int padding2, int stride1, int stride2, int N,
                      int H, int W, int C, int KN, int KH, int KW, float *dev_Y, void *stream)
{
    if (!dev_Y) return fail(TAB_ERR_BAD_ARGUMENT, "null device pointer");
    return conv_packed(dev_QX, dev_QW, dev_btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW,
                       dev_Y, nullptr, 0.f, 0, nullptr, stream);
}

int tab_conv2d_packed_out(const int64_t *dev_QX, const int64_t *dev_QW, const int32_t *dev_btn,
                          int type, int padding1, int padding2, int stride1, int stride2, int N,
                          int H, int W, int C, int KN, int KH, int KW, const float *dev_out_ths,
                          int out_bitwidth, int64_t *dev_QY, void *stream)
{
    if (!dev_QY || !dev_out_ths) return fail(TAB_ERR_BAD_ARGUMENT, "null device pointer");
    return conv_packed(dev_QX, dev_QW, dev_btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW,
                       nullptr, dev_out_ths, 0.f, out_bitwidth, dev_QY, stream);
}

int tab_conv2d_packed_out_const(const int64_t *dev_QX, const int64_t *dev_QW, const int32_t *dev_btn,
                                int type, int padding1, int padding2, int stride1, int stride2, int N,
                                int H, int W, int C, int KN, int KH, int KW, float out_threshold,
                                int out_bitwidth, int64_t *dev_QY, void *stream)
{
    if (!dev_QY) return fail(TAB_ERR_BAD_ARGUMENT, "null device pointer");
    return conv_packed(dev_QX, dev_QW, dev_btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW,
                       nullptr, nullptr, out_threshold, out_bitwidth, dev_QY, stream);
}

/* Test hook, absent from include/tab_amd.h: the shape (12 .. 18) of the kernel that keeps the input patch in LDS which the library would
 * pick for a convolution from fp32, -1 for another kernel; what[0..2]: words of a chunk, pixels and LDS bytes of its patch. */
int tab_internal_conv_patch_shape(int type, int padding1, int padding2, int stride1, int stride2, int N, int H, int W, int C, int KN, int KH,
                                  int KW, int *what, size_t *weight_bytes)
{
    ConvShape s;
    if (check_conv(type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, &s) != TAB_OK) return -1;
    const tab::ConvArgs a = conv_sizes(s, padding1, padding2, stride1, stride2, N, H, W, KN, KH, KW);
    const tab::PatchPlan plan = tab::conv_patch_plan(type, a);
    if (plan.shape < 0) return -1;
    what[0] = plan.kc;
    what[1] = plan.npix;
    what[2] = plan.lds_bytes;
    *weight_bytes = plan.weight_bytes;
    return plan.shape;
}

/* Test hook, absent from include/tab_amd.h: the shape that tab_internal_force_patch holds, on an activation already packed.
 * what: 1 = lay the weights out in `weights` (weight_bytes bytes), 2 = convolve with those there, 3 = both. */
int tab_internal_conv_patch(const int64_t *dev_QX, const int64_t *dev_QW, const int32_t *dev_btn, int type, int padding1, int padding2,
                            int stride1, int stride2, int N, int H, int W, int C, int KN, int KH, int KW, float *dev_Y, void *weights,
                            size_t weight_bytes, int what, void *stream)
{
    ConvShape s;
    int rc = check_conv(type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, &s);
    if (rc == TAB_OK) rc = check_conv_pointers(s, type, dev_QX, dev_QW, dev_btn, dev_Y, nullptr);
    if (rc != TAB_OK) return rc;
    tab::ConvArgs a = conv_args(s, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, dev_QX, dev_QW, dev_btn, dev_Y);
    const tab::PatchPlan plan = tab::conv_patch_plan(type, a);
    if (plan.shape < 0) return fail(TAB_ERR_BAD_SHAPE, "the patch does not fit");
    if (!weights || weight_bytes < plan.weight_bytes) return fail(TAB_ERR_WORKSPACE, "weights take %zu bytes", plan.weight_bytes);
    hipError_t e = hipSuccess;
    if (what & 1) e = tab::launch_patch_weights(tab::patch_weight_job(type, a, plan, static_cast<uint64_t *>(weights)), static_cast<hipStream_t>(stream));
    a.qw = static_cast<const uint64_t *>(weights);
    if (e == hipSuccess && (what & 2)) e = tab::launch_conv_mfma(type, a, plan.shape, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return device_fail(e, "conv launch");
    return TAB_OK;
}

/* Device address of `scratch` on the current device, looked up on the first call made with that device current. */
static int static_scratch(void **out)
{
    constexpr int kMaxDevices = 64;
    static std::mutex mutex;
    static void *address[kMaxDevices] = {};
    int device = -1;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return device_fail(e, "hipGetDevice");
    if (device < 0 || device >= kMaxDevices) return fail(TAB_ERR_DEVICE, "device index %d out of range", device);
    std::lock_guard<std::mutex> lock(mutex);
    if (address[device] == nullptr) {
        void *ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return device_fail(e, "hipGetSymbolAddress(scratch)");
        if (ptr == nullptr) return fail(TAB_ERR_DEVICE, "hipGetSymbolAddress(scratch) gave no address");
        address[device] = ptr;
    }
    *out = address[device];
    return TAB_OK;
}

/* Pointer, alignment and size checks of the calls that start from fp32: everything the second stage would reject is
 * rejected before the quantizer is enqueued. */
static int check_from_floats(const ConvShape &s, int type, const float *dev_X, const int64_t *dev_QW, const int32_t *dev_btn,
                             const float *dev_Y, const void *workspace, size_t workspace_bytes, size_t need)
{
    if (!dev_X) return fail(TAB_ERR_BAD_ARGUMENT, "null device pointer");
    if ((uintptr_t)dev_X % 4) return fail(TAB_ERR_BAD_ARGUMENT, "X must be aligned to its floats");
    if (!workspace || workspace_bytes < need || ((uintptr_t)workspace % 16))
        return fail(TAB_ERR_WORKSPACE, "workspace must be 16-byte aligned and hold %zu bytes (got %zu)", need, workspace_bytes);
    return check_conv_pointers(s, type, workspace, dev_QW, dev_btn, dev_Y, nullptr);
}

/* Which kernel takes a call from fp32 in one launch: 0 none, 1 conv1x1_fused, 2 conv_small.  own_thresholds: each image is one pixel
 * whose threshold the kernel is to find. */
static int one_launch(int type, const float *dev_X, bool nchw, int padding1, int padding2, int stride1, int stride2, int N, int H, int W,
                      int C, int KN, int KH, int KW, const ConvShape &s, bool own_thresholds = false)
{
    if (tab::conv_kernel_forced()) return 0;
    const bool small = tab::conv_small_supported(type, dev_X, nchw, N, H, W, C, KN, KH, KW, padding1, padding2, stride1, stride2, s.OH, s.OW);
    // of 1x1 layers both take, conv_small is the sooner one from five words a pixel on (N=64 512->1000 4.8 against 5.4 us),
    // conv1x1_fused below (64->64 3.8 against 3.0), but where the kernel is to find the thresholds itself, which conv_small can
    // and which is a launch less (N=277 256->55 ternary layer 7.4 -> 5.2)
    if (!nchw && !(small && (s.PC > 4 || own_thresholds)) && tab::conv1x1_fused_supported(type, dev_X, C, KH, KW, padding1, padding2, s.M, KN)) return 1;
    return small ? 2 : 0;
}

/* A convolution of an activation that is still to be quantized: which kernel multiplies it, and where in the workspace (`room`
 * bytes at `spare`, behind the packed activation) the quantizer's launch leaves the weights in that kernel's order. */
struct ConvRoute {
    tab::ConvArgs args;
    tab::PatchPlan plan;
    tab::WeightJob job;
    const tab::WeightJob *weights() const { return plan.shape >= 0 ? &job : nullptr; }
};

/* plan: already made, or null; without room for weights none is made (0.15-0.2 us of the host). */
static ConvRoute conv_route(const tab::ConvArgs &args, int type, const tab::PatchPlan *plan, void *spare, size_t room)
{
    ConvRoute r = {args, plan ? *plan : room ? tab::conv_patch_plan(type, args) : tab::PatchPlan{-1, 0, 0, 0, -1, 0}, {}};
    char *at = reinterpret_cast<char *>(((uintptr_t)spare + 15) & ~(uintptr_t)15);
    const size_t lost = (size_t)(at - static_cast<char *>(spare));
    if (r.plan.shape >= 0 && (room < lost || room - lost < r.plan.weight_bytes)) r.plan.shape = -1;
    if (r.plan.shape >= 0) r.job = tab::patch_weight_job(type, args, r.plan, reinterpret_cast<uint64_t *>(at));
    return r;
}

/* The convolution of a route whose quantizer has been enqueued. */
static int run_route(const ConvRoute &r, int type, void *stream)
{
    tab::ConvArgs a = r.args;
    if (r.plan.shape >= 0) a.qw = r.job.out;
    const int shape = r.plan.shape >= 0 ? r.plan.shape : r.plan.tiled;
    const hipError_t e = shape >= 0 ? tab::launch_conv_mfma(type, a, shape, static_cast<hipStream_t>(stream))
                                    : tab::launch_conv(type, a, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return device_fail(e, "conv launch");
    return TAB_OK;
}

/* Quantize an NHWC activation of types 0..3 into the workspace, then the fused conv kernel; small and strided 1x1 layers
 * take their own ways.  The arguments have been checked.  spare, room: of the workspace, behind what the call needs. */
static int conv_from_nhwc(const float *dev_X, const int64_t *dev_QW, const tab::Thresholds &ths, const int32_t *dev_btn, int type,
                          int padding1, int padding2, int stride1, int stride2, int N, int H, int W, int C, int KN, int KH, int KW,
                          const ConvShape &s, float *dev_Y, void *workspace, const tab::PatchPlan *plan, void *spare, size_t room, void *stream)
{
    // One launch where it pays (only under the automatic kernel choice: a forced kernel is what the caller wants to see run):
    // a 1x1 convolution without padding, the smallest calls of any kernel.  The packed activation stays in LDS.
    if (const int one = one_launch(type, dev_X, false, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, s,
                                   ths.splits == tab::kOwnPixelThresholds)) {
        hipError_t e = one == 1 ? tab::launch_conv1x1_fused(type, dev_X, ths, reinterpret_cast<const uint64_t *>(dev_QW), dev_btn, dev_Y, N, H, W,
                                                            C, KN, stride1, stride2, s.OH, s.OW, static_cast<hipStream_t>(stream))
                                : tab::launch_conv_small(type, dev_X, false, ths, reinterpret_cast<const uint64_t *>(dev_QW), dev_btn, dev_Y, N, H, W,
                                                         C, KN, KH, KW, padding1, padding2, stride1, stride2, s.OH, s.OW, static_cast<hipStream_t>(stream));
        if (e != hipSuccess) return device_fail(e, "conv launch");
        return TAB_OK;
    }
    // A 1x1 convolution with stride and no padding reads one pixel in stride1*stride2: quantize only
    // those, into a compact activation, and convolve it with stride 1 (same outputs, a fraction of
    // the reads of X).
    if (KH == 1 && KW == 1 && padding1 == 0 && padding2 == 0 && (stride1 > 1 || stride2 > 1) && N * (long)s.OH < 65536 &&
        tab::quantize_strided_supported(dev_X, H, W, C, s.OH, s.OW)) {
        hipError_t e = tab::launch_quantize_strided(dev_X, ths, s.abits, N, H, W, C, s.OH, s.OW, stride1, stride2,
                                                    reinterpret_cast<uint64_t *>(workspace), static_cast<hipStream_t>(stream));
        if (e != hipSuccess) return device_fail(e, "quantize launch");
        return tab_conv2d_packed(reinterpret_cast<const int64_t *>(workspace), dev_QW, dev_btn, type, 0, 0, 1, 1, N, s.OH,
                                 s.OW, C, KN, 1, 1, dev_Y, stream);
    }
    const ConvRoute route = conv_route(conv_args(s, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, workspace, dev_QW, dev_btn, dev_Y),
                                       type, plan, spare, room);
    // stage 1: quantize + pack the activation (TAB_GEMM.cu:419-426); no btn for activations
    hipError_t e = tab::launch_quantize(dev_X, ths, s.abits, (long)H * W, N, C, reinterpret_cast<uint64_t *>(workspace), nullptr,
                                        nullptr, static_cast<hipStream_t>(stream), route.weights());
    if (e != hipSuccess) return device_fail(e, "quantize launch");
    // stage 2: pad + im2row + GEMM, fused
    return run_route(route, type, stream);
}

/* Body of tab_conv2d and tab_conv2d_static (builtin: the library's own scratch). */
static int conv_from_floats(const float *dev_X, const int64_t *dev_QW, const float *dev_ths, const int32_t *dev_btn, int type,
                            int padding1, int padding2, int stride1, int stride2, int N, int H, int W, int C, int KN, int KH,
                            int KW, float *dev_Y, void *workspace, size_t workspace_bytes, bool builtin, const tab::PatchPlan *plan, void *stream)
{
    ConvShape s;
    int rc = check_conv(type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, &s);
    if (rc != TAB_OK) return rc;
    if (!dev_X || !dev_ths) return fail(TAB_ERR_BAD_ARGUMENT, "null device pointer");
    const size_t need = tab_conv2d_workspace_bytes(type, N, H, W, C);
    if (builtin) {
        if (need > TAB_STATIC_SCRATCH_BYTES)
            return fail(TAB_ERR_WORKSPACE, "the packed activation needs %zu bytes, the built-in scratch holds %zu; use tab_conv2d with a workspace",
                        need, (size_t)TAB_STATIC_SCRATCH_BYTES);
        rc = static_scratch(&workspace);
        if (rc != TAB_OK) return rc;
        workspace_bytes = TAB_STATIC_SCRATCH_BYTES;
    }
    rc = check_from_floats(s, type, dev_X, dev_QW, dev_btn, dev_Y, workspace, workspace_bytes, need);
    if (rc != TAB_OK) return rc;
    void *const spare = static_cast<char *>(workspace) + need;
    const size_t room = workspace_bytes - need;
    if (type > 3 && !one_launch(type, dev_X, false, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, s)) {
        // the CPU-only types: their own packers, then the same fused kernel
        const ConvRoute route = conv_route(conv_args(s, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, workspace, dev_QW, dev_btn, dev_Y),
                                           type, plan, spare, room);
        hipError_t e = tab::launch_quantize_format(dev_X, dev_ths, type, (long)H * W, N, C, reinterpret_cast<uint64_t *>(workspace),
                                                   static_cast<hipStream_t>(stream), route.weights());
        if (e != hipSuccess) return device_fail(e, "quantize launch");
        return run_route(route, type, stream);
    }
    return conv_from_nhwc(dev_X, dev_QW, tab::given_thresholds(dev_ths), dev_btn, type, padding1, padding2, stride1, stride2, N, H, W, C,
                          KN, KH, KW, s, dev_Y, workspace, plan, spare, room, stream);
}

/* Packed activation bytes of a layer call, rounded up so that the partial sums behind them are aligned. */
static size_t layer_packed_bytes(int bitwidth, int N, int H, int W, int C)
{
    return ((size_t)N * H * W * tab_packed_channels(C) * bitwidth * sizeof(int64_t) + 15) & ~(size_t)15;
}

/* Thresholds of an activation taken from itself: 0 for one plane, act_scale * mean|x| per item for two, whose partial sums
 * (launched here) go to `sums`. */
static hipError_t own_thresholds(const float *dev_X, int bitwidth, float act_scale, int N, long per_item, void *sums,
                                 tab::Thresholds *ths, void *stream)
{
    *ths = tab::given_thresholds(nullptr);
    if (bitwidth == 1) return hipSuccess;
    return tab::launch_abs_sums(dev_X, N, per_item, act_scale, static_cast<float *>(sums), ths, static_cast<hipStream_t>(stream));
}

size_t tab_layer_workspace_bytes(int bitwidth, int N, int H, int W, int C)
{
    if (bitwidth < 1 || bitwidth > 2 || N < 1 || H < 1 || W < 1 || C < 1) return 0;
    const size_t sums = tab_threshold_workspace_bytes(N, (long)H * W * C) + (size_t)N * sizeof(float);
    return layer_packed_bytes(bitwidth, N, H, W, C) + (bitwidth == 2 ? sums : 0);
}

size_t tab_layer_workspace_bytes_full(int type, int N, int H, int W, int C, int KN, int KH, int KW)
{
    if (type < 0 || type > 3 || KN < 1 || KH < 1 || KW < 1) return 0;
    const size_t need = tab_layer_workspace_bytes(type < 2 ? 2 : 1, N, H, W, C);
    return need ? need + spare_weight_bytes(type, C, KN, KH, KW) : 0;
}

/* weights: of the convolution that follows, or null. */
static int layer_quantize(const float *dev_X, int nchw, int bitwidth, float act_scale, int N, int H, int W, int C, int64_t *dev_QX,
                          void *workspace, size_t workspace_bytes, const tab::WeightJob *weights, void *stream)
{
    if (bitwidth != 1 && bitwidth != 2) return fail(TAB_ERR_BAD_ARGUMENT, "bitwidth must be 1 or 2, got %d", bitwidth);
    if (N < 1 || H < 1 || W < 1 || C < 1) return fail(TAB_ERR_BAD_ARGUMENT, "N, H, W, C must be positive");
    if (!dev_X || !dev_QX) return fail(TAB_ERR_BAD_ARGUMENT, "null device pointer");
    if (((uintptr_t)dev_X % 4) || ((uintptr_t)dev_QX % (8 * bitwidth)))
        return fail(TAB_ERR_BAD_ARGUMENT, "X must be aligned to its floats and QX to a whole packed element (%d bytes)", 8 * bitwidth);
    if (nchw && ((long)N * H * W + 255) / 256 * tab_packed_channels(C) > kMaxIndex)
        return fail(TAB_ERR_BAD_SHAPE, "tensor too large for one launch (N*H*W/256 * ceil(C/64) workgroups)");
    const long per_item = (long)H * W * C;
    const size_t need = bitwidth == 2 ? tab_threshold_workspace_bytes(N, per_item) : 0;
    if (need && (!workspace || workspace_bytes < need || ((uintptr_t)workspace % 4)))
        return fail(TAB_ERR_WORKSPACE, "workspace must hold %zu bytes (got %zu)", need, workspace_bytes);
    tab::Thresholds ths;
    uint64_t *q = reinterpret_cast<uint64_t *>(dev_QX);
    if (bitwidth == 2 && !weights && tab::quantize_items_supported(true, nchw && H * W > 1, N, (long)H * W, C)) {
        const hipError_t e = tab::launch_quantize_own(dev_X, act_scale, nchw && H * W > 1, N, (long)H * W, C, q, static_cast<hipStream_t>(stream));
        if (e != hipSuccess) return device_fail(e, "quantize launch");
        return TAB_OK;
    }
    hipError_t e = own_thresholds(dev_X, bitwidth, act_scale, N, per_item, workspace, &ths, stream);
    if (e != hipSuccess) return device_fail(e, "threshold launch");
    // one pixel per image: NCHW and NHWC are the same memory, and the NHWC quantizers read it along the channels
    e = nchw && H * W > 1 ? tab::launch_quantize_nchw(dev_X, ths, bitwidth, N, C, (long)H * W, q, nullptr, nullptr, static_cast<hipStream_t>(stream), weights)
                          : tab::launch_quantize(dev_X, ths, bitwidth, (long)H * W, N, C, q, nullptr, nullptr, static_cast<hipStream_t>(stream), weights);
    if (e != hipSuccess) return device_fail(e, "quantize launch");
    return TAB_OK;
}

int tab_layer_quantize(const float *dev_X, int nchw, int bitwidth, float act_scale, int N, int H, int W, int C, int64_t *dev_QX,
                       void *workspace, size_t workspace_bytes, void *stream)
{
    return layer_quantize(dev_X, nchw, bitwidth, act_scale, N, H, W, C, dev_QX, workspace, workspace_bytes, nullptr, stream);
}

int tab_internal_layer_conv2d(const float *dev_X, int nchw, float act_scale, const int64_t *dev_QW, const int32_t *dev_btn, int type,
                              int padding1, int padding2, int stride1, int stride2, int N, int H, int W, int C, int KN, int KH, int KW,
                              float *dev_Y, void *workspace, size_t workspace_bytes, const tab::PatchPlan *plan, void *stream)
{
    if (type > 3) return fail(TAB_ERR_BAD_ARGUMENT, "type must be 0 (TNN), 1 (TBN), 2 (BTN) or 3 (BNN), got %d", type);
    ConvShape s;
    int rc = check_conv(type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, &s);
    if (rc != TAB_OK) return rc;
    rc = check_from_floats(s, type, dev_X, dev_QW, dev_btn, dev_Y, workspace, workspace_bytes, tab_layer_workspace_bytes(s.abits, N, H, W, C));
    if (rc != TAB_OK) return rc;
    char *sums = static_cast<char *>(workspace) + layer_packed_bytes(s.abits, N, H, W, C);
    const size_t need = tab_layer_workspace_bytes(s.abits, N, H, W, C);
    void *const spare = static_cast<char *>(workspace) + need;
    const size_t room = workspace_bytes - need;
    const bool planes = nchw && H * W > 1;  // one pixel per image: NCHW and NHWC are the same memory
    const bool own = s.abits == 2 && tab::conv_small_own_thresholds(dev_X, H, W, C, KH, KW, padding1, padding2);
    const int one = one_launch(type, dev_X, planes, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, s, own);
    if (planes && !one) {
        const ConvRoute route = conv_route(conv_args(s, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, workspace, dev_QW, dev_btn, dev_Y),
                                           type, plan, spare, room);
        rc = layer_quantize(dev_X, 1, s.abits, act_scale, N, H, W, C, static_cast<int64_t *>(workspace), sums,
                            need - layer_packed_bytes(s.abits, N, H, W, C), route.weights(), stream);
        if (rc != TAB_OK) return rc;
        return run_route(route, type, stream);
    }
    // small images of ternary activations, thresholds and quantizer in one launch; not where only the pixels at a stride are quantized
    if (!one && s.abits == 2 && !(KH == 1 && KW == 1 && (stride1 > 1 || stride2 > 1)) && tab::quantize_items_supported(true, false, N, (long)H * W, C)) {
        const ConvRoute route = conv_route(conv_args(s, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, workspace, dev_QW, dev_btn, dev_Y),
                                           type, plan, spare, room);
        if (!route.weights()) {
            rc = layer_quantize(dev_X, 0, s.abits, act_scale, N, H, W, C, static_cast<int64_t *>(workspace), sums,
                                need - layer_packed_bytes(s.abits, N, H, W, C), nullptr, stream);
            return rc != TAB_OK ? rc : run_route(route, type, stream);
        }
    }
    tab::Thresholds ths;
    hipError_t e = hipSuccess;
    if (one == 2 && own)
        ths = tab::Thresholds{dev_X, (double)act_scale / (double)C, tab::kOwnPixelThresholds, 0};
    else
        e = own_thresholds(dev_X, s.abits, act_scale, N, (long)H * W * C, sums, &ths, stream);
    if (e != hipSuccess) return device_fail(e, "threshold launch");
    if (ths.splits > 4 && one == 2 && !tab::conv_small_in_one_image(s.OH, s.OW)) {
        // this one-launch kernel looks thresholds up lane by lane: with many partial sums an item they are added first
        float *values = reinterpret_cast<float *>(sums + tab_threshold_workspace_bytes(N, (long)H * W * C));
        e = tab::launch_threshold_values(ths, N, values, static_cast<hipStream_t>(stream));
        if (e != hipSuccess) return device_fail(e, "threshold launch");
        ths = tab::given_thresholds(values);
    }
    if (planes) {
        e = tab::launch_conv_small(type, dev_X, true, ths, reinterpret_cast<const uint64_t *>(dev_QW), dev_btn, dev_Y, N, H, W, C, KN, KH, KW,
                                   padding1, padding2, stride1, stride2, s.OH, s.OW, static_cast<hipStream_t>(stream));
        if (e != hipSuccess) return device_fail(e, "conv launch");
        return TAB_OK;
    }
    return conv_from_nhwc(dev_X, dev_QW, ths, dev_btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, s, dev_Y,
                          workspace, plan, spare, room, stream);
}

int tab_layer_conv2d(const float *dev_X, int nchw, float act_scale, const int64_t *dev_QW, const int32_t *dev_btn, int type,
                     int padding1, int padding2, int stride1, int stride2, int N, int H, int W, int C, int KN, int KH, int KW,
                     float *dev_Y, void *workspace, size_t workspace_bytes, void *stream)
{
    return tab_internal_layer_conv2d(dev_X, nchw, act_scale, dev_QW, dev_btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW,
                                     dev_Y, workspace, workspace_bytes, nullptr, stream);
}

size_t tab_internal_conv_plan(int type, int padding1, int padding2, int stride1, int stride2, int N, int H, int W, int C, int KN, int KH, int KW,
                              tab::PatchPlan *plan)
{
    *plan = {-1, 0, 0, 0, -1, 0};
    ConvShape s;
    if (stride1 < 1 || stride2 < 1 ||
        !tab::conv_patch_considered(type, (long)N * tab_out_extent(H, padding1, KH, stride1) * tab_out_extent(W, padding2, KW, stride2), KN, KH, KW) ||
        check_conv(type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, &s) != TAB_OK)
        return 0;
    *plan = tab::conv_patch_plan(type, conv_sizes(s, padding1, padding2, stride1, stride2, N, H, W, KN, KH, KW));
    return plan->shape >= 0 ? plan->weight_bytes + 16 : 0;
}

int tab_internal_conv2d(const float *dev_X, const int64_t *dev_QW, const float *dev_ths, const int32_t *dev_btn, int type, int padding1,
                        int padding2, int stride1, int stride2, int N, int H, int W, int C, int KN, int KH, int KW, float *dev_Y,
                        void *workspace, size_t workspace_bytes, const tab::PatchPlan *plan, void *stream)
{
    return conv_from_floats(dev_X, dev_QW, dev_ths, dev_btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW,
                            dev_Y, workspace, workspace_bytes, false, plan, stream);
}

int tab_conv2d(const float *dev_X, const int64_t *dev_QW, const float *dev_ths,
               const int32_t *dev_btn, int type, int padding1, int padding2, int stride1,
               int stride2, int N, int H, int W, int C, int KN, int KH, int KW, float *dev_Y,
               void *workspace, size_t workspace_bytes, void *stream)
{
    return conv_from_floats(dev_X, dev_QW, dev_ths, dev_btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW,
                            dev_Y, workspace, workspace_bytes, false, nullptr, stream);
}

int tab_conv2d_launches(const float *dev_X, int type, int padding1, int padding2, int stride1, int stride2, int N, int H, int W,
                        int C, int KN, int KH, int KW)
{
    ConvShape s;
    if (check_conv(type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, &s) != TAB_OK) return 0;
    return one_launch(type, dev_X, false, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, s) ? 1 : 2;
}

size_t tab_static_scratch_bytes(void) { return TAB_STATIC_SCRATCH_BYTES; }

int tab_conv2d_static(const float *dev_X, const int64_t *dev_QW, const float *dev_ths, const int32_t *dev_btn, int type,
                      int padding1, int padding2, int stride1, int stride2, int N, int H, int W, int C, int KN, int KH, int KW,
                      float *dev_Y, void *stream)
{
    return conv_from_floats(dev_X, dev_QW, dev_ths, dev_btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW,
                            dev_Y, nullptr, 0, true, nullptr, stream);
}

}  // extern "C"
