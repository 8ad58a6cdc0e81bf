// PyTorch C++ extension front end: the reference's operator boundary (TAB_GPU.cpp:34-65) on
// top of the C ABI of include/tab_amd.h.  Same exported names (`Quantize`, `Conv2d`), same
// positional parameter lists, same return tensors; the CPU module's names (TAB_CPU.cpp:636-639)
// are exported as aliases.  PyTorch only supplies device memory (caching allocator) and the
// current HIP stream; all compute is in libtab_amd.so.
#include <torch/extension.h>

#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/hip/HIPCachingAllocator.h>

#include <array>
#include <memory>
#include <stdexcept>
#include <tuple>
#include <vector>

#include "../../include/tab_amd.h"
#include "tab_route.h"

// CHECK_INPUT of the reference (TAB_GPU.cpp:7-9)
#define CHECK_CUDA(x) TORCH_CHECK(x.device().is_cuda(), #x " must be a CUDA tensor")
#define CHECK_CONTIGUOUS(x) TORCH_CHECK(x.is_contiguous(), #x " must be contiguous")
#define CHECK_INPUT(x) \
    CHECK_CUDA(x);     \
    CHECK_CONTIGUOUS(x)
// The reference converts dtypes with .toType() on a temporary (TAB_GEMM.cu:279-280,341-347),
// which dangles whenever a conversion really happens; exact dtypes are required instead.
#define CHECK_DTYPE(x, t) \
    TORCH_CHECK(x.scalar_type() == torch::t, #x " must have dtype ", dtype_name(torch::t), ", got ", dtype_name(x.scalar_type()))

namespace {

std::string dtype_name(torch::ScalarType t)
{
    switch (t) {
    case torch::kFloat32: return "torch.float32";
    case torch::kInt64: return "torch.int64";
    case torch::kInt32: return "torch.int32";
    default: return std::string("torch.") + c10::toString(t);
    }
}

// A negative status of a C ABI call; Python sees tab_amd.TabError (a RuntimeError).
struct StatusError : std::runtime_error {
    using std::runtime_error::runtime_error;
};

void check_status(int status)
{
    if (status != TAB_OK) throw StatusError(std::string(tab_status_string(status)) + ": " + tab_last_error());
}

hipStream_t current_stream(const torch::Tensor &t)
{
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

// Uninitialised device tensor, straight from the caching allocator: torch::empty's way through the dispatcher costs
// 0.73 us a tensor, this 0.47, beside 2.3 us for a kernel launch.
torch::Tensor device_empty(c10::IntArrayRef sizes, torch::ScalarType dtype, const torch::Tensor &like)
{
    return at::detail::empty_cuda(sizes, dtype, like.device(), c10::nullopt);
}

// Device scratch of one call (0.2 us, no tensor around it).  Given back when the call returns: the allocator hands the
// block only to later work of the same stream.
class Workspace {
public:
    Workspace(size_t bytes, hipStream_t stream)
        : ptr_(c10::hip::HIPCachingAllocator::raw_alloc_with_stream(bytes, stream)) {}
    ~Workspace() { c10::hip::HIPCachingAllocator::raw_delete(ptr_); }
    Workspace(const Workspace &) = delete;
    Workspace &operator=(const Workspace &) = delete;
    void *get() const { return ptr_; }

private:
    void *ptr_;
};

void quantize_counted(const torch::Tensor &X, const torch::Tensor &thresholds, bool nchw, int bitwidth, int N, int H, int W, int C,
                      const torch::Tensor &QX, const torch::Tensor &BTN)
{
    const hipStream_t stream = current_stream(X);
    const size_t bytes = tab_quantize_workspace_bytes(bitwidth, N, H, W, C);
    auto call = [&](void *workspace) {
        check_status(tab_quantize_counted(X.data_ptr<float>(), thresholds.data_ptr<float>(), nchw, bitwidth, N, H, W, C, QX.data_ptr<int64_t>(),
                                          BTN.data_ptr<int32_t>(), workspace, bytes, stream));
    };
    if (bytes) call(Workspace(bytes, stream).get());
    else call(nullptr);
}

}  // namespace

std::vector<torch::Tensor> TAB_Quantize(const torch::Tensor &X, const torch::Tensor &thresholds, int bitwidth, int N,
                                        int H, int W, int C)
{
    CHECK_INPUT(X);
    CHECK_INPUT(thresholds);
    CHECK_DTYPE(X, kFloat32);
    CHECK_DTYPE(thresholds, kFloat32);
    TORCH_CHECK(bitwidth == 1 || bitwidth == 2, "bitwidth must be 1 or 2, got ", bitwidth);
    TORCH_CHECK(N > 0 && H > 0 && W > 0 && C > 0, "N, H, W, C must be positive");
    TORCH_CHECK(X.numel() == (int64_t)N * H * W * C, "X has ", X.numel(), " elements, expected N*H*W*C = ",
                (int64_t)N * H * W * C);
    TORCH_CHECK(thresholds.numel() >= N, "thresholds has ", thresholds.numel(), " elements, expected at least N = ", N);
    TORCH_CHECK(thresholds.device() == X.device(), "X and thresholds must be on the same device");
    const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(X.device());
    const int PC = tab_packed_channels(C);
    auto QX = device_empty({N, H, W, PC, bitwidth}, torch::kInt64, X);
    auto BTN = device_empty({N}, torch::kInt32, X);
    quantize_counted(X, thresholds, false, bitwidth, N, H, W, C, QX, BTN);
    return {QX, BTN};
}

namespace {

// Checks shared by the conv entry points; returns (OH, OW).
std::pair<int, int> check_conv(const torch::Tensor &QW, const torch::Tensor &btn, int type, int padding1, int padding2,
                               int stride1, int stride2, int N, int H, int W, int C, int KN, int KH, int KW)
{
    // types 4 (DoReFa 2-bit) and 5 (RTN) are the further cases of the CPU binding's TAB_Conv2d (TAB_CPU.cpp:577-584, 621-633)
    TORCH_CHECK(type >= 0 && type <= 5, "type must be 0 (TNN), 1 (TBN), 2 (BTN), 3 (BNN), 4 (DRF) or 5 (RTN), got ", type);
    TORCH_CHECK(N > 0 && H > 0 && W > 0 && C > 0 && KN > 0 && KH > 0 && KW > 0 && padding1 >= 0 && padding2 >= 0 &&
                    stride1 > 0 && stride2 > 0,
                "sizes must be positive, padding >= 0 and stride >= 1");
    const int wwords = tab_operand_words(type, 1, C);
    TORCH_CHECK(QW.numel() == (int64_t)KN * KH * KW * wwords, "QW has ", QW.numel(), " words, type ", type,
                " expects KN*KH*KW*", wwords, " = ", (int64_t)KN * KH * KW * wwords);
    TORCH_CHECK(type != TAB_BTN || btn.numel() >= KN, "btn has ", btn.numel(), " elements, expected at least KN = ", KN);
    const int OH = tab_out_extent(H, padding1, KH, stride1), OW = tab_out_extent(W, padding2, KW, stride2);
    TORCH_CHECK(OH > 0 && OW > 0, "empty output: OH=", OH, ", OW=", OW);
    return {OH, OW};
}

}  // namespace

namespace {

// Checks of the calls that take the fp32 activation; returns (OH, OW).
std::pair<int, int> check_conv_from_floats(const torch::Tensor &X, const torch::Tensor &QW, const torch::Tensor &thresholds,
                                           const torch::Tensor &btn, int type, int padding1, int padding2, int stride1, int stride2,
                                           int N, int H, int W, int C, int KN, int KH, int KW)
{
    CHECK_INPUT(X);
    CHECK_INPUT(QW);
    CHECK_INPUT(thresholds);
    CHECK_INPUT(btn);
    CHECK_DTYPE(X, kFloat32);
    CHECK_DTYPE(QW, kInt64);
    CHECK_DTYPE(thresholds, kFloat32);
    CHECK_DTYPE(btn, kInt32);
    const auto out = check_conv(QW, btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW);
    TORCH_CHECK(X.numel() == (int64_t)N * H * W * C, "X has ", X.numel(), " elements, expected N*H*W*C = ",
                (int64_t)N * H * W * C);
    TORCH_CHECK(thresholds.numel() >= N, "thresholds has ", thresholds.numel(), " elements, expected at least N = ", N);
    TORCH_CHECK(QW.device() == X.device() && thresholds.device() == X.device() && btn.device() == X.device(),
                "X, QW, thresholds and btn must be on the same device");
    return out;
}

}  // namespace

torch::Tensor TAB_Conv2d(const torch::Tensor &X, const torch::Tensor &QW, const torch::Tensor &thresholds, const torch::Tensor &btn,
                         int type, int padding1, int padding2, int stride1, int stride2, int N, int H, int W, int C, int KN,
                         int KH, int KW)
{
    const auto [OH, OW] = check_conv_from_floats(X, QW, thresholds, btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW);
    const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(X.device());
    auto Y = device_empty({N, KN, OH, OW}, torch::kFloat32, X);
    tab::PatchPlan plan;
    const size_t ws_bytes = tab_conv2d_workspace_bytes(type, N, H, W, C) +
                            tab_internal_conv_plan(type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, &plan);
    const hipStream_t stream = current_stream(X);
    const Workspace ws(ws_bytes, stream);
    check_status(tab_internal_conv2d(X.data_ptr<float>(), QW.data_ptr<int64_t>(), thresholds.data_ptr<float>(),
                                     btn.data_ptr<int32_t>(), type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH,
                                     KW, Y.data_ptr<float>(), ws.get(), ws_bytes, &plan, stream));
    return Y;
}

// ---- the entry points beyond the reference's two: same conventions, one C ABI call each -----------------------

// Quantize on an NCHW tensor, the layout and argument order of the reference's CPU binding (TAB_CPU.cpp:20-206, 621).
std::vector<torch::Tensor> TAB_QuantizeNCHW(const torch::Tensor &X, const torch::Tensor &thresholds, int bitwidth, int N, int C,
                                            int H, int W)
{
    CHECK_INPUT(X);
    CHECK_INPUT(thresholds);
    CHECK_DTYPE(X, kFloat32);
    CHECK_DTYPE(thresholds, kFloat32);
    TORCH_CHECK(bitwidth == 1 || bitwidth == 2, "bitwidth must be 1 or 2, got ", bitwidth);
    TORCH_CHECK(N > 0 && H > 0 && W > 0 && C > 0, "N, C, H, W must be positive");
    TORCH_CHECK(X.numel() == (int64_t)N * H * W * C, "X has ", X.numel(), " elements, expected N*C*H*W = ",
                (int64_t)N * H * W * C);
    TORCH_CHECK(thresholds.numel() >= N, "thresholds has ", thresholds.numel(), " elements, expected at least N = ", N);
    TORCH_CHECK(thresholds.device() == X.device(), "X and thresholds must be on the same device");
    const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(X.device());
    auto QX = device_empty({N, H, W, tab_packed_channels(C), bitwidth}, torch::kInt64, X);
    auto BTN = device_empty({N}, torch::kInt32, X);
    quantize_counted(X, thresholds, true, bitwidth, N, H, W, C, QX, BTN);
    return {QX, BTN};
}

// The packed activation alone, NHWC or NCHW: without the BTN vector, which nobody reads of an activation.
torch::Tensor TAB_QuantizeActivation(const torch::Tensor &X, const torch::Tensor &thresholds, int bitwidth, int N, int H, int W,
                                     int C, bool nchw)
{
    CHECK_INPUT(X);
    CHECK_INPUT(thresholds);
    CHECK_DTYPE(X, kFloat32);
    CHECK_DTYPE(thresholds, kFloat32);
    TORCH_CHECK(bitwidth == 1 || bitwidth == 2, "bitwidth must be 1 or 2, got ", bitwidth);
    TORCH_CHECK(N > 0 && H > 0 && W > 0 && C > 0, "N, H, W, C must be positive");
    TORCH_CHECK(X.numel() == (int64_t)N * H * W * C, "X has ", X.numel(), " elements, expected N*H*W*C = ",
                (int64_t)N * H * W * C);
    TORCH_CHECK(thresholds.numel() >= N, "thresholds has ", thresholds.numel(), " elements, expected at least N = ", N);
    TORCH_CHECK(thresholds.device() == X.device(), "X and thresholds must be on the same device");
    const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(X.device());
    auto QX = device_empty({N, H, W, tab_packed_channels(C), bitwidth}, torch::kInt64, X);
    const float *x = X.data_ptr<float>(), *ths = thresholds.data_ptr<float>();
    int64_t *q = QX.data_ptr<int64_t>();
    check_status(nchw ? tab_quantize_nchw(x, ths, bitwidth, N, C, H, W, q, nullptr, current_stream(X))
                      : tab_quantize(x, ths, bitwidth, N, H, W, C, q, nullptr, current_stream(X)));
    return QX;
}

// Packer of conv types 4 and 5 (layouts of DRFGEMM_baseline / RTNGEMM_baseline, TAB_CPU.cpp:332-383).
torch::Tensor TAB_QuantizeFormat(const torch::Tensor &X, const torch::Tensor &thresholds, int type, int N, int H, int W, int C)
{
    CHECK_INPUT(X);
    CHECK_INPUT(thresholds);
    CHECK_DTYPE(X, kFloat32);
    CHECK_DTYPE(thresholds, kFloat32);
    TORCH_CHECK(type == TAB_DRF || type == TAB_RTN, "type must be 4 (DRF) or 5 (RTN), got ", type);
    TORCH_CHECK(N > 0 && H > 0 && W > 0 && C > 0, "N, H, W, C must be positive");
    TORCH_CHECK(X.numel() == (int64_t)N * H * W * C, "X has ", X.numel(), " elements, expected N*H*W*C = ",
                (int64_t)N * H * W * C);
    TORCH_CHECK(thresholds.numel() >= N, "thresholds has ", thresholds.numel(), " elements, expected at least N = ", N);
    TORCH_CHECK(thresholds.device() == X.device(), "X and thresholds must be on the same device");
    const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(X.device());
    auto QX = type == TAB_DRF ? device_empty({N, H, W, tab_packed_channels(C), 2}, torch::kInt64, X)
                              : device_empty({N, H, W, (C + 31) / 32}, torch::kInt64, X);
    check_status(tab_quantize_format(X.data_ptr<float>(), thresholds.data_ptr<float>(), type, N, H, W, C,
                                     QX.data_ptr<int64_t>(), current_stream(X)));
    return QX;
}

// thresholds[n] = scale * mean|X[n]|, the rule README.md:45 leaves to the caller.
torch::Tensor TAB_Threshold(const torch::Tensor &X, int N, double scale)
{
    CHECK_INPUT(X);
    CHECK_DTYPE(X, kFloat32);
    TORCH_CHECK(N > 0 && X.numel() > 0 && X.numel() % N == 0, "X has ", X.numel(), " elements, not a positive multiple of N = ", N);
    const long per_item = (long)(X.numel() / N);
    const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(X.device());
    auto ths = device_empty({N}, torch::kFloat32, X);
    const size_t ws_bytes = tab_threshold_workspace_bytes(N, per_item);
    const hipStream_t stream = current_stream(X);
    const Workspace ws(ws_bytes, stream);
    check_status(tab_threshold(X.data_ptr<float>(), N, per_item, (float)scale, ths.data_ptr<float>(), ws.get(), ws_bytes, stream));
    return ths;
}

// Conv2d with the packed activation in the library's built-in scratch; with `out` given nothing is allocated.
torch::Tensor TAB_Conv2dStatic(const torch::Tensor &X, const torch::Tensor &QW, const torch::Tensor &thresholds,
                               const torch::Tensor &btn, int type, int padding1, int padding2, int stride1, int stride2, int N,
                               int H, int W, int C, int KN, int KH, int KW, const c10::optional<torch::Tensor> &given)
{
    const auto [OH, OW] = check_conv_from_floats(X, QW, thresholds, btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW);
    const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(X.device());
    const torch::Tensor out = given ? *given : device_empty({N, KN, OH, OW}, torch::kFloat32, X);
    CHECK_INPUT(out);
    CHECK_DTYPE(out, kFloat32);
    TORCH_CHECK(out.numel() == (int64_t)N * KN * OH * OW, "out has ", out.numel(), " elements, expected ", (int64_t)N * KN * OH * OW);
    check_status(tab_conv2d_static(X.data_ptr<float>(), QW.data_ptr<int64_t>(), thresholds.data_ptr<float>(), btn.data_ptr<int32_t>(),
                                   type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, out.data_ptr<float>(),
                                   current_stream(X)));
    return out;
}

// Conv2d on an activation already packed by Quantize / QuantizeFormat (TAB_GEMM.cu:447-509 only).
torch::Tensor TAB_Conv2dPacked(const torch::Tensor &QX, const torch::Tensor &QW, const torch::Tensor &btn, int type, int padding1, int padding2,
                               int stride1, int stride2, int N, int H, int W, int C, int KN, int KH, int KW)
{
    CHECK_INPUT(QX);
    CHECK_INPUT(QW);
    CHECK_INPUT(btn);
    CHECK_DTYPE(QX, kInt64);
    CHECK_DTYPE(QW, kInt64);
    CHECK_DTYPE(btn, kInt32);
    const auto [OH, OW] = check_conv(QW, btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW);
    const int awords = tab_operand_words(type, 0, C);
    TORCH_CHECK(QX.numel() == (int64_t)N * H * W * awords, "QX has ", QX.numel(), " words, type ", type, " expects N*H*W*", awords);
    TORCH_CHECK(QW.device() == QX.device() && btn.device() == QX.device(), "QX, QW and btn must be on the same device");
    const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(QX.device());
    auto Y = device_empty({N, KN, OH, OW}, torch::kFloat32, QX);
    check_status(tab_conv2d_packed(QX.data_ptr<int64_t>(), QW.data_ptr<int64_t>(), btn.data_ptr<int32_t>(), type, padding1,
                                   padding2, stride1, stride2, N, H, W, C, KN, KH, KW, Y.data_ptr<float>(), current_stream(QX)));
    return Y;
}

// Conv2dPacked with the output thresholded and packed in the epilogue: the next layer's activation, no fp32 Y.
torch::Tensor TAB_Conv2dPackedOut(const torch::Tensor &QX, const torch::Tensor &QW, const torch::Tensor &btn, int type, int padding1, int padding2,
                                  int stride1, int stride2, int N, int H, int W, int C, int KN, int KH, int KW,
                                  const torch::Tensor &out_thresholds, int out_bitwidth)
{
    CHECK_INPUT(QX);
    CHECK_INPUT(QW);
    CHECK_INPUT(btn);
    CHECK_INPUT(out_thresholds);
    CHECK_DTYPE(QX, kInt64);
    CHECK_DTYPE(QW, kInt64);
    CHECK_DTYPE(btn, kInt32);
    CHECK_DTYPE(out_thresholds, kFloat32);
    TORCH_CHECK(out_bitwidth == 1 || out_bitwidth == 2, "out_bitwidth must be 1 or 2, got ", out_bitwidth);
    const auto [OH, OW] = check_conv(QW, btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW);
    const int awords = tab_operand_words(type, 0, C);
    TORCH_CHECK(QX.numel() == (int64_t)N * H * W * awords, "QX has ", QX.numel(), " words, type ", type, " expects N*H*W*", awords);
    TORCH_CHECK(out_thresholds.numel() >= N, "out_thresholds has ", out_thresholds.numel(), " elements, need N = ", N);
    TORCH_CHECK(QW.device() == QX.device() && btn.device() == QX.device() && out_thresholds.device() == QX.device(),
                "QX, QW, btn and out_thresholds must be on the same device");
    const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(QX.device());
    auto QY = device_empty({N, OH, OW, tab_packed_channels(KN), out_bitwidth}, torch::kInt64, QX);
    check_status(tab_conv2d_packed_out(QX.data_ptr<int64_t>(), QW.data_ptr<int64_t>(), btn.data_ptr<int32_t>(), type, padding1,
                                       padding2, stride1, stride2, N, H, W, C, KN, KH, KW, out_thresholds.data_ptr<float>(),
                                       out_bitwidth, QY.data_ptr<int64_t>(), current_stream(QX)));
    return QY;
}

// ---- the layers of tab_amd/nn.py: a forward pass is one call from Python ---------------------------------------------
// Attribute reads, buffer look-ups, a module call, views, an array of zeros and a Python call per operator made some 10 us
// of host work a layer around kernels of 6-30 us; here the module's attributes are read from its dictionaries (30 ns each).

namespace {

namespace py = pybind11;

// module.<name>, from the module's own dictionary where it is there (nn.Module attributes that are no submodules, parameters
// or buffers are)
py::object attribute(py::handle module, py::handle name)
{
    PyObject **dict = _PyObject_GetDictPtr(module.ptr());
    if (dict != nullptr && *dict != nullptr) {
        PyObject *item = PyDict_GetItemWithError(*dict, name.ptr());
        if (item != nullptr) return py::reinterpret_borrow<py::object>(item);
        if (PyErr_Occurred()) throw py::error_already_set();
    }
    return py::reinterpret_steal<py::object>(PyObject_GetAttr(module.ptr(), name.ptr()));
}

PyObject *interned(const char *name) { return PyUnicode_InternFromString(name); }

// The item of a dictionary attribute (_buffers, _modules) or, where it is not there, the attribute itself.
py::object item_or_attribute(py::handle module, py::handle dict_name, py::handle name)
{
    const py::object dict = attribute(module, dict_name);
    PyObject *item = PyDict_Check(dict.ptr()) ? PyDict_GetItemWithError(dict.ptr(), name.ptr()) : nullptr;
    if (item != nullptr) return py::reinterpret_borrow<py::object>(item);
    if (PyErr_Occurred()) throw py::error_already_set();
    return py::reinterpret_steal<py::object>(PyObject_GetAttr(module.ptr(), name.ptr()));
}

torch::Tensor buffer(py::handle module, py::handle name)
{
    static PyObject *const buffers_name = interned("_buffers");
    return item_or_attribute(module, buffers_name, name).cast<torch::Tensor>();
}

int as_int(PyObject *v)
{
    if (PyLong_CheckExact(v)) {
        const long value = PyLong_AsLong(v);
        if (value == (int)value && !(value == -1 && PyErr_Occurred())) return (int)value;
        PyErr_Clear();
    }
    return py::handle(v).cast<int>();
}

int integer(py::handle module, py::handle name) { return as_int(attribute(module, name).ptr()); }

std::pair<int, int> pair_of(py::handle module, py::handle name)
{
    const py::object v = attribute(module, name);
    if (PyTuple_CheckExact(v.ptr()) && PyTuple_GET_SIZE(v.ptr()) == 2)
        return {as_int(PyTuple_GET_ITEM(v.ptr(), 0)), as_int(PyTuple_GET_ITEM(v.ptr(), 1))};
    return {v[py::int_(0)].cast<int>(), v[py::int_(1)].cast<int>()};
}

// What a TABConv2d module holds.
struct Layer {
    torch::Tensor QW, btn;
    int type, C, KN, KH, KW, s1, s2, p1, p2;
    double act_scale;

    explicit Layer(py::handle m)
    {
        static PyObject *const n_qw = interned("QW"), *const n_btn = interned("BTN_W"), *const n_type = interned("conv_type"),
                               *const n_in = interned("in_channels"), *const n_out = interned("out_channels"),
                               *const n_kernel = interned("kernel_size"), *const n_stride = interned("stride"),
                               *const n_padding = interned("padding"), *const n_scale = interned("act_scale");
        QW = buffer(m, n_qw);
        btn = buffer(m, n_btn);
        type = integer(m, n_type);
        C = integer(m, n_in);
        KN = integer(m, n_out);
        std::tie(KH, KW) = pair_of(m, n_kernel);
        std::tie(s1, s2) = pair_of(m, n_stride);
        std::tie(p1, p2) = pair_of(m, n_padding);
        act_scale = attribute(m, n_scale).cast<double>();
        // (act_bits and with it the size of a packed activation hold for these types only)
        TORCH_CHECK(type >= 0 && type <= 3, "conv_type must be 0 (TNN), 1 (TBN), 2 (BTN) or 3 (BNN), got ", type);
    }

    int act_bits() const { return type < 2 ? 2 : 1; }

    // checks against an activation of N images of H x W on X's device; returns (OH, OW)
    std::pair<int, int> check(const torch::Tensor &X, int N, int H, int W) const
    {
        CHECK_INPUT(QW);
        CHECK_INPUT(btn);
        CHECK_DTYPE(QW, kInt64);
        CHECK_DTYPE(btn, kInt32);
        TORCH_CHECK(QW.device() == X.device() && btn.device() == X.device(), "X, QW and btn must be on the same device");
        return check_conv(QW, btn, type, p1, p2, s1, s2, N, H, W, C, KN, KH, KW);
    }
};

// The input as contiguous fp32, what the kernels take.
torch::Tensor plain_input(const torch::Tensor &x)
{
    const torch::Tensor X = x.scalar_type() == torch::kFloat32 ? (x.is_contiguous() ? x : x.contiguous()) : x.to(torch::kFloat32).contiguous();
    CHECK_CUDA(X);
    return X;
}

// (N, H, W, C) of a four-dimensional activation; C checked against the layer's.
std::array<int, 4> activation_sizes(const torch::Tensor &x, bool nchw, int channels)
{
    if (x.dim() != 4) throw py::value_error("expected an activation of four dimensions, got " + std::to_string(x.dim()));
    const std::array<int, 4> s = nchw ? std::array<int, 4>{(int)x.size(0), (int)x.size(2), (int)x.size(3), (int)x.size(1)}
                                      : std::array<int, 4>{(int)x.size(0), (int)x.size(1), (int)x.size(2), (int)x.size(3)};
    TORCH_CHECK(s[3] == channels, "expected ", channels, " input channels, got ", s[3]);
    return s;
}

// A layer's fp32 output: memory (n, oh, ow, kn) (TAB_GEMM.cu:526), shaped NHWC or, as a strided tensor, NCHW.
torch::Tensor layer_output(const torch::Tensor &X, bool nchw, int64_t N, int64_t OH, int64_t OW, int64_t KN)
{
    if (!nchw) return device_empty({N, OH, OW, KN}, torch::kFloat32, X);
    return at::detail::empty_strided_cuda({N, KN, OH, OW}, {OH * OW * KN, 1, OW * KN, KN}, torch::kFloat32, X.device());
}

void run_layer(const Layer &l, const torch::Tensor &X, bool nchw, int N, int H, int W, const torch::Tensor &y)
{
    const hipStream_t stream = current_stream(X);
    tab::PatchPlan plan;
    const size_t ws_bytes = tab_layer_workspace_bytes(l.act_bits(), N, H, W, l.C) +
                            tab_internal_conv_plan(l.type, l.p1, l.p2, l.s1, l.s2, N, H, W, l.C, l.KN, l.KH, l.KW, &plan);
    const Workspace ws(ws_bytes, stream);
    check_status(tab_internal_layer_conv2d(X.data_ptr<float>(), nchw, (float)l.act_scale, l.QW.data_ptr<int64_t>(), l.btn.data_ptr<int32_t>(),
                                           l.type, l.p1, l.p2, l.s1, l.s2, N, H, W, l.C, l.KN, l.KH, l.KW, y.data_ptr<float>(), ws.get(),
                                           ws_bytes, &plan, stream));
}

// TABConv2d.forward
torch::Tensor layer_forward(py::handle module, const torch::Tensor &x, bool nchw)
{
    const Layer l(module);
    const auto [N, H, W, C] = activation_sizes(x, nchw, l.C);
    const torch::Tensor X = plain_input(x);
    const auto [OH, OW] = l.check(X, N, H, W);
    const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(X.device());
    const torch::Tensor y = layer_output(X, nchw, N, OH, OW, l.KN);
    run_layer(l, X, nchw, N, H, W, y);
    return y;
}

// The class of module a one-call path may stand in for: its methods as they were when the class was made, and the
// dictionaries of the hooks of every module.
struct PlainClass {
    py::object type, forward, call;
    std::vector<py::object> global_hooks;

    explicit PlainClass(py::object t) : type(t), forward(t.attr("forward")), call(t.attr("__call__"))
    {
        const py::module_ m = py::module_::import("torch.nn.modules.module");
        for (const char *name : {"_global_forward_hooks", "_global_forward_pre_hooks", "_global_backward_hooks", "_global_backward_pre_hooks"})
            global_hooks.push_back(m.attr(name));
    }
};

// Whether calling the module would run more than its forward: another class's or a replaced method, a forward of the
// module's own, hooks of its own or of every module, a compiled call (Module.compile).
bool plain_call(py::handle module, const PlainClass &plain)
{
    static PyObject *const hooks[] = {interned("_forward_hooks"), interned("_forward_pre_hooks"), interned("_backward_hooks"),
                                      interned("_backward_pre_hooks")};
    static PyObject *const forward_name = interned("forward"), *const call_name = interned("__call__"),
                           *const compiled_name = interned("_compiled_call_impl");
    PyTypeObject *const type = Py_TYPE(module.ptr());
    if ((PyObject *)type != plain.type.ptr() || _PyType_Lookup(type, forward_name) != plain.forward.ptr() ||
        _PyType_Lookup(type, call_name) != plain.call.ptr())
        return false;
    for (PyObject *name : hooks) {
        const py::object d = attribute(module, name);
        if (!PyDict_Check(d.ptr()) || PyDict_GET_SIZE(d.ptr()) != 0) return false;
    }
    for (const py::object &d : plain.global_hooks)
        if (!PyDict_Check(d.ptr()) || PyDict_GET_SIZE(d.ptr()) != 0) return false;
    // (the compiled call and a forward of its own are in the module's dictionary; nn.Module's getattr took 0.06 us to say so)
    PyObject **dict = _PyObject_GetDictPtr(module.ptr());
    if (dict == nullptr || *dict == nullptr) return false;
    PyObject *const compiled = PyDict_GetItemWithError(*dict, compiled_name);
    if (PyErr_Occurred()) throw py::error_already_set();
    return (compiled == nullptr || compiled == Py_None) && PyDict_Contains(*dict, forward_name) == 0;
}

// TABLinear.forward around its TABConv2d (`plain`: that class): (N, F) as N images of one pixel.  None where calling the
// convolution module is more than its forward, it takes another layout, or the input is no tensor (a tracer's proxy): the
// caller then calls it.
py::object linear_forward(py::handle module, const py::capsule &plain, py::handle input)
{
    if (!THPVariable_Check(input.ptr())) return py::none();
    const torch::Tensor &x = THPVariable_Unpack(input.ptr());
    static PyObject *const modules_name = interned("_modules"), *const conv_name = interned("conv"), *const format_name = interned("data_format");
    const py::object conv = item_or_attribute(module, modules_name, conv_name);
    if (!plain_call(conv, *plain.get_pointer<PlainClass>())) return py::none();
    const py::object format = attribute(conv, format_name);
    if (!PyUnicode_Check(format.ptr()) || PyUnicode_CompareWithASCIIString(format.ptr(), "NHWC") != 0) return py::none();
    const Layer l(conv);
    if (x.dim() != 2) throw py::value_error("expected an input of two dimensions, got " + std::to_string(x.dim()));
    const int N = (int)x.size(0);
    TORCH_CHECK(x.size(1) == l.C, "expected ", l.C, " input channels, got ", x.size(1));
    const torch::Tensor X = plain_input(x);
    const auto [OH, OW] = l.check(X, N, 1, 1);
    TORCH_CHECK(OH == 1 && OW == 1, "a linear layer's convolution maps one pixel to one pixel, got ", OH, " x ", OW);
    const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(X.device());
    const torch::Tensor y = device_empty({N, l.KN}, torch::kFloat32, X);
    run_layer(l, X, false, N, 1, 1, y);
    return py::cast(y);
}

// TABPackedChain.forward: packed activations between the layers, in raw blocks of the caching allocator
torch::Tensor chain_forward(const py::list &modules, const py::dict &ternary_thresholds, bool nchw, const torch::Tensor &x)
{
    std::vector<Layer> layers;
    layers.reserve(modules.size());
    for (const py::handle m : modules) layers.emplace_back(m);
    // The module's constructor checks this too, but its list of layers can change afterwards, and the packed activations
    // between them are raw blocks: no tensor's size would say that the next layer reads more than this one wrote.
    if (layers.empty()) throw py::index_error("the chain has no layers");
    for (size_t i = 1; i < layers.size(); i++)
        TORCH_CHECK(layers[i - 1].KN == layers[i].C, layers[i - 1].KN, " output channels feed a layer with ", layers[i].C, " input channels");
    const Layer &first = layers.front();
    auto [N, H, W, C] = activation_sizes(x, nchw, first.C);
    const torch::Tensor X = plain_input(x);
    const c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard(X.device());
    const hipStream_t stream = current_stream(X);
    const auto packed_bytes = [N = N](int H, int W, int C, int bits) { return (size_t)N * H * W * tab_packed_channels(C) * bits * 8; };

    first.check(X, N, H, W);
    const size_t ws_bytes = first.act_bits() == 2 ? tab_threshold_workspace_bytes(N, (long)H * W * C) : 4;
    auto q = std::make_unique<Workspace>(packed_bytes(H, W, C, first.act_bits()), stream);
    {
        const Workspace ws(ws_bytes, stream);
        check_status(tab_layer_quantize(X.data_ptr<float>(), nchw, first.act_bits(), (float)first.act_scale, N, H, W, C,
                                        static_cast<int64_t *>(q->get()), ws.get(), ws_bytes, stream));
    }
    for (size_t i = 0;; i++) {
        const Layer &l = layers[i];
        const auto [OH, OW] = l.check(X, N, H, W);
        const int64_t *in = static_cast<const int64_t *>(q->get());
        if (i + 1 == layers.size()) {
            const torch::Tensor y = layer_output(X, nchw, N, OH, OW, l.KN);
            check_status(tab_conv2d_packed(in, l.QW.data_ptr<int64_t>(), l.btn.data_ptr<int32_t>(), l.type, l.p1, l.p2, l.s1, l.s2, N, H,
                                           W, l.C, l.KN, l.KH, l.KW, y.data_ptr<float>(), stream));
            return y;
        }
        const py::int_ key(i + 1);
        const float th = ternary_thresholds.contains(key) ? (float)(double)py::float_(py::object(ternary_thresholds[key])) : 0.f;
        const int bits = layers[i + 1].act_bits();
        auto out = std::make_unique<Workspace>(packed_bytes(OH, OW, l.KN, bits), stream);
        check_status(tab_conv2d_packed_out_const(in, l.QW.data_ptr<int64_t>(), l.btn.data_ptr<int32_t>(), l.type, l.p1, l.p2, l.s1, l.s2,
                                                 N, H, W, l.C, l.KN, l.KH, l.KW, th, bits, static_cast<int64_t *>(out->get()), stream));
        q = std::move(out);
        H = OH;
        W = OW;
    }
}

}  // namespace

namespace {

// The operators that a program calls in its inner loop, taken as arrays of arguments: pybind11's dispatch of sixteen arguments costs 0.42 us,
// this 0.09, of the 4.7 us a call of one launch takes the host.  Anything but tensors and plain ints in their places goes through the pybind11
// function of the same name, so that conversions and their errors are its own.  An operator is entered once: what it throws after it may have
// launched or allocated reaches the caller, translated as pybind11 would.
template <size_t TENSORS, size_t INTS>
bool plain_arguments(PyObject *const *args, Py_ssize_t count, const torch::Tensor *(&tensors)[TENSORS], int (&ints)[INTS])
{
    if (count != (Py_ssize_t)(TENSORS + INTS)) return false;
    for (size_t i = 0; i < TENSORS; i++) {
        if (!THPVariable_Check(args[i])) return false;
        tensors[i] = &THPVariable_Unpack(args[i]);
    }
    for (size_t i = 0; i < INTS; i++) {
        PyObject *const v = args[TENSORS + i];
        if (!PyLong_CheckExact(v)) return false;
        int overflow = 0;
        const long value = PyLong_AsLongAndOverflow(v, &overflow);
        if (overflow != 0 || value != (int)value) return false;
        ints[i] = (int)value;
    }
    return true;
}

PyObject *wrapped(torch::Tensor &&y) { return THPVariable_Wrap(std::move(y)); }
PyObject *wrapped(std::vector<torch::Tensor> &&ys)
{
    PyObject *const list = PyList_New((Py_ssize_t)ys.size());
    for (size_t i = 0; list != nullptr && i < ys.size(); i++) {
        PyObject *const item = THPVariable_Wrap(std::move(ys[i]));
        if (item == nullptr) {
            Py_DECREF(list);
            return nullptr;
        }
        PyList_SET_ITEM(list, (Py_ssize_t)i, item);
    }
    return list;
}

// The pybind11 function of an operator under one of its names, looked up when the module is made (and kept as long as the process).
template <auto OPERATOR, int ALIAS> PyObject *general = nullptr;

template <auto OPERATOR, size_t... T, size_t... I>
auto call_plain(const torch::Tensor *const *tensors, const int *ints, std::index_sequence<T...>, std::index_sequence<I...>)
{
    return OPERATOR(*tensors[T]..., ints[I]...);
}

template <auto OPERATOR, size_t TENSORS, size_t INTS, int ALIAS>
PyObject *fast_call(PyObject *, PyObject *const *args, Py_ssize_t count, PyObject *keywords)
{
    const torch::Tensor *tensors[TENSORS];
    int ints[INTS];
    if (keywords != nullptr || !plain_arguments(args, count, tensors, ints))
        return PyObject_Vectorcall(general<OPERATOR, ALIAS>, args, (size_t)count, keywords);
    try {
        return wrapped(call_plain<OPERATOR>(tensors, ints, std::make_index_sequence<TENSORS>(), std::make_index_sequence<INTS>()));
    } catch (py::error_already_set &e) {
        e.restore();
    } catch (...) {
        py::detail::try_translate_exceptions();
    }
    return nullptr;
}

// Puts the fast form of an operator in the place of the pybind11 function of this name.
template <auto OPERATOR, size_t TENSORS, size_t INTS, int ALIAS = 0>
void make_fast(py::module_ &m, const char *name)
{
    static PyMethodDef definition;
    general<OPERATOR, ALIAS> = py::object(m.attr(name)).release().ptr();
    const char *const doc = PyUnicode_AsUTF8(py::object(py::handle(general<OPERATOR, ALIAS>).attr("__doc__")).release().ptr());
    definition = PyMethodDef{name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&fast_call<OPERATOR, TENSORS, INTS, ALIAS>)),
                             METH_FASTCALL | METH_KEYWORDS, doc};
    m.attr(name) = py::reinterpret_steal<py::object>(PyCFunction_NewEx(&definition, nullptr, py::str(m.attr("__name__")).ptr()));
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    m.def("layer_forward", &layer_forward, "nn.TABConv2d.forward");
    // (a capsule: looking an object of a bound class up took 0.05 us of the call's 5)
    m.def("plain_class", [](py::object type) { return py::capsule(new PlainClass(type), [](void *p) { delete static_cast<PlainClass *>(p); }); });
    m.def("linear_forward", &linear_forward, "nn.TABLinear.forward");
    m.def("chain_forward", &chain_forward, "nn.TABPackedChain.forward");
    pybind11::register_exception_translator([](std::exception_ptr p) {
        try {
            if (p) std::rethrow_exception(p);
        } catch (const StatusError &e) {
            PyErr_SetString(pybind11::module_::import("tab_amd._capi").attr("TabError").ptr(), e.what());
        }
    });
    m.def("Quantize", &TAB_Quantize, "Ternarization or binarization of NHWC fp32 data, packed 64 channels per int64");
    m.def("Conv2d", &TAB_Conv2d, "Conv2d of all TAB types (0 TNN, 1 TBN, 2 BTN, 3 BNN; 4 DRF and 5 RTN of the CPU path)");
    m.def("TAB_Quantize", &TAB_Quantize, "alias of Quantize");
    m.def("TAB_Conv2d", &TAB_Conv2d, "alias of Conv2d");
    m.def("QuantizeNCHW", &TAB_QuantizeNCHW, "Quantize on NCHW fp32 data (X, thresholds, bitwidth, N, C, H, W)");
    m.def("QuantizeFormat", &TAB_QuantizeFormat, "Packer of conv types 4 (DRF) and 5 (RTN)");
    m.def("Threshold", &TAB_Threshold, "thresholds[n] = scale * mean|X[n]|", pybind11::arg("X"), pybind11::arg("N"),
          pybind11::arg("scale") = 0.7);
    m.def("QuantizeActivation", &TAB_QuantizeActivation, "QX of Quantize or QuantizeNCHW without the BTN vector");
    m.def("Conv2dStatic", &TAB_Conv2dStatic, "Conv2d with the packed activation in the library's built-in scratch");
    m.def("Conv2dPacked", &TAB_Conv2dPacked, "Conv2d on an already packed activation");
    m.def("Conv2dPackedOut", &TAB_Conv2dPackedOut, "Conv2dPacked with the output quantized and packed in the epilogue");
    make_fast<&TAB_Conv2d, 4, 12>(m, "Conv2d");
    make_fast<&TAB_Conv2d, 4, 12, 1>(m, "TAB_Conv2d");
    make_fast<&TAB_Quantize, 2, 5>(m, "Quantize");
    make_fast<&TAB_Quantize, 2, 5, 1>(m, "TAB_Quantize");
    make_fast<&TAB_QuantizeNCHW, 2, 5>(m, "QuantizeNCHW");
    make_fast<&TAB_Conv2dPacked, 3, 12>(m, "Conv2dPacked");
}
