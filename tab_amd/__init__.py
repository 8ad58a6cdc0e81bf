"""tab_amd - MI355X (gfx950) implementation of TAB's quantize + bitwise-conv operators.

Host-side mirror of the reference's operator interface (TAB_GPU.cpp:34-65): the same two
calls, positional argument lists, return tensors and error behaviour, on top of the C ABI
in include/tab_amd.h.  The calls go through the extension tab_amd._C (csrc/torch_binding.cpp), whose
checks, allocations and stream lookup take under 2 us where the same in Python took 13; PyTorch only
supplies device memory and the current stream.

    QW, BTN_W = Quantize(w, w_ths, bitwidth, KN, KH, KW, C)
    y = Conv2d(x, QW, x_ths, BTN_W, type, pad1, pad2, stride1, stride2, N, H, W, C, KN, KH, KW)
"""
import torch

from . import _capi

_lib = _capi.load()
TabError = _capi.TabError

from . import _C  # noqa: E402  (its errors are TabError)

TNN, TBN, BTN, BNN = 0, 1, 2, 3
DRF, RTN = 4, 5  # the types of the reference's CPU path only (TAB_CPU.cpp:332-383)


def version():
    return _lib.tab_version().decode()


def _call(fn, tensors, ints, *rest):
    """The call that the extension refused for an argument's type: whatever is no tensor where one belongs is named
    (CHECK_INPUT of the reference, TAB_GPU.cpp:7-9), everything else is made an int and the call repeated."""
    for name, t in tensors.items():
        if not isinstance(t, torch.Tensor):
            raise TypeError(f"{name} must be a torch.Tensor")
    return fn(*tensors.values(), *(int(v) for v in ints), *rest)


def packed_channels(C):
    return _lib.tab_packed_channels(int(C))


def operand_words(type, operand, C):
    """int64 words per pixel of the activation (operand 0) or per tap of the weight (operand 1)."""
    return _lib.tab_operand_words(int(type), int(operand), int(C))


def out_shape(H, W, KH, KW, pad1, pad2, stride1, stride2):
    """(OH, OW) by the reference's integer-division formula (TAB_GEMM.cu:354-357)."""
    return (_lib.tab_out_extent(H, pad1, KH, stride1), _lib.tab_out_extent(W, pad2, KW, stride2))


def Quantize(X, thresholds, bitwidth, N, H, W, C):
    """Ternarize (bitwidth 2) or binarize (bitwidth 1) NHWC fp32 data and pack 64 channels
    per int64 word.  Returns [QX, BTN]: QX int64 (N,H,W,PC,bitwidth), BTN int32 (N,)
    (TAB_GPU.cpp:53-58, TAB_GEMM.cu:250-322)."""
    try:
        return _C.Quantize(X, thresholds, bitwidth, N, H, W, C)
    except TypeError:
        return _call(_C.Quantize, {"X": X, "thresholds": thresholds}, (bitwidth, N, H, W, C))


def QuantizeActivation(X, thresholds, bitwidth, N, H, W, C, nchw=False):
    """QX of Quantize (or, with nchw, of QuantizeNCHW with X given as N, C, H, W) without the BTN vector: an
    activation's counts are read by nobody, and passing NULL for them to the C ABI skips the launches that
    produce them."""
    try:
        return _C.QuantizeActivation(X, thresholds, bitwidth, N, H, W, C, nchw)
    except TypeError:
        return _call(_C.QuantizeActivation, {"X": X, "thresholds": thresholds}, (bitwidth, N, H, W, C), bool(nchw))


def QuantizeNCHW(X, thresholds, bitwidth, N, C, H, W):
    """Quantize on an NCHW fp32 tensor (the layout the reference's CPU quantizers read, TAB_CPU.cpp:20-206, and
    the argument order of its CPU binding, TAB_CPU.cpp:621): returns [QX, BTN] exactly as
    Quantize(X.permute(0, 2, 3, 1), thresholds, bitwidth, N, H, W, C) would, without the transposed copy."""
    try:
        return _C.QuantizeNCHW(X, thresholds, bitwidth, N, C, H, W)
    except TypeError:
        return _call(_C.QuantizeNCHW, {"X": X, "thresholds": thresholds}, (bitwidth, N, C, H, W))


def QuantizeFormat(X, thresholds, type, N, H, W, C):
    """Packer of conv types 4 (DoReFa 2-bit levels; QX int64 (N,H,W,PC,2), plane 0 = weight-2 bit)
    and 5 (RTN 2-bit fields; QX int64 (N,H,W,ceil(C/32))), for activations and weights alike.  The
    layouts are the ones DRFGEMM_baseline / RTNGEMM_baseline read (TAB_CPU.cpp:332-383); the
    reference has no quantizer for them, the value rules (uniform step thresholds[n]; the
    ternarizer's compares) are this library's."""
    try:
        return _C.QuantizeFormat(X, thresholds, type, N, H, W, C)
    except TypeError:
        return _call(_C.QuantizeFormat, {"X": X, "thresholds": thresholds}, (type, N, H, W, C))


def Threshold(X, N, scale=0.7):
    """ths[n] = scale * mean(|X[n]|) per item (image or filter), fp32 (N,), computed on the
    device in one pass: the threshold rule the reference leaves to the caller (README.md:45).
    Reproducible from run to run; within 1e-5 relative of an fp64 reference."""
    try:
        return _C.Threshold(X, N, scale)
    except TypeError:
        return _call(_C.Threshold, {"X": X}, (N,), float(scale))


def Conv2d(X, QW, thresholds, btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW):
    """Quantize the NHWC fp32 activation on the fly (ternary for types 0/1, binary for 2/3; types 4
    and 5 of the CPU path through QuantizeFormat) and convolve it with the packed weights.  Returns fp32 shaped
    (N,KN,OH,OW) whose memory is ordered (n,oh,ow,kn), exactly as the reference's reshape
    of its GEMM result (TAB_GPU.cpp:34-42, TAB_GEMM.cu:325-527)."""
    try:
        return _C.Conv2d(X, QW, thresholds, btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW)
    except TypeError:
        return _call(_C.Conv2d, {"X": X, "QW": QW, "thresholds": thresholds, "btn": btn},
                     (type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW))


def conv2d_launches(X, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW):
    """Kernels one Conv2d call with these arguments enqueues: 1 (quantize and convolution in one launch) or 2."""
    return _lib.tab_conv2d_launches(X.data_ptr(), *(int(v) for v in (type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW)))


def static_scratch_bytes():
    """Size of the scratch array built into the library that Conv2dStatic packs the activation into."""
    return _lib.tab_static_scratch_bytes()


def Conv2dStatic(X, QW, thresholds, btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, out=None):
    """Conv2d through tab_conv2d_static: the packed activation goes to the library's built-in device scratch
    (static_scratch_bytes() bytes per GPU) instead of a workspace tensor, so the C call allocates nothing.
    With `out` (fp32, N*OH*OW*KN elements) given, this wrapper allocates nothing either.  Calls that may
    overlap on one GPU race on the shared scratch."""
    try:
        return _C.Conv2dStatic(X, QW, thresholds, btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW, out)
    except TypeError:
        return _call(_C.Conv2dStatic, {"X": X, "QW": QW, "thresholds": thresholds, "btn": btn},
                     (type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW), out)


def Conv2dPacked(QX, QW, btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW):
    """Conv2d on an activation already packed by Quantize (bitwidth 2 for types 0/1,
    1 for types 2/3) or by QuantizeFormat (types 4/5): the pad + im2row + GEMM stages of
    TAB_GEMM.cu:447-509 only."""
    try:
        return _C.Conv2dPacked(QX, QW, btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW)
    except TypeError:
        return _call(_C.Conv2dPacked, {"QX": QX, "QW": QW, "btn": btn},
                     (type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW))


def Conv2dPackedOut(QX, QW, btn, type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW,
                    out_thresholds, out_bitwidth):
    """Conv2dPacked whose output is quantized and packed in the kernel's epilogue: returns QY int64
    (N, OH, OW, ceil(KN/64), out_bitwidth), equal bit for bit to
    Quantize(Conv2dPacked(...), out_thresholds, out_bitwidth, N, OH, OW, KN)[0] - the conv output's
    (n, oh, ow, kn) memory read as the next layer's NHWC activation - without the fp32 tensor ever
    being written.  out_thresholds: fp32 [>=N], one threshold per image."""
    args = (type, padding1, padding2, stride1, stride2, N, H, W, C, KN, KH, KW)
    try:
        return _C.Conv2dPackedOut(QX, QW, btn, *args, out_thresholds, out_bitwidth)
    except TypeError:
        if not isinstance(out_thresholds, torch.Tensor):
            raise TypeError("out_thresholds must be a torch.Tensor")
        return _call(_C.Conv2dPackedOut, {"QX": QX, "QW": QW, "btn": btn}, args, out_thresholds, int(out_bitwidth))


CONV_AUTO, CONV_MATRIX, CONV_POPCOUNT = 0, 1, 2


def set_conv_kernel(kernel=CONV_AUTO, tile=-1):
    """Pick the conv kernel (process-wide): CONV_AUTO, CONV_MATRIX (tile 0..11 or -1) or
    CONV_POPCOUNT (tile 0..2 or -1).  Every choice gives bit-identical outputs."""
    _capi.check(_lib, _lib.tab_set_conv_kernel(int(kernel), int(tile)))


# names of the reference's CPU module (TAB_CPU.cpp:636-639)
TAB_Quantize = Quantize
TAB_Conv2d = Conv2d

__all__ = ["Quantize", "QuantizeNCHW", "QuantizeActivation", "conv2d_launches", "QuantizeFormat", "Conv2d", "Conv2dStatic", "static_scratch_bytes", "Conv2dPacked", "Conv2dPackedOut", "Threshold", "TAB_Quantize", "TAB_Conv2d", "TabError",
           "packed_channels", "out_shape", "version", "TNN", "TBN", "BTN", "BNN", "set_conv_kernel",
           "CONV_AUTO", "CONV_MATRIX", "CONV_POPCOUNT"]
