"""The operators through the C ABI and nothing else: ctypes calls of include/tab_amd.h on buffers of torch's, the other side of
the tests that hold the extension's checks, allocations and argument order."""
import torch

from tab_amd import _capi

_lib = _capi.load()


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _empty(shape, dtype):
    """A buffer whose every element the call has to write: -1 is no result of the calls that are compared."""
    return torch.full(shape, -1, dtype=dtype, device="cuda")


def _check(status):
    _capi.check(_lib, status)


def _quantize(entry, X, thresholds, bitwidth, N, H, W, C, *sizes):
    QX = _empty((N, H, W, _lib.tab_packed_channels(C), bitwidth), torch.int64)
    BTN = _empty((N,), torch.int32)
    _check(entry(X.data_ptr(), thresholds.data_ptr(), bitwidth, *sizes, QX.data_ptr(), BTN.data_ptr(), _stream()))
    return [QX, BTN]


def Quantize(X, thresholds, bitwidth, N, H, W, C):
    return _quantize(_lib.tab_quantize, X, thresholds, bitwidth, N, H, W, C, N, H, W, C)


def QuantizeNCHW(X, thresholds, bitwidth, N, C, H, W):
    return _quantize(_lib.tab_quantize_nchw, X, thresholds, bitwidth, N, H, W, C, N, C, H, W)


def QuantizeFormat(X, thresholds, type, N, H, W, C):
    QX = _empty((N, H, W, _lib.tab_packed_channels(C), 2) if type == 4 else (N, H, W, (C + 31) // 32), torch.int64)
    _check(_lib.tab_quantize_format(X.data_ptr(), thresholds.data_ptr(), type, N, H, W, C, QX.data_ptr(), _stream()))
    return QX


def Threshold(X, N, scale):
    ths = _empty((N,), torch.float32)
    per_item = X.numel() // N
    ws = torch.empty(_lib.tab_threshold_workspace_bytes(N, per_item), dtype=torch.uint8, device="cuda")
    _check(_lib.tab_threshold(X.data_ptr(), N, per_item, scale, ths.data_ptr(), ws.data_ptr(), ws.numel(), _stream()))
    return ths


def _out(N, H, W, KN, KH, KW, p1, p2, s1, s2):
    return N, KN, _lib.tab_out_extent(H, p1, KH, s1), _lib.tab_out_extent(W, p2, KW, s2)


def Conv2d(X, QW, thresholds, btn, type, p1, p2, s1, s2, N, H, W, C, KN, KH, KW):
    Y = _empty(_out(N, H, W, KN, KH, KW, p1, p2, s1, s2), torch.float32)
    ws = torch.empty(_lib.tab_conv2d_workspace_bytes(type, N, H, W, C), dtype=torch.uint8, device="cuda")
    _check(_lib.tab_conv2d(X.data_ptr(), QW.data_ptr(), thresholds.data_ptr(), btn.data_ptr(), type, p1, p2, s1, s2, N, H, W, C,
                           KN, KH, KW, Y.data_ptr(), ws.data_ptr(), ws.numel(), _stream()))
    return Y


def Conv2dPacked(QX, QW, btn, type, p1, p2, s1, s2, N, H, W, C, KN, KH, KW):
    Y = _empty(_out(N, H, W, KN, KH, KW, p1, p2, s1, s2), torch.float32)
    _check(_lib.tab_conv2d_packed(QX.data_ptr(), QW.data_ptr(), btn.data_ptr(), type, p1, p2, s1, s2, N, H, W, C, KN, KH, KW,
                                  Y.data_ptr(), _stream()))
    return Y


def Conv2dPackedOut(QX, QW, btn, type, p1, p2, s1, s2, N, H, W, C, KN, KH, KW, out_thresholds, out_bitwidth):
    _, _, OH, OW = _out(N, H, W, KN, KH, KW, p1, p2, s1, s2)
    QY = _empty((N, OH, OW, _lib.tab_packed_channels(KN), out_bitwidth), torch.int64)
    _check(_lib.tab_conv2d_packed_out(QX.data_ptr(), QW.data_ptr(), btn.data_ptr(), type, p1, p2, s1, s2, N, H, W, C, KN, KH, KW,
                                      out_thresholds.data_ptr(), out_bitwidth, QY.data_ptr(), _stream()))
    return QY
