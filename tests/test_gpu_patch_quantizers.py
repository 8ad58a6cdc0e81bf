"""The quantizers that lay out a convolution's weights beside the activation, in the forms that only large or very wide activations take: the
NCHW gather of two and four words, NCHW past the caches, NCHW with a last word's waves apart, NHWC streaming, whole and ragged, very wide pixels.  Layers (their own thresholds and zero) and calls
with given thresholds through the kernel that reads those weights, against QuantizeActivation of the NHWC tensor and Conv2dPacked."""
import ctypes

import pytest
import torch

import tab_amd
from tab_amd import _capi
from tab_amd.nn import TABConv2d

pytestmark = pytest.mark.gpu

KN, SHAPE = 40, 15
# form, N, H, W, C
CASES = [("gather", 84, 56, 56, 128), ("gather", 88, 55, 55, 128), ("gather", 84, 56, 56, 256), ("gather", 88, 55, 55, 256), ("gather two planes", 88, 55, 55, 200),
         ("last past", 42, 56, 56, 75), ("last past", 41, 57, 57, 90), ("last four", 60, 30, 40, 75), ("last", 24, 30, 40, 96), ("last one plane", 44, 48, 64, 130),
         ("past", 42, 56, 56, 64), ("past", 41, 57, 57, 64), ("streaming", 23, 55, 55, 64), ("ragged streaming", 23, 55, 55, 70),
         ("ragged streaming", 23, 55, 55, 33), ("ragged", 2, 9, 7, 3100), ("ragged", 3, 6, 5, 3136)]


def takes_the_form(form, N, H, W, C, lib):
    f = lib.tab_internal_plane_form
    f.argtypes = [ctypes.c_int, ctypes.c_long, ctypes.c_long, ctypes.c_int]
    PC, runs, values = (C + 63) // 64, N * ((H * W + 3) // 4), N * H * W * C
    one, two = f(1, N, H * W, C), f(2, N, H * W, C)  # -1 gathered words, else the waves of a last word apart, 0 of none
    four = (runs + 63) // 64 * PC * 4 >= 2048
    past = four and values >= 8 << 20 and H * W >= 2048 and (H * W % 4 == 0 or values < 32 << 20)
    rows = C > 32 and N * H * W * PC > 512 * 128
    return {"gather": one == two == -1, "gather two planes": one > 0 and two == -1, "last past": one > 0 and two > 0 and past,
            "last four": one > 0 and two > 0 and four and not past, "last": one > 0 and two > 0 and not four, "last one plane": one > 0 and two == 0 and four,
            "past": one == two == 0 and past, "streaming": C % 64 == 0 and rows, "ragged streaming": C % 64 != 0 and rows, "ragged": C > 3072 and not rows}[form]


@pytest.fixture
def lib():
    lib = ctypes.CDLL(_capi.LIB_PATH)
    yield lib
    tab_amd.set_conv_kernel()


@pytest.mark.parametrize("case", CASES)
def test_weights_beside(case, lib):
    form, N, H, W, C = case
    assert takes_the_form(*case, lib)
    print(f"[case] weights beside {case}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(C + N)
    # a scale for every image of its own: a pixel that takes its neighbour's threshold shows
    x = torch.randn((N, H, W, C), device="cuda", generator=g) * torch.logspace(-2, 2, N, device="cuda")[torch.randperm(N, device="cuda", generator=g)].view(N, 1, 1, 1)
    nchw = form.startswith("gather") or form.startswith("last") or form == "past"
    sizes = (1, 1, 2, 2, N, H, W, C, KN, 3, 3)
    x_in, given = x, x.permute(0, 3, 1, 2).contiguous() if nchw else x
    if C == 3136:  # whole words, but x begins between two of them
        x_in = torch.empty(x.numel() + 1, device="cuda")[1:].view_as(x)
        given = x_in.copy_(x)
    OH, OW = tab_amd.out_shape(H, W, 3, 3, 1, 1, 2, 2)
    lib.tab_internal_force_patch(SHAPE)
    for type in range(4):
        w = torch.randn((KN, C, 3, 3), device="cuda", generator=g)
        layer = TABConv2d.from_float(w, type, 2, 1, act_scale=0.6, data_format="NCHW" if nchw else "NHWC")
        ths = tab_amd.Threshold(given, N, 0.6) if type < 2 else torch.zeros(N, device="cuda")
        q = tab_amd.QuantizeActivation(x, ths, 2 if type < 2 else 1, N, H, W, C)
        want = tab_amd.Conv2dPacked(q, layer.QW, layer.BTN_W, type, *sizes)
        what, size = (ctypes.c_int * 3)(), ctypes.c_size_t()
        assert lib.tab_internal_conv_patch_shape(type, *sizes, what, ctypes.byref(size)) == SHAPE
        y = layer(given)
        assert torch.equal(y.permute(0, 2, 3, 1) if nchw else y, want.view(N, OH, OW, KN)), type
        if not nchw:
            assert torch.equal(tab_amd.Conv2d(x_in, layer.QW, ths, layer.BTN_W, type, *sizes), want), type
    if not nchw:
        ths = tab_amd.Threshold(x, N, 0.6)
        w = torch.randn((KN, 3, 3, C), device="cuda", generator=g).abs()
        QW, btn = tab_amd.QuantizeFormat(w, tab_amd.Threshold(w, KN), 4, KN, 3, 3, C), torch.zeros(KN, dtype=torch.int32, device="cuda")
        want = tab_amd.Conv2dPacked(tab_amd.QuantizeFormat(x, ths, 4, N, H, W, C), QW, btn, 4, *sizes)
        assert torch.equal(tab_amd.Conv2d(x_in, QW, ths, btn, 4, *sizes), want)
