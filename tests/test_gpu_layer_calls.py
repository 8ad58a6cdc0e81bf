"""The layer calls (thresholds from the activation itself, constant output thresholds) against the operators they stand for,
which the other tests hold against the oracle."""
import pytest
import torch

import tab_amd
from tab_amd import _capi
from tab_amd.nn import TABConv2d, TABLinear

pytestmark = pytest.mark.gpu

# (N, H, W, C): one slice per image and several; images that end inside a wave's rows or pixels; ragged channels; planes
# that allow 16-byte loads and planes that do not; whole and partial words; an activation of many waves per image
SIZES = [(1, 1, 1, 3), (5, 1, 1, 64), (3, 7, 7, 100), (2, 33, 31, 64), (7, 9, 8, 512), (3, 6, 6, 1024), (40, 16, 16, 65), (2, 64, 64, 320)]


@pytest.mark.parametrize("nchw", [False, True])
@pytest.mark.parametrize("size", SIZES)
def test_layer_equals_threshold_quantize_conv(size, nchw):
    N, H, W, C = size
    g = torch.Generator("cpu").manual_seed(C)
    x = torch.randn((N, H, W, C), generator=g).cuda()
    given = x.permute(0, 3, 1, 2).contiguous() if nchw else x
    for conv_type in range(4):
        for k, stride in ((1, 1), (3, 2)):
            print(f"[case] layer {size} nchw={nchw} type={conv_type} k={k}", flush=True)
            w = torch.randn((70, C, k, k), generator=g)
            layer = TABConv2d.from_float(w, conv_type, stride, k // 2, act_scale=0.6, data_format="NCHW" if nchw else "NHWC")
            if tab_amd.out_shape(H, W, k, k, k // 2, k // 2, stride, stride)[0] < 1:
                continue
            y = layer(given)
            ths = tab_amd.Threshold(given, N, 0.6) if conv_type < 2 else torch.zeros(N, device="cuda")
            q = tab_amd.QuantizeActivation(given, ths, 2 if conv_type < 2 else 1, N, H, W, C, nchw=nchw)
            p = k // 2
            want = tab_amd.Conv2dPacked(q, layer.QW, layer.BTN_W, conv_type, p, p, stride, stride, N, H, W, C, 70, k, k)
            OH, OW = tab_amd.out_shape(H, W, k, k, p, p, stride, stride)
            want = want.view(N, OH, OW, 70)
            assert torch.equal(y, want.permute(0, 3, 1, 2) if nchw else want)
            if (H, W, k) == (1, 1, 1) and not nchw:
                fc = TABLinear(layer)
                assert torch.equal(fc(x.view(N, C)), want.view(N, 70))
                handle = layer.register_forward_hook(lambda m, i, o: o + 1)  # a hook on the inner layer still runs
                assert torch.equal(fc(x.view(N, C)), want.view(N, 70) + 1)
                handle.remove()


@pytest.mark.parametrize("PC", [1, 2, 4])
def test_constant_output_threshold_equals_one_per_image(PC):
    """tab_conv2d_packed_out_const through every shape the packed epilogues have, against the array form."""
    lib = _capi.load()
    g = torch.Generator("cpu").manual_seed(PC)
    N, H, W, C, KN = 3, 9, 10, 64 * PC, 130
    x, w = torch.randn((N, H, W, C), generator=g).cuda(), torch.randn((KN, 3, 3, C), generator=g).cuda()
    for type in range(4):
        ths, w_ths = tab_amd.Threshold(x, N, 0.7), tab_amd.Threshold(w, KN, 0.7)
        QX, _ = tab_amd.Quantize(x, ths, 2 if type < 2 else 1, N, H, W, C)
        QW, btn = tab_amd.Quantize(w, w_ths, 2 if type in (0, 2) else 1, KN, 3, 3, C)
        args = (type, 1, 1, 1, 1, N, H, W, C, KN, 3, 3)
        for bits, th in ((1, -2.5), (2, 6.0)):
            for tile in (-1, 0, 1, 2, 4, 5, 6, 7, 8, 9, 10, 11):
                print(f"[case] constant threshold type={type} bits={bits} tile={tile}", flush=True)
                tab_amd.set_conv_kernel(tab_amd.CONV_AUTO if tile < 0 else tab_amd.CONV_MATRIX, tile)
                want = tab_amd.Conv2dPackedOut(QX, QW, btn, *args, torch.full((N,), th, device="cuda"), bits)
                got = torch.empty_like(want)
                _capi.check(lib, lib.tab_conv2d_packed_out_const(QX.data_ptr(), QW.data_ptr(), btn.data_ptr(), *args, th, bits,
                                                                 got.data_ptr(), torch.cuda.current_stream().cuda_stream))
                assert torch.equal(got, want)
