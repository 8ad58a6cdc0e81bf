"""Layers that compute their own thresholds read the activation twice, the second time in the order that finds it in the caches, and
add the thresholds up in waves that may hold the ends of several images: against Threshold, QuantizeActivation and Conv2dPacked."""
import pytest
import torch

import oracle
import tab_amd
from tab_amd.nn import TABConv2d

pytestmark = pytest.mark.gpu

# N, H, W, C: 63, 64, 64 and 66 workgroups of 128 rows, images that end inside a wave; up to three and more images in a wave's pixels, of
# several partial sums each; ragged channels; more bytes than stay in the caches; one image of many partial sums
SIZES = [(2, 63, 64, 64), (2, 65, 63, 64), (3, 52, 52, 64), (5, 41, 41, 64), (11, 9, 8, 64), (19, 7, 7, 100), (150, 4, 4, 260), (64, 29, 31, 100),
         (37, 55, 53, 64), (21, 75, 67, 72), (13, 57, 55, 192), (1, 257, 255, 64), (1, 300, 301, 70)]


@pytest.mark.parametrize("nchw", [False, True])
@pytest.mark.parametrize("size", SIZES)
def test_layer_in_cache_order(size, nchw):
    N, H, W, C = size
    print(f"[case] layer order {size} nchw={nchw}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(C + N)
    # a scale for every image of its own: a row that takes its neighbour's threshold shows
    x = torch.randn((N, H, W, C), device="cuda", generator=g) * torch.logspace(-2, 2, N, device="cuda")[torch.randperm(N, device="cuda", generator=g)].view(N, 1, 1, 1)
    given = x.permute(0, 3, 1, 2).contiguous() if nchw else x
    for conv_type, k in ((0, 1), (1, 3)):
        w = torch.randn((130, C, k, k), device="cuda", generator=g)
        layer = TABConv2d.from_float(w, conv_type, 1, k // 2, act_scale=0.6, data_format="NCHW" if nchw else "NHWC")
        ths = tab_amd.Threshold(given, N, 0.6)
        torch.testing.assert_close(ths.double(), 0.6 * x.double().abs().mean(dim=(1, 2, 3)), rtol=1e-5, atol=0)
        q = tab_amd.QuantizeActivation(given, ths, 2, N, H, W, C, nchw=nchw)
        want = tab_amd.Conv2dPacked(q, layer.QW, layer.BTN_W, conv_type, k // 2, k // 2, 1, 1, N, H, W, C, 130, k, k).view(N, H, W, 130)
        for _ in range(2):
            assert torch.equal(layer(given), want.permute(0, 3, 1, 2) if nchw else want), conv_type


# N, H, W, C, KN, stride: one launch, whose tiles of 32 pixels hold one image, two and several; every form of input; tiles from the 64th on
ONE_LAUNCH = [(1, 56, 57, 64, 64, 1), (5, 23, 22, 128, 40, 1), (70, 8, 8, 64, 130, 1), (33, 8, 9, 64, 70, 2), (41, 8, 8, 128, 33, 3), (9, 13, 12, 256, 64, 2),
              (31, 7, 7, 192, 96, 1), (23, 7, 7, 512, 100, 1), (6, 15, 14, 512, 64, 3), (17, 9, 10, 70, 48, 1), (35, 7, 7, 100, 65, 2)]


@pytest.mark.parametrize("case", ONE_LAUNCH)
def test_one_launch_adds_up_thresholds(case):
    N, H, W, C, KN, stride = case
    print(f"[case] one launch, own thresholds {case}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(C + N)
    x = torch.randn((N, H, W, C), device="cuda", generator=g) * torch.logspace(-2, 2, N, device="cuda")[torch.randperm(N, device="cuda", generator=g)].view(N, 1, 1, 1)
    ths = tab_amd.Threshold(x, N, 0.6)
    q = tab_amd.QuantizeActivation(x, ths, 2, N, H, W, C)
    for conv_type in (0, 1):
        w = torch.randn((KN, C, 1, 1), device="cuda", generator=g)
        layer = TABConv2d.from_float(w, conv_type, stride, 0, act_scale=0.6, data_format="NHWC")
        want = tab_amd.Conv2dPacked(q, layer.QW, layer.BTN_W, conv_type, 0, 0, stride, stride, N, H, W, C, KN, 1, 1)
        assert torch.equal(layer(x).flatten(), want.flatten()), conv_type


# N, H, W, C: waves of 32 rows (the larger half) and of 8 that hold one image, two and many, the last of them short
GIVEN = [(41000, 1, 1, 64), (9001, 1, 5, 64), (1400, 31, 1, 64), (1250, 3, 11, 64), (700, 3, 7, 192), (90, 1, 7, 64), (33, 1, 1, 64), (11, 3, 3, 128)]


@pytest.mark.parametrize("size", GIVEN)
def test_given_thresholds_of_images_within_a_wave(size):
    N, H, W, C = size
    print(f"[case] given thresholds {size}", flush=True)
    g = torch.Generator().manual_seed(N)
    x = torch.randn((N, H, W, C), generator=g)
    ths = torch.rand(N, generator=g)
    for bits in (1, 2):
        want, _ = oracle.quantize(x.numpy(), ths.numpy(), bits, N, H, W, C)
        q = tab_amd.QuantizeActivation(x.cuda(), ths.cuda(), bits, N, H, W, C)
        assert torch.equal(q.cpu().flatten(), torch.from_numpy(want).flatten().view(q.dtype)), bits
