"""The one-launch kernel of the smallest calls (tab_conv_small.hip) and the general forms of the one-launch 1x1 kernel:
bit-exact against the CPU oracle and equal to the two-launch path."""
import numpy as np
import pytest
import torch

import oracle
import tab_amd
from helpers import TYPE_NAMES, act_bits, make_layer, weight_bits
from tab_amd.nn import TABConv2d, TABLinear

pytestmark = pytest.mark.gpu

# N, H, W, C, KN, KH, KW, p1, p2, s1, s2
CASES = [
    (1, 32, 32, 64, 64, 3, 3, 1, 1, 1, 1),     # two blocks of 16 columns a line, K of nine words
    (1, 1, 1, 64, 1, 1, 1, 1, 1, 1, 1),        # one pixel, padded 1x1
    (2, 7, 7, 128, 70, 3, 3, 1, 1, 1, 1),      # two lines a block, four images' worth of padding, a ragged filter tile
    (3, 5, 9, 192, 33, 3, 3, 0, 1, 2, 1),      # three words a pixel: K of 27 words, weights refilled in registers
    (1, 9, 40, 256, 20, 3, 3, 1, 1, 1, 2),     # K of 36 words through LDS, columns shared at stride 2
    (40, 1, 1, 320, 48, 1, 1, 0, 0, 1, 1),     # one pixel an image: a block spans 16 images and their thresholds
    (5, 2, 3, 64, 17, 2, 3, 1, 2, 3, 4),       # strides beyond the kernel: every output its own slots; images below a block
    (2, 6, 20, 100, 75, 1, 5, 0, 2, 1, 2),     # channels that are no whole words, a kernel of one line
    (4, 3, 3, 3, 10, 3, 3, 1, 1, 1, 1),        # three channels
    (2, 14, 15, 65, 130, 3, 3, 1, 0, 1, 1),    # one channel in the second word, two filter groups
    (1, 20, 17, 512, 16, 1, 1, 0, 0, 1, 1),    # 1x1 with eight words
    (9, 4, 4, 126, 40, 1, 1, 0, 0, 2, 2),      # 1x1, two ragged words (conv1x1_fused)
    (7, 3, 2, 384, 140, 1, 1, 0, 0, 1, 1),     # 1x1, six words
]


@pytest.mark.parametrize("type", [0, 1, 2, 3])
@pytest.mark.parametrize("case", CASES)
def test_one_launch_matches_oracle(type, case):
    N, H, W, C, KN, KH, KW, p1, p2, s1, s2 = case
    print(f"[case] one launch {TYPE_NAMES[type]} {case}", flush=True)
    x, x_ths, w, w_ths = make_layer(type, N, H, W, C, KN, KH, KW, seed=3)
    qw_o, btn_o = oracle.quantize(w.numpy(), w_ths.numpy(), weight_bits(type), KN, KH, KW, C)
    args = (type, p1, p2, s1, s2, N, H, W, C, KN, KH, KW)
    want = oracle.conv2d(x.numpy(), qw_o, x_ths.numpy(), btn_o, *args)
    QW, BTN = torch.from_numpy(qw_o).cuda(), torch.from_numpy(btn_o).cuda()
    xd = x.cuda()
    assert type != 3 or tab_amd.conv2d_launches(xd, *args) == 1  # (the dearer types may take two)
    y = tab_amd.Conv2d(xd, QW, x_ths.cuda(), BTN, *args)
    assert np.array_equal(y.cpu().numpy(), want)
    # an input aligned to its floats only
    base = torch.empty(x.numel() + 1, device="cuda")
    shifted = base[1:].view(x.shape)
    shifted.copy_(xd)
    assert torch.equal(tab_amd.Conv2d(shifted, QW, x_ths.cuda(), BTN, *args), y)
    # a layer, NHWC and NCHW: its own thresholds
    for nchw in (False, True):
        layer = TABConv2d(QW, BTN, type, C, KN, (KH, KW), (s1, s2), (p1, p2), data_format="NCHW" if nchw else "NHWC")
        got = layer(xd.permute(0, 3, 1, 2).contiguous() if nchw else xd)
        ths = tab_amd.Threshold(xd, N) if act_bits(type) == 2 else torch.zeros(N, device="cuda")
        ref = tab_amd.Conv2d(xd, QW, ths, BTN, *args)
        OH, OW = tab_amd.out_shape(H, W, KH, KW, p1, p2, s1, s2)
        ref = ref.view(N, OH, OW, KN)
        if nchw and act_bits(type) == 2:  # the mean of the other layout may differ in its last bit
            assert (got != ref.permute(0, 3, 1, 2)).float().mean() < 0.01
        else:
            assert torch.equal(got, ref.permute(0, 3, 1, 2) if nchw else ref)


def test_special_values_and_negative_thresholds():
    """NaN, infinities, -0.0 and ties, positive and negative thresholds, through both input forms."""
    N, H, W, KN = 2, 8, 8, 20
    for C in (64, 70):
        for type in range(4):
            print(f"[case] special values {TYPE_NAMES[type]} C={C}", flush=True)
            x, _, w, w_ths = make_layer(type, N, H, W, C, KN, 1, 3, seed=1)
            flat = x.view(-1)
            flat[::7], flat[1::11], flat[2::13], flat[3::17], flat[4::5] = float("nan"), float("inf"), -float("inf"), -0.0, 0.5
            x_ths = torch.tensor([0.5, -0.25])
            qw_o, btn_o = oracle.quantize(w.numpy(), w_ths.numpy(), weight_bits(type), KN, 1, 3, C)
            args = (type, 0, 1, 1, 1, N, H, W, C, KN, 1, 3)
            want = oracle.conv2d(x.numpy(), qw_o, x_ths.numpy(), btn_o, *args)
            assert tab_amd.conv2d_launches(x.cuda(), *args) == 1
            y = tab_amd.Conv2d(x.cuda(), torch.from_numpy(qw_o).cuda(), x_ths.cuda(), torch.from_numpy(btn_o).cuda(), *args)
            assert np.array_equal(y.cpu().numpy(), want)


@pytest.mark.parametrize("C", [64, 128, 256, 320, 1024, 1088, 2048])
def test_linear_threshold_inside_the_launch(C):
    """A linear layer's ternary thresholds, taken from the rows inside the one launch, are those of Threshold to the last bit:
    rows of fewer and more words than a turn of the sum, counts that leave the last block of sixteen rows partly empty."""
    for N, KN in ((1, 16), (16, 70), (37, 20)):
        print(f"[case] linear thresholds N={N} C={C}", flush=True)
        g = torch.Generator("cpu").manual_seed(C + N)
        x = torch.randn((N, C), generator=g).cuda()
        fc = TABLinear.from_float(torch.randn((KN, C), generator=g), tab_amd.TBN)
        want = tab_amd.Conv2d(x, fc.conv.QW, tab_amd.Threshold(x, N), fc.conv.BTN_W, 1, 0, 0, 1, 1, N, 1, 1, C, KN, 1, 1)
        assert torch.equal(fc(x), want.view(N, KN))


@pytest.mark.parametrize("type", [4, 5])
@pytest.mark.parametrize("case", CASES)
def test_formats_match_their_two_launches(type, case):
    """Types 4 and 5 (5: channels whose words of 32 come in pairs), negative and zero thresholds included."""
    N, H, W, C, KN, KH, KW, p1, p2, s1, s2 = case
    print(f"[case] one launch type {type} {case}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(C)
    x = torch.randn((N, H, W, C), device="cuda", generator=g)
    w = torch.randn((KN, KH, KW, C), device="cuda", generator=g)
    ths = torch.linspace(-0.1, 0.9, N, device="cuda")
    QW = tab_amd.QuantizeFormat(w, torch.full((KN,), 0.4, device="cuda"), type, KN, KH, KW, C)
    btn = torch.zeros(KN, dtype=torch.int32, device="cuda")
    args = (type, p1, p2, s1, s2, N, H, W, C, KN, KH, KW)
    if type == 5 and (C + 31) // 32 % 2:
        assert tab_amd.conv2d_launches(x, *args) == 2
    want = tab_amd.Conv2dPacked(tab_amd.QuantizeFormat(x, ths, type, N, H, W, C), QW, btn, *args)
    assert torch.equal(tab_amd.Conv2d(x, QW, ths, btn, *args), want)
    base = torch.empty(x.numel() + 1, device="cuda")  # aligned to its floats only
    shifted = base[1:].view(x.shape)
    shifted.copy_(x)
    assert torch.equal(tab_amd.Conv2d(shifted, QW, ths, btn, *args), want)
