"""Rows of 64 channels of any channel count (quantize_rows_ragged): pixels that end inside a load, a row or a wave, items that end inside a
wave, both sizes of workgroups, views aligned to their floats only, with and without counts; all formats against the oracle, whole layers
(thresholds of their own) against the operators they stand for."""
import numpy as np
import pytest
import torch

import oracle
import tab_amd
from tab_amd.nn import TABConv2d

pytestmark = pytest.mark.gpu

# N, H, W, C: one and two channels past a row, one short of it, a whole row from between two floats; 1, 31, 32, 33 and 128 rows, 65536 (the
# last of the small workgroups) and one more pixel; items of one row, of a wave's rows and one less
CASES = [(1, 1, 1, 33), (31, 1, 1, 64), (1, 4, 4, 65), (3, 1, 11, 63), (32, 1, 1, 66), (2, 1, 31, 97), (2, 3, 11, 34), (1, 8, 8, 127), (4, 1, 8, 255),
         (5, 1, 1, 4099), (2, 128, 128, 100), (1, 1, 32769, 68), (3, 113, 97, 131)]


@pytest.mark.parametrize("case", CASES)
def test_matches_oracle(case):
    N, H, W, C = case
    g = torch.Generator("cpu").manual_seed(C)
    x = torch.randn(case, generator=g)
    x.view(-1)[::13] = 0.5
    x.view(-1)[5::17] = float("nan")
    x.view(-1)[-1] = float("inf")
    ths = torch.linspace(-0.3, 0.9, N) if N > 1 else torch.tensor([0.5])
    base = torch.full((x.numel() + 1,), float("inf"), device="cuda")
    views = [x.cuda(), base[1:].view(case)]
    views[1].copy_(views[0])
    for bits in (1, 2):
        print(f"[case] ragged rows {case} bits={bits}", flush=True)
        want_q, want_btn = oracle.quantize(x.numpy(), ths.numpy(), bits, N, H, W, C)
        for v in views:
            q, btn = tab_amd.Quantize(v, ths.cuda(), bits, N, H, W, C)
            assert np.array_equal(q.cpu().numpy(), want_q) and np.array_equal(btn.cpu().numpy(), want_btn)
            assert np.array_equal(tab_amd.QuantizeActivation(v, ths.cuda(), bits, N, H, W, C).cpu().numpy(), want_q)
    for fmt in (tab_amd.DRF, tab_amd.RTN):
        print(f"[case] ragged rows {case} format={fmt}", flush=True)
        want = oracle.quantize_format(x.numpy(), ths.numpy(), fmt, N, H, W, C)
        for v in views:
            assert np.array_equal(tab_amd.QuantizeFormat(v, ths.cuda(), fmt, N, H, W, C).cpu().numpy(), want)


@pytest.mark.parametrize("case", [(9, 55, 55, 70), (23, 55, 55, 70), (2, 60, 61, 333)])
def test_layers(case):
    N, H, W, C = case
    g = torch.Generator(device="cuda").manual_seed(C + N)
    scales = torch.logspace(-2, 2, N, device="cuda").view(N, 1, 1, 1)
    x = torch.randn(case, device="cuda", generator=g) * scales
    for type in range(4):
        print(f"[case] ragged layer {case} type={type}", flush=True)
        layer = TABConv2d.from_float(torch.randn((64, C, 3, 3), device="cuda", generator=g), type, 2, 1, act_scale=0.6, data_format="NHWC")
        bits = 2 if type < 2 else 1
        ths = tab_amd.Threshold(x, N, 0.6) if bits == 2 else torch.zeros(N, device="cuda")
        q = tab_amd.QuantizeActivation(x, ths, bits, N, H, W, C)
        want = tab_amd.Conv2dPacked(q, layer.QW, layer.BTN_W, type, 1, 1, 2, 2, N, H, W, C, 64, 3, 3)
        assert torch.equal(layer(x), want.view(N, *tab_amd.out_shape(H, W, 3, 3, 1, 1, 2, 2), 64)), type
