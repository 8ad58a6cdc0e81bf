"""Layers of at most 32 filters: the 128x32 and 64x32 tiles (matrix shapes 1 and 8, K split over two and four waves) at one filter,
31 and 32, rows past M, words of K that fill no chunk, types 0..5, and 33 filters, which take the wide tiles; against the kernel of
64x64 tiles, and the popcount kernel for types 0..3."""
import pytest
import torch

import tab_amd

pytestmark = pytest.mark.gpu

CASES = [
    # N, H, W, C, KN, KH, KW, p, s
    (3, 13, 11, 128, 1, 3, 3, 1, 1), (2, 17, 16, 212, 31, 5, 5, 2, 1), (5, 9, 9, 100, 32, 1, 3, 0, 2), (1, 40, 41, 512, 32, 1, 1, 0, 1),
    (2, 20, 20, 128, 33, 3, 3, 1, 1), (7, 30, 30, 384, 7, 3, 3, 1, 1),
]


@pytest.mark.parametrize("type", range(6))
@pytest.mark.parametrize("case", CASES)
def test_narrow_tiles(case, type):
    N, H, W, C, KN, KH, KW, p, s = case
    print(f"[case] narrow type={type} {case}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(KN + C)
    x = torch.randn((N, H, W, C), device="cuda", generator=g)
    w = torch.randn((KN, KH, KW, C), device="cuda", generator=g)
    if type > 3:
        QX = tab_amd.QuantizeFormat(x, tab_amd.Threshold(x, N), type, N, H, W, C)
        QW, btn = tab_amd.QuantizeFormat(w, tab_amd.Threshold(w, KN), type, KN, KH, KW, C), torch.zeros(KN, dtype=torch.int32, device="cuda")
    else:
        QX = tab_amd.QuantizeActivation(x, tab_amd.Threshold(x, N), 2 if type < 2 else 1, N, H, W, C)
        QW, btn = tab_amd.Quantize(w, tab_amd.Threshold(w, KN), 2 if type in (0, 2) else 1, KN, KH, KW, C)
    run = lambda: tab_amd.Conv2dPacked(QX, QW, btn, type, p, p, s, s, N, H, W, C, KN, KH, KW)  # noqa: E731
    got = {"auto": run()}
    try:
        for tile in (1, 8, 2):
            tab_amd.set_conv_kernel(tab_amd.CONV_MATRIX, tile)
            got[tile] = run()
        if type <= 3:
            tab_amd.set_conv_kernel(tab_amd.CONV_POPCOUNT)
            got["popcount"] = run()
    finally:
        tab_amd.set_conv_kernel()
    for name, y in got.items():
        assert torch.equal(y, got[2]), name
