"""Rows of Y that are no whole cache lines: fp32 output on either side of the size from which it is written through the caches
(M * KN of 6 << 20), by the one-launch 1x1 kernel and by the tiled kernels, against the popcount kernel."""
import pytest
import torch

import tab_amd
from helpers import two_launches

pytestmark = pytest.mark.gpu

# N, H, W, C, KN, K, p: M * KN just below and from the line on, 33 filters, a multiple of 32 for comparison
CASES = [(8, 104, 104, 64, 72, 1, 0), (8, 105, 104, 64, 73, 1, 0), (3, 255, 250, 128, 33, 1, 0), (2, 240, 230, 64, 57, 3, 1),
         (2, 241, 230, 64, 57, 3, 1), (4, 100, 100, 64, 160, 1, 0)]


@pytest.mark.parametrize("case", CASES)
def test_cached_and_streamed_rows(case):
    N, H, W, C, KN, K, p = case
    print(f"[case] ragged rows {case}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(KN)
    x = torch.randn((N, H, W, C), device="cuda", generator=g)
    w = torch.randn((KN, K, K, C), device="cuda", generator=g)
    ths = tab_amd.Threshold(x, N)
    for type in range(4):
        QW, btn = tab_amd.Quantize(w, tab_amd.Threshold(w, KN), 2 if type in (0, 2) else 1, KN, K, K, C)
        run = lambda: tab_amd.Conv2d(x, QW, ths, btn, type, p, p, 1, 1, N, H, W, C, KN, K, K)  # noqa: E731
        got = [run()]
        with two_launches():
            got.append(run())
        try:
            tab_amd.set_conv_kernel(tab_amd.CONV_POPCOUNT)
            want = run()
        finally:
            tab_amd.set_conv_kernel()
        assert all(torch.equal(y, want) for y in got), type
