"""The quantizer of up to 32 channels (quantize_tile) at the edges of its tiles: lanes per word, tiles that span items, several hundred tiles, views
aligned to their floats only; and, from 33 channels on, the rows that take the wider pixels; all formats, against the oracle."""
import numpy as np
import pytest
import torch

import oracle
import tab_amd

pytestmark = pytest.mark.gpu

# N, H, W, C: each lane count's first and last channel count, tails of one channel, items of one pixel, tensors of one read and of several hundred
# tiles (more than 512, which keep their full size)
CASES = [(1, 1, 1, 1), (3, 5, 7, 4), (2, 9, 9, 5), (7, 3, 3, 8), (2, 8, 8, 9), (5, 4, 4, 16), (2, 7, 7, 17), (70, 1, 1, 32),
         (3, 6, 5, 33), (2, 10, 10, 63), (130, 1, 1, 65), (2, 3, 5, 129), (3, 4, 4, 333), (5, 1, 1, 3071), (2, 1, 2, 3073),
         (2, 1, 1, 8250), (9, 40, 41, 100), (9, 90, 91, 27), (2, 300, 301, 13), (7, 150, 151, 4)]


@pytest.mark.parametrize("case", CASES)
def test_quantize_tile_matches_oracle(case):
    N, H, W, C = case
    g = torch.Generator("cpu").manual_seed(C)
    x = torch.randn(case, generator=g)
    x.view(-1)[::13] = 0.5
    ths = torch.linspace(-0.3, 0.9, N) if N > 1 else torch.tensor([0.5])
    base = torch.empty(x.numel() + 1, device="cuda")
    views = [x.cuda(), base[1:].view(case)]
    views[1].copy_(views[0])
    for bits in (1, 2):
        print(f"[case] quantize_tile {case} bits={bits}", flush=True)
        want_q, want_btn = oracle.quantize(x.numpy(), ths.numpy(), bits, N, H, W, C)
        for v in views:
            q, btn = tab_amd.Quantize(v, ths.cuda(), bits, N, H, W, C)
            assert np.array_equal(q.cpu().numpy(), want_q) and np.array_equal(btn.cpu().numpy(), want_btn)
    for fmt in (tab_amd.DRF, tab_amd.RTN):
        print(f"[case] quantize_tile {case} format={fmt}", flush=True)
        want = oracle.quantize_format(x.numpy(), ths.numpy(), fmt, N, H, W, C)
        for v in views:
            assert np.array_equal(tab_amd.QuantizeFormat(v, ths.cuda(), fmt, N, H, W, C).cpu().numpy(), want)
