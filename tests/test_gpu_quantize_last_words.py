"""NCHW with a last word of at most 32 channels, which workgroups of its own take for several groups of pixels: one and two planes, counts, weights'
companion launches aside, at planes that end inside a run, a group and a workgroup's groups, small and large enough for four pixels a thread."""
import numpy as np
import pytest
import torch

import oracle
import tab_amd
from tab_amd import _capi

pytestmark = pytest.mark.gpu

# N, C, H, W: last words of 1, 16, 17, 32 channels (and 33, which has no units of its own), PC = 2, 3, 4, 5
CASES = [(1, 65, 1, 1), (3, 70, 4, 8), (5, 130, 3, 7), (2, 80, 3, 5), (1, 81, 8, 8), (3, 96, 7, 13), (2, 97, 8, 9), (1, 129, 16, 17), (2, 160, 5, 53), (1, 193, 9, 29), (2, 208, 15, 15), (1, 257, 11, 13),
         (1, 75, 61, 47), (4, 75, 48, 64), (9, 70, 67, 71), (30, 70, 59, 61), (24, 144, 56, 57), (2, 80, 255, 257), (17, 66, 40, 60)]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("bits", [1, 2])
def test_words_and_counts(case, bits):
    N, C, H, W = case
    print(f"[case] last words {case} bits {bits}", flush=True)
    g = torch.Generator("cuda").manual_seed(C + H)
    x = torch.randn((N, C, H, W), generator=g, device="cuda")
    x.view(-1)[::11] = 0.5
    ths = torch.full((N,), 0.5, device="cuda") if bits == 2 else torch.linspace(-0.5, 0.5, N, device="cuda")
    nhwc = x.permute(0, 2, 3, 1).contiguous()
    want, want_btn = oracle.quantize(nhwc.cpu().numpy(), ths.cpu().numpy(), bits, N, H, W, C)
    lib = _capi.load()
    for _ in range(2):
        q, btn = tab_amd.QuantizeNCHW(x, ths, bits, N, C, H, W)
        assert np.array_equal(q.cpu().numpy(), want) and np.array_equal(btn.cpu().numpy(), want_btn)
        assert np.array_equal(tab_amd.QuantizeActivation(x, ths, bits, N, H, W, C, True).cpu().numpy(), want)
        q.fill_(-1), btn.fill_(-1)  # without a workspace
        _capi.check(lib, lib.tab_quantize_nchw(x.data_ptr(), ths.data_ptr(), bits, N, C, H, W, q.data_ptr(), btn.data_ptr(), torch.cuda.current_stream().cuda_stream))
        assert np.array_equal(q.cpu().numpy(), want) and np.array_equal(btn.cpu().numpy(), want_btn)
        moved = torch.empty(x.numel() + 1, device="cuda")[1:].view(x.shape)
        moved.copy_(x)
        x = moved
