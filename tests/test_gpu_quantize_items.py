"""Small items of two planes, a workgroup each (quantize_items): counts against the oracle, thresholds of the items' own against Threshold and
QuantizeActivation, NHWC and NCHW, at and past the sizes at which they are taken and change their workgroup: slices that end with the item and
short of it, rows and planes that end inside a wave, channels that fill no word, views aligned to their floats only."""
import numpy as np
import pytest
import torch

import oracle
import tab_amd
from tab_amd import _capi

pytestmark = pytest.mark.gpu

# N, H, W, C: one pixel; 4096 values (four waves) and past; 12288 (the most with thresholds) and past; 26624
# (the most with counts; 24576 in ragged rows) and past, channels filled up to whole words; NCHW 32 pieces of 64 pixels and 16 channels (counts), 16 (thresholds), more than 256 items
CASES = [(5, 1, 1, 33), (3, 1, 1, 4096), (2, 1, 1, 4100), (7, 8, 8, 64), (3, 5, 13, 63), (2, 12, 16, 64), (2, 3, 43, 95), (3, 64, 3, 64), (4, 11, 17, 65),
         (300, 3, 3, 70), (2, 13, 32, 64), (3, 26, 16, 64), (2, 417, 1, 64), (2, 384, 1, 64), (2, 385, 1, 64), (2, 16, 12, 65), (2, 193, 1, 65), (2, 32, 64, 10), (2, 2049, 1, 10), (3, 32, 32, 20),
         (2, 1025, 1, 20), (2, 8, 64, 48), (2, 3, 171, 48), (300, 4, 4, 96), (257, 5, 13, 33), (2, 6, 13, 321), (1, 2, 3, 4099), (2, 1, 5, 2100)]


@pytest.mark.parametrize("case", CASES)
def test_counts_and_thresholds(case):
    N, H, W, C = case
    print(f"[case] items {case}", flush=True)
    g = torch.Generator("cpu").manual_seed(C + N)
    x = torch.randn(case, generator=g) * torch.logspace(-2, 2, N).view(N, 1, 1, 1)
    x.view(N, -1)[:, ::13] = 0.5
    x.view(-1)[5::97] = -0.0
    ths = 0.7 * x.abs().reshape(N, -1).mean(dim=1)
    want_q, want_btn = oracle.quantize(x.numpy(), ths.numpy(), 2, N, H, W, C)
    lib = _capi.load()
    ws = torch.empty(lib.tab_layer_workspace_bytes(2, N, H, W, C), dtype=torch.uint8, device="cuda")
    for nchw in (False, True):
        plain = (x.permute(0, 3, 1, 2) if nchw else x).contiguous().cuda()
        moved = torch.empty(x.numel() + 1, device="cuda")[1:].view(plain.shape)
        moved.copy_(plain)
        for v in (plain, moved):
            q, btn = tab_amd.QuantizeNCHW(v, ths.cuda(), 2, N, C, H, W) if nchw else tab_amd.Quantize(v, ths.cuda(), 2, N, H, W, C)
            assert np.array_equal(q.cpu().numpy(), want_q) and np.array_equal(btn.cpu().numpy(), want_btn)
            # without a workspace
            entry, sizes = (lib.tab_quantize_nchw, (N, C, H, W)) if nchw else (lib.tab_quantize, (N, H, W, C))
            q.fill_(-1), btn.fill_(-1)
            stream = torch.cuda.current_stream().cuda_stream
            _capi.check(lib, entry(v.data_ptr(), ths.cuda().data_ptr(), 2, *sizes, q.data_ptr(), btn.data_ptr(), stream))
            assert np.array_equal(q.cpu().numpy(), want_q) and np.array_equal(btn.cpu().numpy(), want_btn)
            # an item's own threshold, to the last bit that of Threshold
            own = tab_amd.Threshold(v, N, 0.6)
            want = tab_amd.QuantizeActivation(v, own, 2, N, H, W, C, nchw)
            q.fill_(-1)
            _capi.check(lib, lib.tab_layer_quantize(v.data_ptr(), nchw, 2, 0.6, N, H, W, C, q.data_ptr(), ws.data_ptr(), ws.numel(), stream))
            assert torch.equal(q, want)


def test_special_values():
    """An item whose mean is no number or infinite keeps nothing; its neighbours are as they are alone."""
    for C in (64, 70):
        x = torch.randn((4, 6, 7, C), device="cuda")
        x[1, 2, 3, 4], x[2, 0, 0, 0] = float("nan"), float("inf")
        lib = _capi.load()
        q = torch.full((4, 6, 7, (C + 63) // 64, 2), -1, dtype=torch.int64, device="cuda")
        ws = torch.empty(lib.tab_layer_workspace_bytes(2, 4, 6, 7, C), dtype=torch.uint8, device="cuda")
        _capi.check(lib, lib.tab_layer_quantize(x.data_ptr(), 0, 2, 0.7, 4, 6, 7, C, q.data_ptr(), ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
        assert not q[1].any() and not q[2].any()
        assert torch.equal(q, tab_amd.QuantizeActivation(x, tab_amd.Threshold(x, 4, 0.7), 2, 4, 6, 7, C))
