"""The counts of the two-plane quantizers at the edges of their slices: items of one workgroup and just beyond it, last units of
a few pixels, runs of four that overlap at an image's end, every layout's kernels; with a workspace and, through the C ABI,
without one.  Against the packed output's own nonzero plane."""
import ctypes

import pytest
import torch

import tab_amd

pytestmark = pytest.mark.gpu

CASES = [
    # layout, N, H, W, C
    ("NHWC", 700, 3, 3, 64), ("NHWC", 5, 8, 16, 64), ("NHWC", 3, 43, 3, 64), ("NHWC", 2, 32, 32, 64), ("NHWC", 2, 41, 25, 64),
    ("NHWC", 40, 56, 57, 256),                                                    # whole words
    ("NHWC", 300, 2, 5, 3), ("NHWC", 4, 31, 33, 7), ("NHWC", 3, 30, 41, 20), ("NHWC", 2, 90, 91, 30), ("NHWC", 64, 30, 31, 100),
    ("NHWC", 3, 9, 9, 900), ("NHWC", 2, 2, 2, 3100),                              # tiles
    ("NCHW", 9, 5, 5, 64), ("NCHW", 2, 19, 20, 64), ("NCHW", 2, 21, 31, 40), ("NCHW", 3, 50, 51, 20), ("NCHW", 4, 61, 43, 3),
    ("NCHW", 64, 57, 57, 64), ("NCHW", 400, 3, 5, 30), ("NCHW", 9, 1, 2, 70),     # words, one and four pixels a thread
    ("NCHW", 128, 27, 27, 128), ("NCHW", 2048, 8, 8, 512), ("NCHW", 300, 15, 15, 200), ("NCHW", 90, 28, 28, 128),  # gathered stores
]


@pytest.mark.parametrize("case", CASES)
def test_counts_are_those_of_the_packed_output(case):
    layout, N, H, W, C = case
    print(f"[case] counts {case}", flush=True)
    nchw = layout == "NCHW"
    x = torch.randn((N, C, H, W) if nchw else (N, H, W, C), device="cuda", generator=torch.Generator(device="cuda").manual_seed(N + C))
    ths = torch.linspace(0.1, 1.2, N, device="cuda")
    QX, BTN = tab_amd.QuantizeNCHW(x, ths, 2, N, C, H, W) if nchw else tab_amd.Quantize(x, ths, 2, N, H, W, C)
    same = x.permute(0, 2, 3, 1) if nchw else x
    want = (same.reshape(N, -1).abs() > ths[:, None]).sum(1).int()
    assert torch.equal(BTN, want)
    assert torch.equal(QX, tab_amd.QuantizeActivation(x, ths, 2, N, H, W, C, nchw=nchw))
    # the entry point without a workspace
    q, b = torch.zeros_like(QX), torch.full_like(BTN, -1)
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    f, sizes = (tab_amd._lib.tab_quantize_nchw, (N, C, H, W)) if nchw else (tab_amd._lib.tab_quantize, (N, H, W, C))
    assert f(p(x), p(ths), 2, *sizes, p(q), p(b), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    assert torch.equal(q, QX) and torch.equal(b, BTN)
