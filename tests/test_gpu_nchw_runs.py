"""QuantizeNCHW where its runs of four pixels can go wrong: planes whose size four does not divide (the last run of an image
moves back over the one before it), every number of waves per word, a word's last few channels, the loads past the caches,
the gathered stores on odd planes.  Against Quantize on the transposed tensor, which the CPU oracle pins; bit-exact."""
import pytest
import torch

import tab_amd

pytestmark = pytest.mark.gpu

CASES = [
    # N, C, H, W
    (32768, 128, 1, 5), (22000, 200, 1, 6),  # gathered stores, two and four words a thread
    (8200, 100, 7, 1),  # four waves a word, the second word of 36 channels
    (33000, 30, 1, 7), (66000, 16, 7, 1), (66000, 3, 1, 5),  # two waves and one wave a word
    (64, 64, 3, 683), (64, 70, 41, 50),  # past the caches
    (5, 33, 1, 3), (700, 20, 1, 1), (3, 17, 2, 33),  # one pixel a thread
]


@pytest.mark.parametrize("bits", [1, 2])
@pytest.mark.parametrize("case", CASES)
def test_nchw_equals_the_nhwc_quantizer(bits, case):
    N, C, H, W = case
    print(f"[case] QuantizeNCHW runs bits={bits} N={N} C={C} {H}x{W}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(C + W)
    x = torch.randn((N, C, H, W), device="cuda", generator=g)
    ths = torch.linspace(-0.1, 0.9, N, device="cuda")
    x[:, 0, 0, 0] = ths  # ties
    x[:, -1, -1, -1] = float("nan")
    QX, BTN = tab_amd.QuantizeNCHW(x, ths, bits, N, C, H, W)
    want, want_btn = tab_amd.Quantize(x.permute(0, 2, 3, 1).contiguous(), ths, bits, N, H, W, C)
    assert torch.equal(QX, want) and torch.equal(BTN, want_btn)
