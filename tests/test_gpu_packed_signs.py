"""Packed output: bits taken from the signs of differences, at the thresholds where a difference could disagree with the comparison it stands
for: zeros of either sign, ties, denormal, negative, infinite and no number, in every kernel that packs, against the oracle's comparisons."""
import numpy as np
import pytest
import torch

import oracle
import tab_amd

pytestmark = pytest.mark.gpu

THRESHOLDS = np.array([0.0, -0.0, 1e-40, -1e-40, 0.5, -0.5, 2.0, -2.0, 7.999999, 1e30, -1e30, np.inf, -np.inf, np.nan], dtype=np.float32)
KERNELS = [(tab_amd.CONV_AUTO, -1)] + [(tab_amd.CONV_MATRIX, t) for t in (0, 1, 2, 4, 5, 6, 7, 8, 9)]


@pytest.mark.parametrize("type", [0, 1, 2, 3, 4, 5])
def test_thresholds(type):
    N = len(THRESHOLDS)
    # words a pixel: two and an odd number (whose operands go through registers), K of each length that the weights in registers are held for
    for H, W, C, KN, K in ((7, 5, 128, 130, 1), (6, 7, 70, 96, 3), (6, 7, 64, 96, 3), (5, 6, 192, 70, 3), (7, 5, 64, 130, 1), (7, 5, 192, 130, 1), (6, 7, 320, 64, 1)):
        rng = np.random.default_rng(type + C)
        words = lambda *shape: rng.integers(-2**63, 2**63, shape, dtype=np.int64)
        qx, qw = words(N, H, W, tab_amd.operand_words(type, 0, C)), words(KN, K, K, tab_amd.operand_words(type, 1, C))
        btn = np.zeros(KN, dtype=np.int32)
        if type == 2:
            btn = np.array([sum(bin(int(v) & (2**64 - 1)).count("1") for v in f[..., 1::2].ravel()) for f in qw], dtype=np.int32)
        args = (type, K // 2, K // 2, 1, 1, N, H, W, C, KN, K, K)
        y = np.ascontiguousarray(oracle.conv2d_packed(qx, qw, btn, *args)).reshape(N, H, W, KN)
        assert K == 3 or type > 3 or (y == 0).any()
        device = [torch.from_numpy(v).cuda() for v in (qx, qw, btn)]
        for bits in (1, 2):
            want, _ = oracle.quantize(y, THRESHOLDS, bits, N, H, W, KN)
            for kernel in KERNELS:
                if kernel[1] == 7 and (type > 3 or K * K * ((C + 63) // 64) > 9):
                    continue
                print(f"[case] packed signs type {type} {H}x{W}x{C}->{KN} k{K} bits {bits} kernel {kernel}", flush=True)
                tab_amd.set_conv_kernel(*kernel)
                try:
                    got = tab_amd.Conv2dPackedOut(*device, *args, torch.from_numpy(THRESHOLDS).cuda(), bits).cpu().numpy()
                finally:
                    tab_amd.set_conv_kernel()
                assert np.array_equal(got, want)
