"""Packed layers of short K whose launches have fewer workgroups a CU than fit, at the edges of their rounds, against the oracle."""
import numpy as np
import pytest
import torch

import oracle
import tab_amd

pytestmark = pytest.mark.gpu


# (type, N, H, W, C, KN, K): four words in 2 and 4 filter tiles, one and nine words; more and fewer workgroups than two a CU, a last tile of
# one pixel and of 31
@pytest.mark.parametrize("type,N,H,W,C,KN,K", [(2, 2, 331, 167, 256, 64, 1), (3, 1, 501, 133, 200, 130, 1), (3, 3, 97, 229, 256, 300, 1), (2, 1, 263, 251, 64, 64, 3),
                                               (0, 7, 103, 91, 64, 129, 1), (1, 1, 257, 255, 128, 64, 1)])
@pytest.mark.parametrize("bits", [1, 2])
def test_against_the_oracle(type, N, H, W, C, KN, K, bits):
    print(f"[case] regs workgroups type {type} {N}x{H}x{W}x{C}->{KN} k{K} bits {bits}", flush=True)
    rng = np.random.default_rng(type + C + bits)
    words = lambda *shape: rng.integers(-2**63, 2**63, shape, dtype=np.int64)
    keep = np.array([2**(C - 64 * w) - 1 if C - 64 * w < 63 else -1 for w in range((C + 63) // 64)], dtype=np.int64)  # channels that exist
    aw, bw = tab_amd.operand_words(type, 0, C), tab_amd.operand_words(type, 1, C)
    qx, qw = (words(*shape) & np.repeat(keep, shape[-1] // len(keep)) for shape in ((N, H, W, aw), (KN, K, K, bw)))
    btn = np.zeros(KN, dtype=np.int32)
    if type == 2:
        btn = np.array([sum(bin(int(v) & (2**64 - 1)).count("1") for v in f[..., 1::2].ravel()) for f in qw], dtype=np.int32)
    args = (type, K // 2, K // 2, 1, 1, N, H, W, C, KN, K, K)
    ths = rng.uniform(-3, 9, N).astype(np.float32)
    y = np.ascontiguousarray(oracle.conv2d_packed(qx, qw, btn, *args)).reshape(N, H, W, KN)
    want, _ = oracle.quantize(y, ths, bits, N, H, W, KN)
    tab_amd.set_conv_kernel(tab_amd.CONV_MATRIX, 7)
    device = [torch.from_numpy(v).cuda() for v in (qx, qw, btn)]
    got = tab_amd.Conv2dPackedOut(*device, *args, torch.from_numpy(ths).cuda(), bits).cpu().numpy()
    assert np.array_equal(got, want)
