"""The convolution that splits K over the waves of a workgroup, every shape forced, on arbitrary bits against the oracle: one word of K, fewer
units than waves, as many and one more, units beyond those requested first, odd and even numbers of words per pixel, rows past M, filters
past a tile, tiles that span images, strides, padding, 1x1 layers of single pixels."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
import tab_amd
from tab_amd import _capi

pytestmark = pytest.mark.gpu

SHAPES = range(19, 23)
CASES = [
    # N, H, W, C, KN, KH, KW, p1, p2, s1, s2
    (1, 1, 1, 1, 1, 1, 1, 0, 0, 1, 1), (33, 1, 1, 640, 65, 1, 1, 0, 0, 1, 1), (2, 5, 7, 64, 31, 3, 3, 1, 1, 1, 1), (3, 4, 4, 128, 33, 3, 3, 1, 1, 1, 1),
    (2, 9, 8, 192, 64, 3, 3, 1, 0, 2, 1), (1, 7, 7, 1024, 40, 3, 3, 1, 1, 1, 1), (5, 3, 3, 2112, 96, 2, 3, 1, 2, 1, 2), (2, 11, 6, 256, 70, 5, 5, 2, 1, 2, 2),
    (1, 33, 2, 70, 97, 1, 1, 0, 0, 1, 1), (4, 1, 9, 320, 130, 1, 2, 0, 1, 1, 1),
]


@pytest.fixture(scope="module")
def lib():
    return ctypes.CDLL(_capi.LIB_PATH)


@pytest.mark.parametrize("case", CASES)
def test_arbitrary_bits(case, lib):
    N, H, W, C, KN, KH, KW, p1, p2, s1, s2 = case
    print(f"[case] waves {case}", flush=True)
    g = np.random.default_rng(KN + C)
    for type in range(6):
        qx = g.integers(-2**63, 2**63 - 1, (N, H, W, tab_amd.operand_words(type, 0, C)), dtype=np.int64)
        qw = g.integers(-2**63, 2**63 - 1, (KN, KH, KW, tab_amd.operand_words(type, 1, C)), dtype=np.int64)
        btn = g.integers(0, 99, KN, dtype=np.int32)
        want = oracle.conv2d_packed(qx, qw, btn, type, p1, p2, s1, s2, N, H, W, C, KN, KH, KW)
        a = [torch.from_numpy(v).cuda() for v in (qx, qw, btn)]
        for shape in SHAPES:
            lib.tab_internal_force_patch(shape)
            got = tab_amd.Conv2dPacked(*a, type, p1, p2, s1, s2, N, H, W, C, KN, KH, KW)
            assert np.array_equal(got.cpu().numpy().reshape(want.shape), want), (type, shape)
