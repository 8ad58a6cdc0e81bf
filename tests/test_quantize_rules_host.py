"""The rules that pick a quantizer's form, on the host: the library's choices on measured calls of both forms, with the regret that the rules'
comments state."""
import ctypes
import os
import re

import numpy as np
import pytest

from tab_amd import _capi

TUNING = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tab_amd", "tuning")


def geometric(ratios):
    return float(np.exp(np.mean(np.log(ratios))))


def parse(name, pattern):
    with open(os.path.join(TUNING, name)) as f:
        for line in f:
            m = re.match(pattern, line)
            if m:
                yield m.groups()


def test_items_by_workgroups():
    f = ctypes.CDLL(_capi.LIB_PATH).tab_internal_quantize_items
    f.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_long, ctypes.c_long, ctypes.c_int]
    taken, best, chosen = [], [], 0
    for kind, layout, N, H, W, C, two, one in parse("quantize_items_timings.txt", r"(own|counts) (NHWC|NCHW) (\d+)x(\d+)x(\d+)x(\d+) \| (\S+) (\S+)"):
        two, one = float(two), float(one)
        items = bool(f(kind == "own", layout == "NCHW", int(N), int(H) * int(W), int(C)))
        taken.append((one if items else two) / two)
        best.append(min(one, two) / two)
        chosen += items
    slower = np.array(taken)
    stated = (len(taken), chosen, geometric(taken), geometric(best), sorted(slower)[-3:])
    assert len(taken) > 1150 and 650 < chosen < 720, stated
    assert geometric(taken) < 0.883 and geometric(best) > 0.879, stated  # fitted: 0.8824, 0.8792
    assert (slower > 1.02).sum() <= 4 and (slower > 1.05).sum() <= 2 and slower.max() < 1.14, stated


def test_last_words():
    f = ctypes.CDLL(_capi.LIB_PATH).tab_internal_plane_form
    f.argtypes = [ctypes.c_int, ctypes.c_long, ctypes.c_long, ctypes.c_int]
    taken, apart, best = [], [], []
    for bits, N, H, W, C, alike, last, units in parse("quantize_last_words_timings.txt", r"planes (\d) (\d+)x(\d+)x(\d+)x(\d+) \| (\S+) (\S+) (\S+)"):
        alike, last, units = float(alike), float(last), float(units)
        form = f(int(bits), int(N), int(H) * int(W), int(C))
        assert form in (-1, 0, 1, 2)
        PC = (int(C) + 63) // 64
        unit = 4 if PC % 4 == 0 else 2 if PC % 2 == 0 else 1
        large = unit > 1 and (int(N) * ((int(H) * int(W) + 3) // 4) + 63) // 64 * (PC // unit) >= 1024  # (else "alike" is "units" timed twice)
        assert form >= 0 or large
        taken.append((last if form > 0 else units if large and form == 0 else alike) / alike)
        apart.append(form > 0)
        best.append(min(alike, last, units) / alike)
    slower = np.array(taken)
    stated = (len(taken), sum(apart), geometric(taken), geometric(best), (slower > 1.03).sum(), (slower > 1.05).sum(), slower.max())
    assert len(taken) == 1500 and 480 < sum(apart) < 500, stated
    assert geometric(taken) < 0.978 and geometric(best) > 0.969, stated  # fitted: 0.9771, 0.9693
    assert (slower > 1.03).sum() <= 15 and (slower > 1.05).sum() <= 7 and slower.max() < 1.1, stated
