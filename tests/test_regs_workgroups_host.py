"""How many workgroups a CU holds of a packed layer of short K, on the host: the library's choices on measured layers, with the regret that the
rule's comment states."""
import ctypes
import os
import re

import numpy as np

from tab_amd import _capi

TIMINGS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tab_amd", "tuning", "regs_workgroups_timings.txt")


def on_cu(*args):
    return ctypes.CDLL(_capi.LIB_PATH).tab_internal_regs_on_cu(*args)


def test_choices_on_the_measured_layers():
    chosen, best = [], []
    for line in open(TIMINGS):
        m = re.match(r"type (\d) planes (\d) \S+ G (\d) tiles (\d+) columns (\d+) fit (\d) \| (.*)", line)
        if m:
            type, planes, G, tiles, columns, fit = map(int, m.groups()[:6])
            times = {n: float(us) for n, us in (t.split(":") for t in m.group(7).split())}
            two = type == 3 and planes == 1 and G == 4 and fit == 3  # (the kernel's own limit)
            n = on_cu(G, tiles, columns, 2 if two else fit, 256)
            all_of_them = times["all"]
            chosen.append(times[str(n)] / all_of_them)
            best.append(min(times.values()) / all_of_them)
    chosen = np.array(chosen)
    stated = len(chosen), np.exp(np.log(chosen).mean()), np.exp(np.log(best).mean()), (chosen > 1.03).sum(), chosen.max()
    assert len(chosen) == 819 and stated[1] < 0.9675 and stated[2] > 0.957 and stated[3] <= 7 and stated[4] < 1.06, stated


def test_rounds_of_fewer_waves():
    """Layers that took 1.1 to 1.3 times as long when one more workgroup had come to fit."""
    for tiles, columns, fit in ((3621, 1, 4), (6272, 2, 3), (4688, 2, 3), (4752, 4, 3), (14452, 1, 4)):
        assert on_cu(4, tiles, columns, fit, 256) < fit


def test_any_sizes():
    for G in (1, 2, 4, 8, 9):
        for tiles in (1, 3, 1023, 1024, 1025, 2**26):
            for columns in (1, 2, 7, 65535):
                for most in range(1, 9):
                    for cus in (1, 256):
                        assert min(2, most) <= on_cu(G, tiles, columns, most, cus) <= most
