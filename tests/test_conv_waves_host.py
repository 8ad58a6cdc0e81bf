"""The rule that takes a convolution to the kernel that splits K over waves, on the host: the library's choices on the measured layers are the
fit script's, with the regret that its comment states."""
import ctypes
import importlib.util
import os

import numpy as np

from tab_amd import _capi

SCRIPT = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tab_amd", "tuning", "fit_conv_waves_model.py")


def test_choices_on_the_measured_layers():
    spec = importlib.util.spec_from_file_location("fit_conv_waves_model", SCRIPT)
    fit = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(fit)
    rows = fit.parse()
    assert len(rows) >= 2700
    fit.tiled_choice(rows)
    coefficients = fit.fit(rows)
    f = ctypes.CDLL(_capi.LIB_PATH).tab_internal_conv_launch_shape
    differ, taken, best, alone = 0, [], [], []
    for r in rows:
        shape = f(r["type"], r["M"], r["KN"], r["G"], r["PC"], 0)
        assert shape in fit.SHAPES or shape == r["shape"] != 3
        differ += (shape if shape in fit.SHAPES else "tiled") != fit.choose(r, coefficients)
        if r["tiled"] is None:
            alone.append(r["times"][shape] / min(r["times"].values()))
        else:
            call = r["quantizer"] + r["tiled"]
            taken.append((r["quantizer"] + r["times"].get(shape, r["tiled"])) / call)
            best.append((r["quantizer"] + min(r["tiled"], *r["times"].values())) / call)
    assert differ <= 3  # (coefficients of six digits)
    assert np.exp(np.mean(np.log(taken))) < 0.945 and np.exp(np.mean(np.log(best))) > 0.92 and max(taken) < 1.05  # fitted: 0.9427, 0.9249, 1.045
    assert np.exp(np.mean(np.log(alone))) < 1.005


def test_packed_output_and_large_launches_stay_with_the_tiles():
    f = ctypes.CDLL(_capi.LIB_PATH).tab_internal_conv_launch_shape
    tiled = ctypes.CDLL(_capi.LIB_PATH).tab_internal_conv_shape
    for type in range(6):
        for M, KN, G, PC in ((2**31 - 600, 1, 9, 1), (2**31 - 600, 4096, 65535, 65535), (200704, 64, 9, 1)):
            assert f(type, M, KN, G, PC, 0) == tiled(type, M, KN, G, PC, 0, None), (type, M, KN, G, PC)
        # few tiles: the split kernel for fp32 output, never for packed
        for M, KN, G, PC in ((1, 1, 1, 1), (1, 4096, 65534, 65534), (196, 512, 72, 8), (784, 512, 72, 8)):
            assert 19 <= f(type, M, KN, G, PC, 0) <= 22, (type, M, KN, G, PC)
            assert f(type, M, KN, G, PC, 1) == tiled(type, M, KN, G, PC, 1, None) < 12, (type, M, KN, G, PC)


def test_large_launches_have_no_more_threads_than_a_launch_may():
    """A forced tile 3 on an output of 34 GB and more: eight waves a tile of 32x32 would be 2^32 threads."""
    f = ctypes.CDLL(_capi.LIB_PATH).tab_internal_conv_waves_shape
    threads = {19: (32, 32, 512), 20: (32, 32, 256), 21: (64, 32, 256), 22: (32, 64, 256)}
    for type in range(6):
        for M in (2**23, 2**28 - 32, 2**28, 2**28 + 2**27):
            for G, PC in ((1, 1), (9, 1), (72, 8), (575, 64), (4608, 512)):
                rows, filters, each = threads[f(type, M, 32, G, PC)]
                assert -(-M // rows) * -(-32 // filters) * each < 2**32, (type, M, G)
