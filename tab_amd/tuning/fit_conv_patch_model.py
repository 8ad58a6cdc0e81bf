"""Coefficients of the rule that takes a convolution to the kernel that keeps its input patch in LDS (tab_conv_patch_model.h), by
non-negative least squares of the relative error on conv_patch_timings.txt: the conv kernel alone, in graph replays, on random
packed operands, as the tiled kernels run it by their own choice ("tiled") and in the patch kernel's shapes 12 .. 18.

    python tab_amd/tuning/fit_conv_patch_model.py            fit on everything, write the header
    python tab_amd/tuning/fit_conv_patch_model.py --check    fit on one half of the geometries, regret on the other
"""
import ctypes
import os
import re
import sys

import numpy as np
from scipy.optimize import nnls

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "csrc")
DATA = os.path.join(HERE, "conv_patch_timings.txt")
SHAPES = {12: (256, 128, 8, 2), 13: (128, 128, 4, 3), 14: (128, 64, 2, 4), 15: (64, 64, 1, 4), 16: (256, 64, 4, 3),
          17: (64, 256, 4, 3), 18: (64, 128, 2, 4)}  # kPatchTile
CUS, ITEMS, LDS = 256, {1: 3, 2: 3, 4: 2}, 64 * 1024
MARGIN, NARROW_MARGIN, WEIGHTS_US = 0.93, 0.85, 0.5  # the weights' part of the quantizer's launch, measured 0.1-0.8 us


def parse(path):
    rows = []
    pattern = re.compile(r"type (\d) N(\d+)_(\d+)x(\d+)x(\d+)->(\d+)_k(\d+)x(\d+)_p(\d+)\.(\d+)_s(\d+) \| (.*)")
    for line in open(path):
        m = pattern.match(line)
        if m:
            r = dict(zip(("type", "N", "H", "W", "C", "KN", "KH", "KW", "p1", "p2", "s"), map(int, m.groups()[:11])))
            r["OH"], r["OW"] = (r["H"] + 2 * r["p1"] - r["KH"] + 1) // r["s"], (r["W"] + 2 * r["p2"] - r["KW"] + 1) // r["s"]
            r["M"], r["PC"] = r["N"] * r["OH"] * r["OW"], (r["C"] + 63) // 64
            r["G"] = r["KH"] * r["KW"] * r["PC"]
            times = dict(t.split(":") for t in m.group(12).split())
            r["tiled"] = float(times.pop("tiled"))
            r["times"] = {int(k): float(v) for k, v in times.items()}
            rows.append(r)
    return rows


def eligible(r):
    """The launches the rule looks at."""
    return r["type"] <= 4 and r["G"] > r["PC"] and r["KN"] > 32 and (r["M"] + 63) // 64 * ((r["KN"] + 63) // 64) >= 128


def patch_pixels(r, rows):
    lines = (r["OW"] - np.gcd(r["OW"], rows) + rows - 1) // r["OW"] + 1
    crossings = (lines - 1 + r["OH"] - 1) // r["OH"]
    return int(((lines - 1) * r["s"] + crossings * max(0, r["KH"] - r["s"]) + r["KH"]) * ((r["OW"] - 1) * r["s"] + r["KW"]))


def chunk(r, shape):
    """(words of a chunk, pixels, LDS bytes) or None: patch_chunk of tab_conv_patch.h."""
    rows, _, tiles, _ = SHAPES[shape]
    pixels, kc = patch_pixels(r, rows), 1 if r["PC"] == 1 else (2 if tiles >= 8 else 4)
    while pixels <= ITEMS[1] * 256 and kc >= 1:
        if not ((kc == 4 and r["PC"] % 4 not in (0, 3)) or (kc == 2 and r["PC"] == 3)):
            planes = pixels + (kc == 1)
            size = planes * 32 * kc * (2 if r["PC"] > kc else 1)
            if size <= LDS and not (kc == 4 and pixels > ITEMS[4] * 256):
                return kc, planes, max(size, 4096)
        kc //= 2
    return None


def patch_features(r, shape):
    got = chunk(r, shape)
    if got is None or SHAPES[shape][1] >= 128 * ((r["KN"] + 63) // 64):
        return None
    kc, npix, lds = got
    rows, filters, _, held = SHAPES[shape]
    taps, chunks = r["KH"] * r["KW"], -(-r["PC"] // kc)
    K = chunks * ((taps + 1) // 2 * 2 if kc == 1 else taps * kc)
    tiles = -(-r["M"] // rows) * -(-r["KN"] // filters)
    held = min(held, 160 * 1024 // lds)
    n = -(-tiles // CUS)
    rounds, busy, y = -(-n // held), min(1.0, tiles / CUS), r["M"] * r["KN"] * 4e-6
    patch = npix * kc * chunks * 1e-3
    return np.array([1, busy, K * n, K * rounds, n, rounds, y, y * busy, patch * n, patch * rounds, chunks * rounds, tiles / CUS,
                     y if r["KN"] % 32 else 0])


def tiled_prediction():
    lib = ctypes.CDLL(os.path.join(os.path.dirname(HERE), "lib", "libtab_amd.so"))
    f = lib.tab_internal_conv_shape
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_int] * 6 + [ctypes.POINTER(ctypes.c_float)]

    def predict(r):
        cost = ctypes.c_float()
        f(r["type"], r["M"], r["KN"], r["G"], r["PC"], 0, ctypes.byref(cost))
        return cost.value

    return predict


def tiled_features(r, us):
    y, odd = r["M"] * r["KN"] * 4e-6, r["PC"] % 2
    products = r["M"] * (-(-r["KN"] // 64) * 64) * r["G"] * 1e-9
    return np.array([1, us, y, products, odd * products, odd * us, 0.1 * r["G"], odd * 0.1 * r["G"], r["M"] * r["G"] * 1e-6,
                     y if r["KN"] % 32 else 0])


def fit(rows, predict):
    tiled, patch = {}, {}
    for t in range(5):
        mine = [r for r in rows if r["type"] == t]
        A = np.array([tiled_features(r, predict(r)) / r["tiled"] for r in mine])
        tiled[t] = nnls(A, np.ones(len(A)))[0]
        for s in SHAPES:
            A = [patch_features(r, s) / r["times"][s] for r in mine if s in r["times"] and patch_features(r, s) is not None]
            patch[t, s] = nnls(np.array(A), np.ones(len(A)))[0]
    return tiled, patch


def choose(r, tiled, patch, predict):
    tiles64 = (r["M"] + 63) // 64 * ((r["KN"] + 63) // 64)
    margin = NARROW_MARGIN if 3 * CUS <= 2 * tiles64 <= 4 * CUS else MARGIN
    limit, best = margin * float(tiled[r["type"]] @ tiled_features(r, predict(r))), None
    for s in SHAPES:
        f = patch_features(r, s)
        if f is not None and WEIGHTS_US + float(patch[r["type"], s] @ f) < limit:
            limit, best = WEIGHTS_US + float(patch[r["type"], s] @ f), s
    return best


def regret(rows, chosen):
    """(geometric mean, total) of the chosen and of the best times over the tiled ones, and the worst choice."""
    got = np.array([r["tiled"] if c is None else r["times"][c] + WEIGHTS_US for r, c in zip(rows, chosen)])
    best, tiled = np.array([min([r["tiled"]] + [t + WEIGHTS_US for t in r["times"].values()]) for r in rows]), np.array([r["tiled"] for r in rows])
    return np.exp(np.log(got / tiled).mean()), got.sum() / tiled.sum(), np.exp(np.log(best / tiled).mean()), best.sum() / tiled.sum(), (got / tiled).max()


def write_header(tiled, patch):
    def rows_of(values):
        return ", ".join("%.5gf" % v if v != int(v) else "%d.f" % v for v in values)

    with open(os.path.join(CSRC, "tab_conv_patch_model.h"), "w") as f:
        f.write("// Written by tab_amd/tuning/fit_conv_patch_model.py from conv_patch_timings.txt: microseconds, linear in patch_features and\n"
                "// tiled_features (tab_conv_patch.h), per type 0 .. 4 and, for the patch kernel, shape 12 .. 18.\n#pragma once\n"
                "#include \"tab_conv_patch.h\"\n\nnamespace tab {\n\n")
        f.write("constexpr float kTiledCost[5][kTiledFeatures] = {\n" + "".join("    {%s},\n" % rows_of(tiled[t]) for t in range(5)) + "};\n\n")
        f.write("constexpr float kPatchCost[5][kPatchShapes][kPatchFeatures] = {\n")
        for t in range(5):
            f.write("    {\n" + "".join("        {%s},\n" % rows_of(patch[t, s]) for s in SHAPES) + "    },\n")
        f.write("};\n\n}  // namespace tab\n")


if __name__ == "__main__":
    data, predicted = [r for r in parse(DATA) if eligible(r)], tiled_prediction()
    if "--check" in sys.argv:
        half = [hash((r["N"], r["H"], r["W"], r["C"], r["KN"])) % 2 for r in data]
        for h in (0, 1):
            fitted = fit([r for r, x in zip(data, half) if x != h], predicted)
            held_out = [r for r, x in zip(data, half) if x == h]
            print("held out %d: chosen / tiled %.3f (geometric) %.3f (total), best %.3f %.3f, worst choice %.2f" % (
                (len(held_out),) + regret(held_out, [choose(r, *fitted, predicted) for r in held_out])))
    else:
        fitted = fit(data, predicted)
        write_header(*fitted)
        print("all %d: chosen / tiled %.3f (geometric) %.3f (total), best %.3f %.3f, worst choice %.2f" % (
            (len(data),) + regret(data, [choose(r, *fitted, predicted) for r in data])))
