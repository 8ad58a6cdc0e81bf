"""Coefficients of the rule that takes a convolution from fp32 to the kernel that keeps its input patch in LDS
(tab_conv_patch_model.h), from conv_patch_timings.txt: whole calls, quantizer and convolution, of random layers of at least 256 tiles of
64x64, as the tiled kernels run them by their own choice ("tiled") and in the patch kernel's shapes 12 .. 18.

A timing is the mean of two, of calls that follow each other on three sets of inputs and of calls with a copy of 48 MB behind each,
which empties the L2s.  The convolution alone, replayed on the same operands, is no measure of this kernel: its weights are laid out by
the quantizer's launch, and where the convolution's waves fetch them for the first time they come from behind the L2s, two pairs of
words ahead, which a long K waits for (N=64 7x7x512->512 ternary 11.0 us replayed, 15.1 behind its quantizer; the tiled kernel 11.4
and 12.4).

All calls of a layer have the quantizer in common, so the fit is one of differences: non-negative least squares of what the tiled kernel
and every shape take beyond the best of them, over the tiled kernel's time, all kernels of a type at once, small differences weighing
more.  The durations themselves, with the quantizer's as a form in bytes, join in at a tenth of the weight, which gives the predictions
their scale; they are the convolution's up to a summand that all share.

All times are of one session.  "waves": the kernel that splits K over waves, where its rule takes the call from the tiled ones.  Where
conv_mfma_shape ranks 32x32 tiles first there is no tiled kernel and the patch is not looked at; elsewhere the choice is between the two as
conv_patch_plan makes it.

    python tab_amd/tuning/fit_conv_patch_model.py            fit on everything, write the header
    python tab_amd/tuning/fit_conv_patch_model.py --check    fit on two thirds of the geometries, regret on the other third
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
MARGIN, MARGIN_US = 0.985, 0.1  # what the patch kernel has to be predicted below: MARGIN of the tiled kernel's duration, less MARGIN_US
PATCH_FEATURES, TILED_FEATURES = 26, 32  # kPatchFeatures, kTiledFeatures
TILED_SHAPES = (0, 1, 2, 4, 5, 6, 8, 9, 10, 11)  # kTiledShapes
BORDER, SCALE = 0.1, 0.1  # a difference of the share BORDER of a call weighs 0.7 of one that is none; a duration SCALE


def parse(path):
    rows = []
    pattern = re.compile(r"type (\d) N(\d+)_(\d+)x(\d+)x(\d+)->(\d+)_k(\d+)x(\d+)_p(\d+)\.(\d+)_s(\d+) \| (.*)")
    for line in open(path):
        m = pattern.match(line)
        if m:
            r = dict(zip(("type", "N", "H", "W", "C", "KN", "KH", "KW", "p1", "p2", "s"), map(int, m.groups()[:11])))
            r["OH"], r["OW"] = (r["H"] + 2 * r["p1"] - r["KH"] + 1) // r["s"], (r["W"] + 2 * r["p2"] - r["KW"] + 1) // r["s"]
            r["M"], r["PC"] = r["N"] * r["OH"] * r["OW"], (r["C"] + 63) // 64
            r["G"], r["planes"] = r["KH"] * r["KW"] * r["PC"], 2 if r["type"] in (0, 2, 4) else 1
            times = dict(t.split(":") for t in m.group(12).split())
            r["tiled"], r["waves"] = (float(times.pop(k, "nan")) for k in ("tiled", "waves"))
            r["without"] = r["tiled"] if np.isnan(r["waves"]) else r["waves"]  # the call without the patch kernel
            r["times"] = {int(k): float(v) for k, v in times.items()}  # (those above 1.7 times the tiled kernel's were left out)
            rows.append(r)
    return rows


def eligible(r):
    """The launches the rule looks at."""
    return r["type"] <= 4 and r["G"] > r["PC"] and r["KN"] > 32 and (r["M"] + 63) // 64 * ((r["KN"] + 63) // 64) >= CUS


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
    x = r["N"] * r["H"] * r["W"] * r["PC"] * (16e-6 if r["type"] in (0, 1, 4) else 8e-6)
    taps, chunks = r["KH"] * r["KW"], -(-r["PC"] // kc)
    pairs = chunks * ((taps + 1) // 2 if kc == 1 else taps * kc // 2)
    K = 2 * pairs
    down, across = -(-r["M"] // rows), -(-r["KN"] // filters)
    tiles, load = down * across, down * across / CUS
    held = min(held, 160 * 1024 // lds)
    n = -(-tiles // CUS)
    rounds, busy, y = -(-n // held), min(1.0, tiles / CUS), r["M"] * r["KN"] * 4e-6
    patch = npix * kc * chunks * 1e-3
    weights = -(-r["KN"] // 32) * pairs * 512e-6 * r["planes"]
    ragged, uncached = r["KN"] % 32 != 0, r["M"] * r["KN"] < 6 << 20
    beyond = max(0.0, y - 256)
    return np.array([1, busy, K * n, K * rounds, n, rounds, y, y * busy, patch * n, patch * rounds, chunks * rounds, tiles / CUS,
                     y * ragged, weights, 0.01 * pairs, r["PC"] == 1, y * (r["PC"] == 1), y * (ragged and uncached), beyond, beyond * ragged,
                     weights / max(1, load), K * load, patch * load, chunks * load, x * across, 0.01 * weights * down])


def tiled_prediction():
    lib = ctypes.CDLL(os.path.join(os.path.dirname(HERE), "lib", "libtab_amd.so"))
    f = lib.tab_internal_conv_shape
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_int] * 6 + [ctypes.POINTER(ctypes.c_float)]

    def predict(r, shape=False):
        cost = ctypes.c_float()
        chosen = f(r["type"], r["M"], r["KN"], r["G"], r["PC"], 0, ctypes.byref(cost))
        return chosen if shape else cost.value

    return predict


def waves_gain(r):
    f = ctypes.CDLL(os.path.join(os.path.dirname(HERE), "lib", "libtab_amd.so")).tab_internal_conv_waves_gain
    f.restype = ctypes.c_float
    return f(r["type"], r["M"], r["KN"], r["G"], r["PC"])


def tiled_features(r, us, shape):
    y, odd, one = r["M"] * r["KN"] * 4e-6, r["PC"] % 2, r["PC"] == 1
    ragged, cached, beyond = r["KN"] % 32 != 0, r["M"] * r["KN"] >= 6 << 20, max(0.0, y - 256)
    pairs = r["PC"] % 4 == 2 and r["G"] % 6 != 0
    products = r["M"] * (-(-r["KN"] // 64) * 64) * r["G"] * 1e-9
    return np.array([1, us, y, products, odd * products, odd * us, 0.1 * r["G"], odd * 0.1 * r["G"], r["M"] * r["G"] * 1e-6,
                     y * ragged, r["KN"] * r["G"] * r["planes"] * 8e-6, one, us * one, y * (one and ragged and cached), us * pairs, 0.1 * r["G"] * pairs,
                     beyond, beyond * ragged, beyond * one, beyond * (ragged and one), y * (ragged and not cached),
                     max(0.0, y - 12) * (ragged and not cached and shape != 2)] + [us * (shape == s) for s in TILED_SHAPES])


def quantizer_features(r):
    x, ragged = r["N"] * r["H"] * r["W"] * r["C"] * 4e-6, r["C"] % 64 != 0
    return np.array([1, x, x * ragged, ragged, r["N"] * r["H"] * r["W"] * r["PC"] * 8e-6 * (2 if r["type"] in (0, 1, 4) else 1)])


def prepared(rows):
    """The forms of every row, worked out once."""
    predict = tiled_prediction()
    for r in rows:
        shape = predict(r, True)
        r["tiled form"] = None if shape == 3 else tiled_features(r, predict(r), shape)
        r["forms"] = {s: patch_features(r, s) for s in SHAPES}
        r["waves gain"] = waves_gain(r)
    return rows


def fit(rows):
    tiled, patch = {}, {}
    at = {s: TILED_FEATURES + k * PATCH_FEATURES for k, s in enumerate(SHAPES)}
    quantizer = TILED_FEATURES + len(SHAPES) * PATCH_FEATURES
    for t in range(5):
        A, b = [], []
        for r in rows:
            if r["type"] != t or r["tiled form"] is None:
                continue
            kernels = []  # (duration, its form)
            for s in [None] + [s for s in SHAPES if s in r["times"] and r["forms"][s] is not None]:
                form = np.zeros(quantizer + 5)
                if s is None:
                    form[:TILED_FEATURES] = r["tiled form"]
                else:
                    form[at[s]:at[s] + PATCH_FEATURES] = r["forms"][s]
                kernels.append((r["tiled"] if s is None else r["times"][s], form))
            best = min(range(len(kernels)), key=lambda i: kernels[i][0])
            for i, (us, form) in enumerate(kernels):
                if i != best:
                    difference = (us - kernels[best][0]) / r["tiled"]
                    weight = (1 + (difference / BORDER) ** 2) ** -0.5
                    A.append(weight * (form - kernels[best][1]) / r["tiled"])
                    b.append(weight * difference)
                whole = form.copy()
                whole[quantizer:] = quantizer_features(r)
                A.append(SCALE * whole / us)
                b.append(SCALE)
        x = nnls(np.array(A), np.array(b), maxiter=50000)[0]
        tiled[t] = x[:TILED_FEATURES]
        for s in SHAPES:
            patch[t, s] = x[at[s]:at[s] + PATCH_FEATURES]
    return tiled, patch


def choose(r, tiled, patch):
    tiles = -(-r["M"] // 64) * -(-r["KN"] // 64)
    if r["tiled form"] is None or (r["G"] > 192 and (r["KN"] > 256 or r["G"] > 448) and tiles < CUS * (1 + r["G"] / 512)):
        return None
    call = float(tiled[r["type"]] @ r["tiled form"])
    limit, best = MARGIN * call - MARGIN_US, None
    wide = r["KN"] > 64 and r["M"] * r["KN"] * 4e-6 > 150
    for s in SHAPES:
        f = r["forms"][s]
        if f is not None and not (s == 15 and wide) and float(patch[r["type"], s] @ f) < limit:
            limit, best = float(patch[r["type"], s] @ f), s
    return best if best and r["waves gain"] <= call - limit else None


def regret(rows, chosen):
    """(geometric mean, total) of the chosen and of the best times over those without the patch kernel, and every choice's."""
    without = np.array([r["without"] for r in rows])
    got = np.array([r["without"] if c is None else r["times"].get(c, 1.7 * r["without"]) for r, c in zip(rows, chosen)])
    best = np.array([min([r["without"]] + list(r["times"].values())) for r in rows])
    return np.exp(np.log(got / without).mean()), got.sum() / without.sum(), np.exp(np.log(best / without).mean()), best.sum() / without.sum(), got / without, got / best


def stated(rows, chosen):
    geometric, total, best_geometric, best_total, each, missed = regret(rows, chosen)
    return ("chosen / without %.4f (geometric) %.4f (total), best %.4f %.4f; %d of %d in the patch kernel, more than 2 / 5 / 8 %% slower there "
            "%d / %d / %d, worst %.3f; more than 5 / 10 %% above the best %d / %d" % (
                geometric, total, best_geometric, best_total, sum(c is not None for c in chosen), len(rows), (each > 1.02).sum(),
                (each > 1.05).sum(), (each > 1.08).sum(), each.max(), (missed > 1.05).sum(), (missed > 1.1).sum()))


def write_header(tiled, patch):
    def rows_of(values):
        return ", ".join("%.5gf" % v if v != int(v) else "%d.f" % v for v in values)

    with open(os.path.join(CSRC, "tab_conv_patch_model.h"), "w") as f:
        f.write("// Written by tab_amd/tuning/fit_conv_patch_model.py from conv_patch_timings.txt: microseconds up to a summand that both sides\n"
                "// share, linear in the terms of patch_durations and in tiled_features (tab_conv_patch.h), per type 0 .. 4 and, for the patch\n"
                "// kernel, shape 12 .. 18.\n"
                "#pragma once\n#include \"tab_conv_patch.h\"\n\nnamespace tab {\n\n")
        f.write("constexpr float kTiledCost[5][kTiledFeatures] = {\n" + "".join("    {%s},\n" % rows_of(tiled[t]) for t in range(5)) + "};\n\n")
        f.write("// (a row per feature, its columns the shapes and a last one of zeros: the host adds the shapes' sums up side by side)\n"
                "constexpr float kPatchCost[5][kPatchFeatures][kPatchColumns] = {\n")
        for t in range(5):
            f.write("    {\n" + "".join("        {%s, 0.f},\n" % rows_of([patch[t, s][k] for s in SHAPES]) for k in range(PATCH_FEATURES)) + "    },\n")
        f.write("};\n\n}  // namespace tab\n")


if __name__ == "__main__":
    data = prepared([r for r in parse(DATA) if eligible(r)])
    if "--check" in sys.argv:
        part = [(7 * r["N"] + 3 * r["H"] + 5 * r["W"] + 11 * r["C"] + r["KN"]) % 3 for r in data]
        fitted = [fit([r for r, x in zip(data, part) if x != h]) for h in range(3)]
        print("held out:", stated(data, [choose(r, *fitted[h]) for r, h in zip(data, part)]))
    else:
        fitted = fit(data)
        write_header(*fitted)
        print(stated(data, [choose(r, *fitted) for r in data]))
