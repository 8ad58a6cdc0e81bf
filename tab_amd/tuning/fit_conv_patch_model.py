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

The tiled kernel has become faster since for odd numbers of words a pixel; the fit takes its later times (conv_patch_tiled_timings.txt).

Where conv_mfma_shape ranks 32x32 tiles first, the kernel that splits K over waves ran in their place ("tiled"): the patch was never faster.

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
TILED = os.path.join(HERE, "conv_patch_tiled_timings.txt")  # later times of the tiled kernel, where it has become faster
SHAPES = {12: (256, 128, 8, 2), 13: (128, 128, 4, 3), 14: (128, 64, 2, 4), 15: (64, 64, 1, 4), 16: (256, 64, 4, 3),
          17: (64, 256, 4, 3), 18: (64, 128, 2, 4)}  # kPatchTile
CUS, ITEMS, LDS = 256, {1: 3, 2: 3, 4: 2}, 64 * 1024
MARGIN, MARGIN_US = 0.985, 0.1  # what the patch kernel has to be predicted below: MARGIN of the tiled kernel's duration, less MARGIN_US
PATCH_FEATURES, TILED_FEATURES = 18, 14  # kPatchFeatures, kTiledFeatures
ROUNDS, SLOWER = 5, 1.05
BORDER, SCALE = 0.1, 0.1  # a difference of the share BORDER of a call weighs 0.7 of one that is none; a duration SCALE


def key(r):
    return tuple(r[k] for k in ("type", "N", "H", "W", "C", "KN", "KH", "KW", "p1", "p2", "s"))


def parse(path):
    rows, later = [], {} if path == TILED else {key(r): r["tiled"] for r in parse(TILED)}
    pattern = re.compile(r"type (\d) N(\d+)_(\d+)x(\d+)x(\d+)->(\d+)_k(\d+)x(\d+)_p(\d+)\.(\d+)_s(\d+) \| (.*)")
    for line in open(path):
        m = pattern.match(line)
        if m:
            r = dict(zip(("type", "N", "H", "W", "C", "KN", "KH", "KW", "p1", "p2", "s"), map(int, m.groups()[:11])))
            r["OH"], r["OW"] = (r["H"] + 2 * r["p1"] - r["KH"] + 1) // r["s"], (r["W"] + 2 * r["p2"] - r["KW"] + 1) // r["s"]
            r["M"], r["PC"] = r["N"] * r["OH"] * r["OW"], (r["C"] + 63) // 64
            r["G"], r["planes"] = r["KH"] * r["KW"] * r["PC"], 2 if r["type"] in (0, 2, 4) else 1
            times = dict(t.split(":") for t in m.group(12).split())
            r["tiled"] = float(times.pop("tiled"))
            r["now"] = min(r["tiled"], later.get(key(r), r["tiled"]))
            r["times"] = {int(k): float(v) for k, v in times.items()}  # (those above 1.5 times the tiled kernel's were left out)
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
    taps, chunks = r["KH"] * r["KW"], -(-r["PC"] // kc)
    pairs = chunks * ((taps + 1) // 2 if kc == 1 else taps * kc // 2)
    K = 2 * pairs
    tiles = -(-r["M"] // rows) * -(-r["KN"] // filters)
    held = min(held, 160 * 1024 // lds)
    n = -(-tiles // CUS)
    rounds, busy, y = -(-n // held), min(1.0, tiles / CUS), r["M"] * r["KN"] * 4e-6
    patch = npix * kc * chunks * 1e-3
    weights = -(-r["KN"] // 32) * pairs * 512e-6 * r["planes"]
    ragged, uncached = r["KN"] % 32 != 0, r["M"] * r["KN"] < 6 << 20
    return np.array([1, busy, K * n, K * rounds, n, rounds, y, y * busy, patch * n, patch * rounds, chunks * rounds, tiles / CUS,
                     y * ragged, weights, 0.01 * pairs, r["PC"] == 1, y * (r["PC"] == 1), y * (ragged and uncached)])


def tiled_prediction():
    lib = ctypes.CDLL(os.path.join(os.path.dirname(HERE), "lib", "libtab_amd.so"))
    f = lib.tab_internal_conv_shape
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_int] * 6 + [ctypes.POINTER(ctypes.c_float)]

    def predict(r, shape=False):
        cost = ctypes.c_float()
        chosen = f(r["type"], r["M"], r["KN"], r["G"], r["PC"], 0, ctypes.byref(cost))
        return chosen if shape else cost.value

    return predict


def tiled_features(r, us):
    y, odd, one = r["M"] * r["KN"] * 4e-6, r["PC"] % 2, r["PC"] == 1
    ragged, cached = r["KN"] % 32 != 0, r["M"] * r["KN"] >= 6 << 20
    products = r["M"] * (-(-r["KN"] // 64) * 64) * r["G"] * 1e-9
    return np.array([1, us, y, products, odd * products, odd * us, 0.1 * r["G"], odd * 0.1 * r["G"], r["M"] * r["G"] * 1e-6,
                     y * ragged, r["KN"] * r["G"] * r["planes"] * 8e-6, one, us * one, y * (one and ragged and cached)])


def quantizer_features(r):
    x, ragged = r["N"] * r["H"] * r["W"] * r["C"] * 4e-6, r["C"] % 64 != 0
    return np.array([1, x, x * ragged, ragged, r["N"] * r["H"] * r["W"] * r["PC"] * 8e-6 * (2 if r["type"] in (0, 1, 4) else 1)])


def fit_weighted(rows, predict, emphasis):
    tiled, patch = {}, {}
    at = {s: TILED_FEATURES + k * PATCH_FEATURES for k, s in enumerate(SHAPES)}
    quantizer = TILED_FEATURES + len(SHAPES) * PATCH_FEATURES
    for t in range(5):
        A, b = [], []
        for r, emphasised in zip(rows, emphasis):
            if r["type"] != t:
                continue
            kernels = []  # (duration, its form)
            for s in [None] + [s for s in SHAPES if s in r["times"] and patch_features(r, s) is not None]:
                form = np.zeros(quantizer + 5)
                if s is None:
                    form[:TILED_FEATURES] = tiled_features(r, predict(r))
                else:
                    form[at[s]:at[s] + PATCH_FEATURES] = patch_features(r, s)
                kernels.append((r["now"] if s is None else r["times"][s], form))
            best = min(range(len(kernels)), key=lambda i: kernels[i][0])
            for i, (us, form) in enumerate(kernels):
                if i != best:
                    difference = (us - kernels[best][0]) / r["now"]
                    weight = (1 + (difference / BORDER) ** 2) ** -0.5 * emphasised
                    A.append(weight * (form - kernels[best][1]) / r["now"])
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


def fit(rows, predict):
    """Calls that the choices slow down by more than SLOWER count threefold in the next of ROUNDS fits."""
    emphasis = np.ones(len(rows))
    for _ in range(ROUNDS):
        fitted = fit_weighted(rows, predict, emphasis)
        each = regret(rows, [choose(r, *fitted, predict) for r in rows], "now")[4]
        emphasis[each > SLOWER] *= 3
    return fitted


def choose(r, tiled, patch, predict):
    if predict(r, True) == 3:
        return None
    limit, best = MARGIN * float(tiled[r["type"]] @ tiled_features(r, predict(r))) - MARGIN_US, None
    for s in SHAPES:
        f = patch_features(r, s)
        if f is not None and float(patch[r["type"], s] @ f) < limit:
            limit, best = float(patch[r["type"], s] @ f), s
    return best


def regret(rows, chosen, base="tiled"):
    """(geometric mean, total) of the chosen and of the best times over the tiled ones, and every choice's over the tiled one.
    base: the tiled kernel's times with the patch's ("tiled") or its later ones ("now")."""
    tiled = np.array([r[base] for r in rows])
    got = np.array([r["now"] if c is None else r["times"].get(c, 1.5 * r["now"]) for r, c in zip(rows, chosen)])
    best = np.array([min([r["now"]] + list(r["times"].values())) for r in rows])
    return np.exp(np.log(got / tiled).mean()), got.sum() / tiled.sum(), np.exp(np.log(best / tiled).mean()), best.sum() / tiled.sum(), got / tiled


def stated(rows, chosen, base="tiled"):
    geometric, total, best_geometric, best_total, each = regret(rows, chosen, base)
    return ("chosen / tiled %.3f (geometric) %.3f (total), best %.3f %.3f; %d of %d in the patch kernel, more than 2 / 5 / 8 %% slower there "
            "%d / %d / %d, worst %.3f" % (geometric, total, best_geometric, best_total, sum(c is not None for c in chosen), len(rows),
                                         (each > 1.02).sum(), (each > 1.05).sum(), (each > 1.08).sum(), each.max()))


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
    data, predicted = [r for r in parse(DATA) if eligible(r)], tiled_prediction()
    if "--check" in sys.argv:
        half = [(7 * r["N"] + 3 * r["H"] + 5 * r["W"] + 11 * r["C"] + r["KN"]) % 2 for r in data]
        for h in (0, 1):
            fitted = fit([r for r, x in zip(data, half) if x != h], predicted)
            held_out = [r for r, x in zip(data, half) if x == h]
            print("held out:", stated(held_out, [choose(r, *fitted, predicted) for r in held_out], "now"))
    else:
        fitted = fit(data, predicted)
        write_header(*fitted)
        for base in ("tiled", "now"):
            print(base + ":", stated(data, [choose(r, *fitted, predicted) for r in data], base))
