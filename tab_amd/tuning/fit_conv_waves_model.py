"""Coefficients of the rule that takes a convolution with fp32 output to the kernel that splits K over the waves of a workgroup
(tab_conv_waves_model.h), from conv_waves_timings.txt: 1900 random layers and 800 of residual and other networks' sizes, of at most 5000 tiles of
32x32, that take two launches, as the tiled kernels
run them by their own choice ("tiled"; left out where that was their 32x32 shape, whose place this kernel takes) and in this kernel's shapes
19 .. 22.

A timing is that of a quantizer and the convolution behind it on three sets of inputs in turn, in HIP-graph replays of 18 such calls, less the
quantizer's alone ("quantizer").

Model, per (type, shape): duration ~ c . f, non-negative least squares of the relative error, with the features
    f = [1, steps, busy, n, n * G, load, load * G, rounds, Y, W, n * G * lines]
    load   = ceil(M / BM) * ceil(KN / BN) / CUs      workgroups a CU gets
    n      = ceil(load), busy = min(1, load)         the busiest CU's; the share of the CUs that have work at all
    rounds = ceil(n / workgroups a CU holds)
    steps  = words of K of the longest wave          its chain of loads, expansions and multiplications
    lines  = pixels of whole cache lines: a load's lanes then read the same bytes of different lines
    G      = KH*KW*PC words of K, Y = 4*M*KN bytes / 1e6, W = bytes of the weights / 1e6 (fetched from behind the L2s)
and for the tiled kernels, with the duration `us` that conv_mfma_shape predicts (fitted to convolutions replayed on the same operands)
    f = [1, us, Y, us * odd, G / 10, G / 10 * odd, W, Y * ragged, one, us * one]
    odd, one: an odd number of words a pixel, a single one; ragged: KN is no multiple of 32

    python tab_amd/tuning/fit_conv_waves_model.py            fit on everything, write the header
    python tab_amd/tuning/fit_conv_waves_model.py --check    fit on three quarters of the layers in turn, regret on the fourth
"""
import ctypes
import os
import re
import sys

import numpy as np
from scipy.optimize import nnls

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
DATA = os.path.join(HERE, "conv_waves_timings.txt")
HEADER = os.path.join(ROOT, "tab_amd", "csrc", "tab_conv_waves_model.h")
SHAPES = {19: (32, 32, 8, 4), 20: (32, 32, 4, 8), 21: (64, 32, 4, 4), 22: (32, 64, 4, 4)}  # kWavesTile
CUS, LIMIT_US, MARGIN = 256, 12.0, 0.98
ROUNDS, SLOWER = 4, 1.05


def parse(path=DATA):
    rows = []
    pattern = re.compile(r"type (\d) N(\d+)_(\d+)x(\d+)x(\d+)->(\d+)_k(\d+)_p(\d+)_s(\d+) \| (.*)")
    for line in open(path):
        m = pattern.match(line)
        if m:
            r = dict(zip(("type", "N", "H", "W", "C", "KN", "K", "p", "s"), map(int, m.groups()[:9])))
            r["M"] = r["N"] * ((r["H"] + 2 * r["p"] - r["K"] + 1) // r["s"]) * ((r["W"] + 2 * r["p"] - r["K"] + 1) // r["s"])
            r["PC"] = (r["C"] + 31) // 32 if r["type"] == 5 else (r["C"] + 63) // 64
            r["G"] = r["K"] * r["K"] * r["PC"]
            times = {k: float(v) for k, v in (t.split(":") for t in m.group(10).split())}
            r["quantizer"], r["tiled"] = times.pop("quantizer"), times.pop("tiled", None)
            r["times"] = {int(k): v for k, v in times.items()}
            rows.append(r)
    return rows


def common(r):
    return r["M"] * r["KN"] * 4e-6, r["KN"] * r["G"] * (16e-6 if r["type"] in (0, 2, 4) else 8e-6)


def features(r, shape):
    bm, bn, waves, held = SHAPES[shape]
    y, w = common(r)
    words = 2 if r["PC"] % 2 == 0 and r["type"] not in (0, 4) else 1
    units = -(-r["G"] // (2 * words))
    tiles = -(-r["M"] // bm) * -(-r["KN"] // bn)
    load, n = tiles / CUS, -(-tiles // CUS)
    lines = r["PC"] * (16 if r["type"] in (0, 1, 4) else 8) % 128 == 0
    return [1.0, -(-units // waves) * words, min(1.0, load), n, n * r["G"], load, load * r["G"], -(-n // held), y, w, n * r["G"] * lines]


def tiled_features(r, us):
    y, w = common(r)
    odd, one = r["PC"] % 2, float(r["PC"] == 1)
    return [1.0, us, y, us * odd, 0.1 * r["G"], 0.1 * r["G"] * odd, w, y * (r["KN"] % 32 != 0), one, us * one]


def tiled_choice(rows):
    f = ctypes.CDLL(os.path.join(ROOT, "tab_amd", "lib", "libtab_amd.so")).tab_internal_conv_shape
    f.argtypes = [ctypes.c_int] * 6 + [ctypes.POINTER(ctypes.c_float)]
    for r in rows:
        us = ctypes.c_float()
        r["shape"] = f(r["type"], r["M"], r["KN"], r["G"], r["PC"], 0, ctypes.byref(us))
        r["us"] = us.value


def fit_weighted(rows, emphasis):
    def solve(x, y, w):
        return nnls(np.array(x) / np.array(y)[:, None] * np.array(w)[:, None], np.array(w))[0]

    coefficients = {}
    for t in range(6):
        some = [(r, w) for r, w in zip(rows, emphasis) if r["type"] == t]
        for s in SHAPES:
            coefficients[t, s] = solve([features(r, s) for r, _ in some], [r["times"][s] for r, _ in some], [w for _, w in some])
        some = [(r, w) for r, w in some if r["tiled"] is not None]
        coefficients[t, "tiled"] = solve([tiled_features(r, r["us"]) for r, _ in some], [r["tiled"] for r, _ in some], [w for _, w in some])
    return coefficients


def fit(rows):
    """Calls that the choices slow down by more than SLOWER count threefold in the next of ROUNDS fits."""
    emphasis = np.ones(len(rows))
    for _ in range(ROUNDS):
        coefficients = fit_weighted(rows, emphasis)
        for i, r in enumerate(rows):
            c = choose(r, coefficients)
            if c != "tiled" and r["tiled"] is not None and r["quantizer"] + r["times"][c] > SLOWER * (r["quantizer"] + r["tiled"]):
                emphasis[i] *= 3
    return coefficients


def choose(r, coefficients):
    """The shape the rule takes, or "tiled"."""
    us = {s: float(coefficients[r["type"], s] @ np.array(features(r, s))) for s in SHAPES}
    best = min(us, key=us.get)
    if r["shape"] == 3:
        return best
    tiled = float(coefficients[r["type"], "tiled"] @ np.array(tiled_features(r, r["us"])))
    return best if us[best] < LIMIT_US and us[best] < MARGIN * tiled else "tiled"


def report(rows, choices, what):
    rows_choices = [(r, c) for r, c in zip(rows, choices) if r["tiled"] is not None]
    taken = [(r["quantizer"] + (r["tiled"] if c == "tiled" else r["times"][c])) / (r["quantizer"] + r["tiled"]) for r, c in rows_choices]
    best = [(r["quantizer"] + min(r["tiled"], *r["times"].values())) / (r["quantizer"] + r["tiled"]) for r, _ in rows_choices]
    other = [r["times"][c] / min(r["times"].values()) for r, c in zip(rows, choices) if r["tiled"] is None]
    print("%s: quantizer and convolution %.4f of the tiled kernels' (geometric), the better of each %.4f; %d of %d choices more than 2 %% slower, %d "
          "more than 5 %%, worst %.3f; in place of 32x32 tiles %.4f of the best shape's convolution, worst %.3f" %
          (what, np.exp(np.mean(np.log(taken))), np.exp(np.mean(np.log(best))), sum(t > 1.02 for t in taken), sum(c != "tiled" for _, c in rows_choices),
           sum(t > 1.05 for t in taken), max(taken), np.exp(np.mean(np.log(other))), max(other)))


def main():
    rows = parse()
    tiled_choice(rows)
    if "--check" in sys.argv:
        fold = np.random.RandomState(0).randint(0, 4, len(rows))
        choices = [None] * len(rows)
        for f in range(4):
            coefficients = fit([r for r, k in zip(rows, fold) if k != f])
            for i, r in enumerate(rows):
                if fold[i] == f:
                    choices[i] = choose(r, coefficients)
        report(rows, choices, "held out")
        return
    coefficients = fit(rows)
    report(rows, [choose(r, coefficients) for r in rows], "fitted")

    def row(c):
        return "{" + ", ".join("%.6gf" % v if "." in "%.6g" % v or "e" in "%.6g" % v else "%.6g.0f" % v for v in c) + "}"

    with open(HEADER, "w") as f:
        f.write("// Written by tab_amd/tuning/fit_conv_waves_model.py from conv_waves_timings.txt (%d layers): microseconds per feature\n"
                "// (waves_features, tiled features in conv_waves_or, tab_conv.hip), types 0..5.\n#pragma once\n\nnamespace tab {\n\n" % len(rows))
        f.write("constexpr float kWavesCost[6][kWavesShapes][kWavesFeatures] = {\n")
        for t in range(6):
            f.write("    {\n" + "".join("        %s,\n" % row(coefficients[t, s]) for s in SHAPES) + "    },\n")
        f.write("};\n\nconstexpr float kWavesTiledCost[6][kWavesTiledFeatures] = {\n" + "".join("    %s,\n" % row(coefficients[t, "tiled"]) for t in range(6)) + "};\n\n}  // namespace tab\n")


if __name__ == "__main__":
    main()
