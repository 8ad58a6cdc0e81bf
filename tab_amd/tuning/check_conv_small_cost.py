"""What the cost that conv_small is chosen by (tab_conv_small.hip: SmallCost, kMostUs) is worth on conv_small_timings.txt.

Prints, per input layout, the median and the 90th percentile of the predicted duration's error against the measured one, and,
as a share of always taking two launches, the time of the calls under the rule and under the better choice of each; the same for
graph replays, where a launch costs the host nothing; and what other limits would give.  Last, the coefficients that non-negative
least squares on the relative error gives for the same three numbers (scipy).  Needs the built library and no GPU.

    python tab_amd/tuning/check_conv_small_cost.py"""
import ctypes
import os
import re

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
LIMIT_US = 6.3  # kMostUs


def parse(path):
    lib = ctypes.CDLL(os.path.join(os.path.dirname(HERE), "lib", "libtab_amd.so"))
    cost = (ctypes.c_float * 4)()
    rows = []
    for line in open(path):
        m = re.match(r"type (\d) (nhwc|nchw) N(\d+)_(\d+)x(\d+)x(\d+)->(\d+)_k(\d+)_p(\d+)_s(\d+) \| one:(\S+) two:(\S+) one_call:(\S+) two_calls:(\S+)", line)
        if not m:
            continue
        type, nchw = int(m[1]), m[2] == "nchw"
        N, H, W, C, KN, k, p, s = map(int, m.groups()[2:10])
        one, two, one_call, two_calls = map(float, m.groups()[10:])
        # (any address aligned for 16-byte loads: nothing is read)
        assert lib.tab_internal_conv_small_cost(type, ctypes.c_void_p(4096), int(nchw), N, H, W, C, KN, k, k, p, p, s, s, cost)
        rows.append(dict(type=type, nchw=nchw, N=N, H=H, W=W, C=C, KN=KN, k=k, p=p, s=s, one=one, two=two, one_call=one_call,
                         two_calls=two_calls, predicted=cost[0], passes=cost[1], pairs=cost[2], more=cost[3]))
    return rows


def column(rows, key):
    return np.array([r[key] for r in rows])


def shares(rows, one, two, limit=LIMIT_US):
    """Time under the rule and under the better choice of each case, as shares of always two launches."""
    a, b = column(rows, one), column(rows, two)
    return np.where(column(rows, "predicted") <= limit, a, b).sum() / b.sum(), np.minimum(a, b).sum() / b.sum()


def errors(rows):
    """|predicted / measured - 1| of the conv_small launch (rows whose graph holds that launch alone)."""
    rows = [r for r in rows if not (r["nchw"] and r["type"] < 2)]
    return np.abs(column(rows, "predicted") / column(rows, "one") - 1)


def main():
    rows = parse(os.path.join(HERE, "conv_small_timings.txt"))
    for name, some in (("NHWC", [r for r in rows if not r["nchw"]]), ("NCHW", [r for r in rows if r["nchw"]]), ("all", rows)):
        e = errors(some)
        print("%-4s %d cases, error median %.1f %%, 90th percentile %.1f %%; calls %.1f %% of two launches' (best choices %.1f), graph replays %.1f %% (%.1f)"
              % (name, len(some), 100 * np.median(e), 100 * np.quantile(e, 0.9), *(100 * v for v in shares(some, "one_call", "two_calls")),
                 *(100 * v for v in shares(some, "one", "two"))))
    for limit in (5.0, 5.5, 6.0, 6.3, 6.6, 7.0, 8.0):
        print("limit %.1f us: calls %.1f %%, graph replays %.1f %%" % (limit, 100 * shares(rows, "one_call", "two_calls", limit)[0],
                                                                     100 * shares(rows, "one", "two", limit)[0]))
    from scipy.optimize import nnls

    some = [r for r in rows if not r["nchw"]]
    x = np.array([[1, r["passes"], r["pairs"], r["more"] * r["passes"], r["more"] * r["pairs"], r["more"]] for r in some])
    y = column(some, "one")
    c = nnls(x / y[:, None], np.ones(len(y)))[0]
    print("least squares (NHWC): %.2f + %.3f passes + %.3f pairs + more * (%.3f passes + %.3f pairs + %.2f), error median %.1f %%"
          % (*c, 100 * np.median(np.abs(x @ c / y - 1))))


if __name__ == "__main__":
    main()
