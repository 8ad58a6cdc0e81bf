"""The convolution that keeps its input patch in LDS, host side: the patch the plan allots holds what every tile of the launch reads
(by brute force over the tiles), the workspace's room holds the weights of every plan, and the rule that takes a call there, on its
measured launches, is within what its comment states."""
import ctypes
import importlib.util
import itertools
import os
import random

import pytest

from tab_amd import _capi

TUNING = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tab_amd", "tuning")
ROWS = {12: 256, 13: 128, 14: 128, 15: 64, 16: 256, 17: 64, 18: 64}


@pytest.fixture(scope="module")
def lib():
    lib = ctypes.CDLL(_capi.LIB_PATH)
    lib.tab_internal_conv_patch_shape.argtypes = [ctypes.c_int] * 12 + [ctypes.POINTER(ctypes.c_int), ctypes.POINTER(ctypes.c_size_t)]
    for f in (lib.tab_conv2d_workspace_bytes_full, lib.tab_conv2d_workspace_bytes, lib.tab_layer_workspace_bytes_full, lib.tab_layer_workspace_bytes):
        f.restype = ctypes.c_size_t
    yield lib
    lib.tab_set_conv_kernel(0, -1)


def plan(lib, type, p1, p2, s1, s2, N, H, W, C, KN, KH, KW):
    what, size = (ctypes.c_int * 3)(), ctypes.c_size_t()
    shape = lib.tab_internal_conv_patch_shape(type, p1, p2, s1, s2, N, H, W, C, KN, KH, KW, what, ctypes.byref(size))
    return shape, what[0], what[1], what[2], size.value


def test_every_tile_fits_its_patch_and_every_plan_its_room(lib):
    rng, planned = random.Random(3), 0
    for _ in range(4000):
        KH, KW, s1, s2 = rng.randint(1, 7), rng.randint(1, 7), rng.choice((1, 1, 2, 3, 9)), rng.choice((1, 1, 2, 3))
        p1, p2 = rng.randint(0, KH), rng.randint(0, KW)
        H, W = rng.randint(max(1, KH - 2 * p1), 40), rng.randint(max(1, KW - 2 * p2), 60)
        N, C, KN, type = rng.randint(1, 12), rng.choice((3, 64, 100, 128, 192, 256, 320, 448, 512, 1000)), rng.randint(1, 300), rng.randint(0, 4)
        OH, OW = (H + 2 * p1 - KH + 1) // s1, (W + 2 * p2 - KW + 1) // s2
        if OH < 1 or OW < 1:
            continue
        shape = rng.choice(tuple(ROWS))
        lib.tab_internal_force_patch(shape)
        got, kc, npix, lds, weights = plan(lib, type, p1, p2, s1, s2, N, H, W, C, KN, KH, KW)
        if got < 0:
            continue
        assert got == shape
        planned += 1
        PH, PW, PC = (OH - 1) * s1 + KH, (OW - 1) * s2 + KW, (C + 63) // 64
        line = lambda m: m // (OH * OW) * PH + m % (OH * OW) // OW * s1  # noqa: E731
        M, rows = N * OH * OW, ROWS[shape]
        need = max((line(min(m0 + rows, M) - 1) + KH - line(m0)) * PW for m0 in range(0, M, rows))
        chunks = -(-PC // kc)
        assert need + (kc == 1) <= npix <= (2 if kc == 4 else 3) * 256 + (kc == 1)
        assert npix * 32 * kc * (2 if chunks > 1 else 1) <= lds <= 64 * 1024
        planes = 2 if type in (0, 2, 4) else 1
        pairs = (KH * KW + 1) // 2 if kc == 1 else KH * KW * kc // 2
        assert weights == -(-KN // 32) * chunks * pairs * 512 * planes
        a = (type, N, H, W, C)
        if KH * KW > 1:
            assert lib.tab_conv2d_workspace_bytes_full(*a, KN, KH, KW) >= lib.tab_conv2d_workspace_bytes(*a) + weights + 15
            if type < 4:
                bits = 2 if type < 2 else 1
                assert lib.tab_layer_workspace_bytes_full(*a, KN, KH, KW) >= lib.tab_layer_workspace_bytes(bits, N, H, W, C) + weights + 15
    assert planned > 1500


def test_sizes_of_refused_arguments(lib):
    assert lib.tab_conv2d_workspace_bytes_full(7, 1, 1, 1, 1, 1, 3, 3) == 0 and lib.tab_conv2d_workspace_bytes_full(0, 1, 1, 1, 1, 0, 3, 3) == 0
    assert lib.tab_layer_workspace_bytes_full(4, 1, 1, 1, 1, 1, 3, 3) == 0
    for type in range(6):  # one tap, or type 5: no room beyond the packed activation
        KH = 1 if type < 5 else 3
        assert lib.tab_conv2d_workspace_bytes_full(type, 2, 9, 9, 100, 64, KH, KH) == lib.tab_conv2d_workspace_bytes(type, 2, 9, 9, 100)


def test_the_front_end_asks_for_the_room_of_the_plan(lib):
    """tab_internal_conv_plan, what the PyTorch front end allocates by: the weights' room where the rule takes a call to this kernel, else
    none (the room of every plan for every call moved the blocks of the calls behind it, which then ran slower)."""
    lib.tab_set_conv_kernel(0, -1)
    lib.tab_internal_conv_plan.restype, plan_of = ctypes.c_size_t, (ctypes.c_byte * 64)()
    seen = set()
    for type in range(6):
        for N in (1, 16, 36, 256):
            for H, C, KN, KH, p, s in ((56, 64, 64, 3, 1, 1), (28, 128, 128, 3, 1, 1), (14, 256, 256, 3, 1, 1), (7, 512, 512, 3, 1, 1),
                                       (56, 64, 128, 3, 1, 2), (56, 64, 128, 1, 0, 2), (40, 100, 75, 5, 2, 1), (9, 64, 64, 11, 0, 1)):
                a = (type, p, p, s, s, N, H, H, C, KN, KH, KH)
                shape, _, _, _, weights = plan(lib, *a)
                assert lib.tab_internal_conv_plan(*a, plan_of) == (weights + 16 if shape >= 0 else 0), a
                assert ctypes.c_int.from_buffer(plan_of).value == shape
                seen.add(shape >= 0)
    assert seen == {False, True}


def test_the_rule_on_its_measured_calls(lib):
    """The compiled choices (256 compute units where no device is present) against the calls without this kernel, whole calls: the script's
    own choices, with the figures that its fit states, and none beyond."""
    spec = importlib.util.spec_from_file_location("fit", os.path.join(TUNING, "fit_conv_patch_model.py"))
    fit = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(fit)
    lib.tab_set_conv_kernel(0, -1)
    rows = [r for r in fit.parse(fit.DATA) if fit.eligible(r)]
    assert len(rows) > 11000
    chosen = []
    for r in rows:
        shape, kc, npix, lds, _ = plan(lib, r["type"], r["p1"], r["p2"], r["s"], r["s"], r["N"], r["H"], r["W"], r["C"], r["KN"], r["KH"], r["KW"])
        if shape >= 0:
            assert fit.patch_features(r, shape) is not None and fit.chunk(r, shape) == (kc, npix, lds), r
        chosen.append(shape if shape >= 0 else None)
    geometric, total, _, _, each, missed = fit.regret(rows, chosen)
    stated = fit.stated(rows, chosen)
    # (to the last digit of what the script prints: float arithmetic may turn a call or two on the border)
    assert geometric < 0.9438 and total < 0.9140 and each.max() < 1.18, stated
    assert (each > 1.02).sum() <= 151 and (each > 1.05).sum() <= 35 and (each > 1.08).sum() <= 18, stated
    assert (missed > 1.05).sum() <= 483 and (missed > 1.1).sum() <= 114, stated
    assert len({c for c in chosen if c is not None}) == len(ROWS), stated  # every shape has launches of its own
    # launches of fewer tiles than compute units are not looked at
    assert plan(lib, 0, 1, 1, 1, 1, 16, 14, 14, 256, 256, 3, 3)[0] < 0 and plan(lib, 0, 1, 1, 1, 1, 64, 14, 14, 256, 256, 3, 3)[0] >= 0


def test_a_plan_without_its_room_leaves_the_kernel_of_calls_without_any(lib):
    """PatchPlan.tiled, what runs where the workspace cannot hold the weights: the kernel that launch_conv takes."""
    lib.tab_set_conv_kernel(0, -1)
    lib.tab_internal_conv_plan.restype, plan_of = ctypes.c_size_t, (ctypes.c_int * 16)()
    planned, split = 0, 0
    for type in range(5):
        for N, H, C, KN, K in itertools.product((12, 20, 28, 36, 50, 64, 100, 256), (9, 11, 14, 18, 20, 28), (64, 128, 192, 320, 512), (64, 128, 192, 256, 320, 512), (3, 5)):
            lib.tab_internal_conv_plan(type, K // 2, K // 2, 1, 1, N, H, H, C, KN, K, K, plan_of)
            if plan_of[0] < 0:
                continue
            PC = (C + 63) // 64
            want = lib.tab_internal_conv_launch_shape(type, N * H * H, KN, K * K * PC, PC, 0)
            assert plan_of[4] == want, (type, N, H, C, KN, K)
            planned, split = planned + 1, split + (want >= 19)
    assert planned > 1000 and split >= 20, (planned, split)
