"""The convolution that keeps its input patch in LDS, every shape forced on whole calls, layers (NHWC and NCHW) and packed activations,
against the tiled kernel of 64x64: chunks of one, two and four words, one and several of them, odd words per pixel, an odd number of taps,
tiles that span images and lines, rows past M, filters past a tile, strides, asymmetric padding, arbitrary weight bits."""
import ctypes

import pytest
import torch

import tab_amd
from tab_amd import _capi
from tab_amd import nn as tab_nn

pytestmark = pytest.mark.gpu

SHAPES = range(12, 19)
CASES = [
    # N, H, W, C, KN, KH, KW, p1, p2, s1, s2
    (2, 14, 14, 128, 64, 3, 3, 1, 1, 1, 1), (3, 7, 7, 64, 70, 3, 3, 1, 1, 1, 1), (2, 13, 11, 192, 130, 3, 3, 1, 0, 1, 1),
    (3, 9, 10, 256, 40, 5, 5, 2, 2, 2, 2), (1, 30, 31, 100, 75, 3, 3, 1, 1, 1, 1), (5, 6, 7, 320, 33, 2, 3, 0, 1, 1, 2),
    (9, 23, 23, 832, 49, 3, 3, 1, 1, 1, 1), (1, 56, 56, 64, 65, 3, 3, 1, 1, 1, 1), (2, 8, 12, 3, 35, 1, 7, 0, 3, 1, 1),
    (2, 17, 3, 448, 99, 3, 3, 1, 1, 2, 1), (7, 1, 9, 130, 31, 1, 2, 0, 1, 1, 1), (3, 20, 20, 70, 256, 3, 3, 2, 3, 3, 1),
]


@pytest.fixture(scope="module")
def lib():
    return ctypes.CDLL(_capi.LIB_PATH)


@pytest.fixture(autouse=True)
def automatic_kernel():
    yield
    tab_amd.set_conv_kernel()


def weights(type, g, KN, KH, KW, C):
    w = torch.randn((KN, KH, KW, C), device="cuda", generator=g)
    ths = tab_amd.Threshold(w, KN)
    if type == 4:
        return tab_amd.QuantizeFormat(w, ths, 4, KN, KH, KW, C), torch.zeros(KN, dtype=torch.int32, device="cuda")
    return tab_amd.Quantize(w, ths, 2 if type in (0, 2) else 1, KN, KH, KW, C)


def fitting(lib, type, sizes):
    """(the shape that the test hook holds, its weights' bytes) where the patch of these sizes fits it, else (-1, 0)."""
    what, size = (ctypes.c_int * 3)(), ctypes.c_size_t(0)
    shape = lib.tab_internal_conv_patch_shape(type, *sizes, what, ctypes.byref(size))
    return (shape, size.value) if shape >= 0 else (-1, 0)


def requested(call):
    """(the call's result, the most bytes it has asked the allocator for)."""
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_stats()["requested_bytes.all.current"]
    y = call()
    return y, torch.cuda.memory_stats()["requested_bytes.all.peak"] - before


@pytest.mark.parametrize("case", CASES)
def test_calls_and_layers(case, lib):
    """That the kernel ran shows in the memory a call asks for: room for its weights, which no other kernel is given, and only where the
    patch fits.  (The quantizer lays them out there exactly when this kernel follows; test_the_weights_are_laid_out_behind_the_activation.)"""
    N, H, W, C, KN, KH, KW, p1, p2, s1, s2 = case
    print(f"[case] patch {case}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(KN + C)
    x = torch.randn((N, H, W, C), device="cuda", generator=g)
    ths = tab_amd.Threshold(x, N)
    for type in range(5):
        QW, btn = weights(type, g, KN, KH, KW, C)
        run = lambda: tab_amd.Conv2d(x, QW, ths, btn, type, p1, p2, s1, s2, N, H, W, C, KN, KH, KW)  # noqa: E731
        layers = []
        if type < 4:
            w = torch.randn((KN, C, KH, KW), device="cuda", generator=g)
            for layout in ("NHWC", "NCHW"):
                layer = tab_nn.TABConv2d.from_float(w, type, (s1, s2), (p1, p2), data_format=layout)
                layers.append((layer, x if layout == "NHWC" else x.permute(0, 3, 1, 2).contiguous()))
        tab_amd.set_conv_kernel(tab_amd.CONV_MATRIX, 2)
        calls = [run] + [lambda layer=layer, a=a: layer(a) for layer, a in layers]
        want = [requested(call) for call in calls]
        for shape in SHAPES:
            lib.tab_internal_force_patch(shape)
            fits, room = fitting(lib, type, (p1, p2, s1, s2, N, H, W, C, KN, KH, KW))
            assert fits in (shape, -1)
            for call, (y, least) in zip(calls, want):
                z, more = requested(call)
                assert torch.equal(z, y), (type, shape)
                assert more == least + (room + 16 if fits == shape else 0), (type, shape)


@pytest.mark.parametrize("case", CASES)
def test_arbitrary_bits(case, lib):
    N, H, W, C, KN, KH, KW, p1, p2, s1, s2 = case
    print(f"[case] patch, arbitrary bits {case}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(KN + W)
    OH, OW = (H + 2 * p1 - KH + 1) // s1, (W + 2 * p2 - KW + 1) // s2
    bits = lambda *shape: torch.randint(-2**63, 2**63 - 1, shape, device="cuda", generator=g, dtype=torch.int64)  # noqa: E731
    room = torch.empty((((KN + 31) // 32) * ((KH * KW + 1) * ((C + 63) // 64 + 1) // 2 + 1) * 1024,), dtype=torch.uint8, device="cuda")
    fitted = 0
    for type in range(5):
        QX, QW = bits(N * H * W * tab_amd.operand_words(type, 0, C)), bits(KN * KH * KW * tab_amd.operand_words(type, 1, C))
        btn = torch.randint(0, 99, (KN,), device="cuda", generator=g, dtype=torch.int32)
        a = (QX, QW, btn, type, p1, p2, s1, s2, N, H, W, C, KN, KH, KW)
        tab_amd.set_conv_kernel(tab_amd.CONV_MATRIX, 2)
        want = tab_amd.Conv2dPacked(*a)
        for shape in SHAPES:
            lib.tab_internal_force_patch(shape)
            got = torch.empty_like(want)
            p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
            status = lib.tab_internal_conv_patch(p(QX), p(QW), p(btn), *a[3:], p(got), p(room), ctypes.c_size_t(room.numel()), 3,
                                                 ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
            if status == 0:  # (else the patch does not fit LDS)
                fitted += 1
                assert torch.equal(got, want), (type, shape)
    assert fitted >= 5


def test_a_small_workspace_and_the_built_in_scratch(lib):
    """A workspace of tab_conv2d_workspace_bytes takes the kernels that read the weights where they lie; the built-in scratch has room
    for them; a capture replays with both."""
    N, H, W, C, KN = 64, 14, 14, 256, 256
    g = torch.Generator(device="cuda").manual_seed(5)
    x, ths = torch.randn((N, H, W, C), device="cuda", generator=g), torch.full((N,), 0.5, device="cuda")
    QW, btn = weights(0, g, KN, 3, 3, C)
    lib.tab_internal_force_patch(14)
    lib.tab_conv2d_workspace_bytes.restype = ctypes.c_size_t
    size = lib.tab_conv2d_workspace_bytes(0, N, H, W, C)
    ws, y = torch.empty(size, dtype=torch.uint8, device="cuda"), torch.empty((N, KN, H, W), device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731

    def call():
        assert lib.tab_conv2d(p(x), p(QW), p(ths), p(btn), 0, 1, 1, 1, 1, N, H, W, C, KN, 3, 3, p(y), p(ws), ctypes.c_size_t(size),
                              ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0

    call()
    a = (x, QW, ths, btn, 0, 1, 1, 1, 1, N, H, W, C, KN, 3, 3)
    want = tab_amd.Conv2d(*a)
    assert torch.equal(y, want) and torch.equal(tab_amd.Conv2dStatic(*a), want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = tab_amd.Conv2d(*a)
        call()
    for seed in range(3):
        x.copy_(torch.randn((N, H, W, C), device="cuda", generator=torch.Generator(device="cuda").manual_seed(seed)))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, y)
        tab_amd.set_conv_kernel(tab_amd.CONV_MATRIX, 2)
        assert torch.equal(out, tab_amd.Conv2d(*a))
        lib.tab_internal_force_patch(14)


@pytest.mark.parametrize("case", CASES)
def test_the_weights_are_laid_out_behind_the_activation(case, lib):
    """What a call or a layer leaves behind its packed activation: the weights in the order of the shape in force, as a launch of their own
    lays them out, where the patch fits; nothing where it does not, or where the workspace has no room for them.  The output is right either
    way, and the kernels read the weights in two different orders: so it came from the kernel that the workspace shows."""
    N, H, W, C, KN, KH, KW, p1, p2, s1, s2 = case
    print(f"[case] patch, weights laid out {case}", flush=True)
    sizes = (p1, p2, s1, s2, N, H, W, C, KN, KH, KW)
    g = torch.Generator(device="cuda").manual_seed(KN + H)
    x = torch.randn((N, H, W, C), device="cuda", generator=g)
    x_nchw, ths = x.permute(0, 3, 1, 2).contiguous(), tab_amd.Threshold(x, N)
    stream, p = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    for f in (lib.tab_conv2d_workspace_bytes, lib.tab_conv2d_workspace_bytes_full, lib.tab_layer_workspace_bytes, lib.tab_layer_workspace_bytes_full):
        f.restype = ctypes.c_size_t
    for type in range(5):
        QW, btn = weights(type, g, KN, KH, KW, C)
        y = torch.empty_like(tab_amd.Conv2d(x, QW, ths, btn, type, *sizes))
        need, full = lib.tab_conv2d_workspace_bytes(type, N, H, W, C), lib.tab_conv2d_workspace_bytes_full(type, N, H, W, C, KN, KH, KW)
        calls = [(need, full, lambda ws, n: lib.tab_conv2d(p(x), p(QW), p(ths), p(btn), type, *sizes, p(y), p(ws), ctypes.c_size_t(n), stream))]
        if type < 4:
            need, full = lib.tab_layer_workspace_bytes(2 if type < 2 else 1, N, H, W, C), lib.tab_layer_workspace_bytes_full(type, N, H, W, C, KN, KH, KW)
            for nchw, a in ((0, x), (1, x_nchw)):
                calls.append((need, full, lambda ws, n, nchw=nchw, a=a: lib.tab_layer_conv2d(p(a), nchw, ctypes.c_float(0.7), p(QW), p(btn), type, *sizes,
                                                                                              p(y), p(ws), ctypes.c_size_t(n), stream)))
        want = []
        tab_amd.set_conv_kernel(tab_amd.CONV_MATRIX, 2)
        for need, _, call in calls:
            ws = torch.empty(need, dtype=torch.uint8, device="cuda")
            assert call(ws, need) == 0
            want.append(y.clone())
        for shape in SHAPES:
            lib.tab_internal_force_patch(shape)
            fits, room = fitting(lib, type, sizes)
            alone = torch.empty(max(room, 16), dtype=torch.uint8, device="cuda")
            if fits == shape:
                assert lib.tab_internal_conv_patch(p(x), p(QW), p(btn), type, *sizes, p(y), p(alone), ctypes.c_size_t(room), 1, stream) == 0
            for (need, full, call), right in zip(calls, want):
                assert (need + 15) // 16 * 16 + room <= full
                for size in (need, full):
                    ws = torch.full((full,), 0xA5, dtype=torch.uint8, device="cuda")
                    assert call(ws, size) == 0 and torch.equal(y, right), (type, shape)
                    at = (need + 15) // 16 * 16
                    if fits == shape and size == full:
                        assert torch.equal(ws[at:at + room], alone), (type, shape)
                        at += room
                    assert bool((ws[at:] == 0xA5).all()), (type, shape)


@pytest.mark.parametrize("full", [False, True])
def test_nothing_behind_the_workspace_is_written(full, lib):
    """The call writes inside the workspace_bytes it is given: of the packed activation alone, and with room for the weights."""
    N, H, C, KN = 64, 14, 192, 70
    g = torch.Generator(device="cuda").manual_seed(9)
    x, ths = torch.randn((N, H, H, C), device="cuda", generator=g), torch.full((N,), 0.5, device="cuda")
    y, p = torch.empty((N, H, H, KN), device="cuda"), lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for f in (lib.tab_conv2d_workspace_bytes, lib.tab_conv2d_workspace_bytes_full, lib.tab_layer_workspace_bytes, lib.tab_layer_workspace_bytes_full):
        f.restype = ctypes.c_size_t
    for type in range(5):
        QW, btn = weights(type, g, KN, 3, 3, C)
        a = (type, N, H, H, C)
        sizes = [lib.tab_conv2d_workspace_bytes_full(*a, KN, 3, 3) if full else lib.tab_conv2d_workspace_bytes(*a)]
        if type < 4:
            sizes.append(lib.tab_layer_workspace_bytes_full(*a, KN, 3, 3) if full else lib.tab_layer_workspace_bytes(2 if type < 2 else 1, N, H, H, C))
        for layer, size in enumerate(sizes):
            buffer = torch.full((size + 4096,), 0xA5, dtype=torch.uint8, device="cuda")
            room, sizes_of = ctypes.c_size_t(size), (type, 1, 1, 1, 1, N, H, H, C, KN, 3, 3)
            lib.tab_internal_force_patch(18)
            status = (lib.tab_layer_conv2d(p(x), 0, ctypes.c_float(0.7), p(QW), p(btn), *sizes_of, p(y), p(buffer), room, stream) if layer else
                      lib.tab_conv2d(p(x), p(QW), p(ths), p(btn), *sizes_of, p(y), p(buffer), room, stream))
            assert status == 0 and bool((buffer[size:] == 0xA5).all()), (type, layer)


@pytest.mark.parametrize("N", [16, 64])
def test_calls_allocate_the_room_they_use(N, lib):
    """Y, the packed activation and, where the rule takes the call to this kernel (N = 64), its weights: nothing else."""
    H, C, KN, type = 14, 256, 256, 4
    g = torch.Generator(device="cuda").manual_seed(6)
    x, ths = torch.randn((N, H, H, C), device="cuda", generator=g).abs(), torch.full((N,), 0.5, device="cuda")
    QW, btn = weights(type, g, KN, 3, 3, C)
    what, size = (ctypes.c_int * 3)(), ctypes.c_size_t(0)
    shape = lib.tab_internal_conv_patch_shape(type, 1, 1, 1, 1, N, H, H, C, KN, 3, 3, what, ctypes.byref(size))
    assert (shape >= 0) == (N == 64)
    room = lambda n: (n + 511) // 512 * 512  # noqa: E731
    want = room(N * H * H * KN * 4) + room(N * H * H * tab_amd.operand_words(type, 0, C) * 8 + (size.value + 16 if shape >= 0 else 0))
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    y = tab_amd.Conv2d(x, QW, ths, btn, type, 1, 1, 1, 1, N, H, H, C, KN, 3, 3)
    assert torch.cuda.max_memory_allocated() - before == want, y.shape
