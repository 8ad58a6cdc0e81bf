"""Workloads of the library as its users run them, one dict of plain values per case.

`listed()` holds the fixed cases, `draw(rng)` makes further ones of the same ranges, `prepare` builds what a program has
at hand before the call (inputs, packed weights, layers), `run` is one pass through the public entry points, `work` the
bytes and operations no implementation can do without and `tolerance` how far two correct implementations may differ.

The operations are the ones the library offers:
  conv      Quantize-on-the-fly convolution with packed weights, through the drop-in module or the package
  step      the ten ResNet-18 layer shapes one after the other through the drop-in module (a network's binary layers)
  quantize  packing a tensor, NHWC or NCHW, one or two bit planes, with the per-item counts
  layer     nn.TABConv2d.forward: activation thresholds, quantizer and convolution
  linear    nn.TABLinear.forward
  chain     nn.TABPackedChain.forward: packed activations between the layers
"""
import math

import torch

import TAB_CUDA
import tab_amd
from tab_amd import nn as tab_nn

APIS = {"TAB_CUDA": TAB_CUDA, "tab_amd": tab_amd}
TNN, TBN, BTN, BNN, DRF, RTN = range(6)

# (H, W, C, KN, kernel, pad, stride) of the ResNet-18 layers and their stride-2 variants
RESNET18 = (
    (56, 56, 64, 64, 3, 1, 1), (28, 28, 128, 128, 3, 1, 1), (14, 14, 256, 256, 3, 1, 1), (7, 7, 512, 512, 3, 1, 1),
    (56, 56, 64, 128, 3, 1, 2), (28, 28, 128, 256, 3, 1, 2), (14, 14, 256, 512, 3, 1, 2),
    (56, 56, 64, 128, 1, 0, 2), (28, 28, 128, 256, 1, 0, 2), (14, 14, 256, 512, 1, 0, 2),
)


def _conv(api, type, N, H, W, C, KN, KH, KW, p1, p2, s1, s2, relu=False):
    return {"op": "conv", "api": api, "type": type, "N": N, "H": H, "W": W, "C": C, "KN": KN, "KH": KH, "KW": KW,
            "p1": p1, "p2": p2, "s1": s1, "s2": s2, "relu": relu}


def _layer(type, layout, N, H, W, C, KN, K, pad, stride):
    return {"op": "layer", "type": type, "layout": layout, "N": N, "H": H, "W": W, "C": C, "KN": KN, "K": K, "pad": pad,
            "stride": stride}


def _chain(type, layout, N, H, W, C, depth, growth):
    return {"op": "chain", "type": type, "layout": layout, "N": N, "H": H, "W": W, "C": C, "depth": depth, "growth": growth}


def _quantize(api, layout, bits, N, H, W, C):
    return {"op": "quantize", "api": api, "layout": layout, "bits": bits, "N": N, "H": H, "W": W, "C": C}


def listed():
    return [
        # one image at a time: an interactive caller, where launches and the call itself are all there is
        dict(_conv("tab_amd", TNN, 1, 32, 32, 64, 64, 3, 3, 1, 1, 1, 1), name="conv_one_image_tnn"),
        # the binary layers of a residual network at a small batch, as a program written for the drop-in module calls them
        {"op": "step", "type": BNN, "N": 16, "relu": False, "name": "step_resnet18_bnn_n16"},
        # 2-bit levels at an ordinary batch, mid-size layer
        dict(_conv("tab_amd", DRF, 64, 14, 14, 256, 256, 3, 3, 1, 1, 1, 1, True), name="conv_levels_n64"),
        # a layer of a plain ternary stack, large image plane
        dict(_conv("TAB_CUDA", TNN, 32, 56, 56, 256, 256, 3, 3, 1, 1, 1, 1), name="conv_stack_tnn_n32"),
        # bulk processing, the largest convolution: large batch, many channels, asymmetric padding
        dict(_conv("tab_amd", BNN, 256, 28, 28, 512, 512, 3, 3, 1, 0, 1, 1), name="conv_bulk_bnn_n256"),
        # the shortcut of a residual block: 1x1, stride 2, binary activations and ternary weights
        dict(_conv("TAB_CUDA", BTN, 128, 28, 28, 256, 512, 1, 1, 0, 0, 2, 2, True), name="conv_shortcut_btn_n128"),
        # sizes that are no multiple of anything: channels pruned to 100 -> 75, 5x5, odd image
        dict(_conv("tab_amd", TBN, 5, 37, 53, 100, 75, 5, 5, 2, 1, 2, 2, True), name="conv_ragged_tbn"),
        # packing a whole activation set, the largest tensor: streams through memory once
        dict(_quantize("TAB_CUDA", "NHWC", 2, 256, 56, 56, 256), name="quantize_bulk_ternary"),
        # packing PyTorch's own layout at an odd plane size and a ragged channel count
        dict(_quantize("tab_amd", "NCHW", 1, 24, 61, 47, 75), name="quantize_ragged_nchw"),
        # a layer in a torch model: NCHW in and out, the activation threshold taken from the activation
        dict(_layer(TNN, "NCHW", 32, 56, 56, 64, 64, 3, 1, 1), name="layer_tnn_nchw_n32"),
        # the classifier behind the convolutions
        {"op": "linear", "type": BNN, "N": 64, "C": 512, "KN": 1000, "name": "linear_bnn_n64"},
        # a binary network's stages with packed activations in between
        dict(_chain(BNN, "NCHW", 64, 56, 56, 64, 4, 2), name="chain_bnn_n64"),
    ]


# ---- further cases of the same ranges ---------------------------------------------------------------------------------

def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _channels(rng, low=3, high=1024):
    """Two in three a multiple of 64, as networks have them, the rest anything."""
    c = _log(rng, low, high)
    return max(64, round(c / 64) * 64) if rng.random() < 2 / 3 else c


def _kernel(rng):
    k = rng.choice((1, 3, 3, 3, 5))
    return k, k // 2, rng.choice((1, 1, 2))


def _draw(rng):
    op = rng.choice(("conv", "conv", "conv", "conv", "step", "quantize", "quantize", "layer", "layer", "linear", "chain"))
    N, H = _log(rng, 1, 256), _log(rng, 7, 224)
    W = H if rng.random() < 0.5 else max(7, min(224, round(H * rng.uniform(0.6, 1.6))))
    layout = rng.choice(("NHWC", "NCHW"))
    if op == "conv":
        k, pad, stride = _kernel(rng)
        p2 = 0 if rng.random() < 0.2 else pad
        return _conv(rng.choice(("TAB_CUDA", "tab_amd")), rng.choice((TNN, TBN, BTN, BNN, TNN, TBN, BTN, BNN, DRF, RTN)), N, H, W,
                     _channels(rng), _channels(rng), k, k, pad, p2, stride, stride, rng.random() < 0.5)
    if op == "step":
        return {"op": "step", "type": rng.choice((TNN, TBN, BTN, BNN)), "N": _log(rng, 1, 64), "relu": rng.random() < 0.5}
    if op == "quantize":
        return _quantize(rng.choice(("TAB_CUDA", "tab_amd")), layout, rng.choice((1, 2)), N, H, W, _channels(rng))
    if op == "layer":
        k, pad, stride = _kernel(rng)
        return _layer(rng.choice((TNN, TBN, BTN, BNN)), layout, N, H, W, _channels(rng), _channels(rng), k, pad, stride)
    if op == "linear":
        return {"op": "linear", "type": rng.choice((TNN, TBN, BTN, BNN)), "N": _log(rng, 1, 1024), "C": _channels(rng, 64, 8192),
                "KN": _log(rng, 10, 4096)}
    return _chain(rng.choice((TBN, BTN, BNN)), layout, N, max(H, 14), max(W, 14), 64 * rng.choice((1, 1, 2, 3)), rng.randint(2, 4),
                  rng.choice((1, 2)))


def draw(rng):
    while True:
        case = _draw(rng)
        # no dearer than the largest listed cases: two thirds of the bulk convolution's bytes and of its operations, these
        # counted over whole 64-channel words and 64-filter tiles, which few channels leave mostly unused
        flops = 0
        for c in [] if case["op"] == "quantize" else _convs(case):
            _, N, _, _, C, KN, KH, KW = c[:8]
            flops += 2 * N * math.prod(_out(c)) * KH * KW * 64 * _words(C) * 64 * _words(KN)
        if work(case)["bytes"] <= 600e6 and flops <= 600e9:
            return case


# ---- geometry ---------------------------------------------------------------------------------------------------------

def _act_bits(type):
    return 2 if type in (TNN, TBN) else 1


def _weight_bits(type):
    return 2 if type in (TNN, BTN) else 1


def _convs(case):
    """The convolutions of a case: (type, N, H, W, C, KN, KH, KW, p1, p2, s1, s2) each."""
    t, N = case["type"], case["N"]
    if case["op"] == "conv":
        return [(t, N) + tuple(case[k] for k in ("H", "W", "C", "KN", "KH", "KW", "p1", "p2", "s1", "s2"))]
    if case["op"] == "step":
        return [(t, N, H, W, C, KN, k, k, p, p, s, s) for H, W, C, KN, k, p, s in RESNET18]
    if case["op"] == "layer":
        K, p, s = case["K"], case["pad"], case["stride"]
        return [(t, N, case["H"], case["W"], case["C"], case["KN"], K, K, p, p, s, s)]
    if case["op"] == "linear":
        return [(t, N, 1, 1, case["C"], case["KN"], 1, 1, 0, 0, 1, 1)]
    out, H, W, C = [], case["H"], case["W"], case["C"]
    for i in range(case["depth"]):
        KN = C if i == 0 else C * case["growth"]
        s = 1 if KN == C else 2
        out.append((t, N, H, W, C, KN, 3, 3, 1, 1, s, s))
        (H, W), C = _out(out[-1]), KN
    return out


def _out(conv):
    _, _, H, W, _, _, KH, KW, p1, p2, s1, s2 = conv
    return (H + 2 * p1 - KH + 1) // s1, (W + 2 * p2 - KW + 1) // s2


def _words(C):
    return (C + 63) // 64


def _weight_bytes(conv):
    t, _, _, _, C, KN, KH, KW = conv[:8]
    words = (C + 31) // 32 if t == RTN else _words(C) * (2 if t == DRF else _weight_bits(t))
    return 8 * KN * KH * KW * words


def work(case):
    N = case["N"]
    if case["op"] == "quantize":
        pixels = N * case["H"] * case["W"]
        return {"bytes": 4 * pixels * case["C"] + 4 * N + 8 * pixels * _words(case["C"]) * case["bits"] + 4 * N, "flops": 0}
    nbytes = flops = 0
    convs = _convs(case)
    for i, c in enumerate(convs):
        _, n, H, W, C, KN, KH, KW, p1, p2, s1, s2 = c
        OH, OW = _out(c)
        flops += 2 * n * OH * OW * KN * KH * KW * C
        nbytes += _weight_bytes(c)
        if case["op"] != "chain" or i == 0:
            # a 1x1 convolution without padding needs the pixels at its stride only; one that takes its threshold from the
            # activation needs them all
            some = KH == KW == 1 and not (case["op"] in ("layer", "linear") and _act_bits(c[0]) == 2)
            nbytes += 4 * n * C * (OH * OW if some else H * W)
        if case["op"] != "chain" or i == len(convs) - 1:
            nbytes += 4 * n * OH * OW * KN
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Packed words, counts and convolution sums are whole numbers, the same in every implementation.  Where the path takes
    the activation threshold from the activation itself (a mean of 32-bit floats), its last bits depend on the order of the
    sum, and now and then an element on the threshold falls to the other side."""
    if case["op"] in ("layer", "linear", "chain") and _act_bits(case["type"]) == 2:
        return {"rel": 1e-3, "max": 0.5}
    return "exact"


# ---- one pass ---------------------------------------------------------------------------------------------------------

def _randn(gen, shape):
    return torch.randn(shape, generator=gen, device="cuda")


def _mean_abs(x, scale=0.7):
    return (scale * x.abs().reshape(x.shape[0], -1).mean(dim=1)).float().contiguous()


def _conv_state(gen, conv, relu):
    """(arguments of Conv2d) for NHWC data, weights packed as the library packs them."""
    t, N, H, W, C, KN, KH, KW, p1, p2, s1, s2 = conv
    x, w = _randn(gen, (N, H, W, C)), _randn(gen, (KN, KH, KW, C))
    x = torch.relu(x) if relu else x
    if t in (DRF, RTN):
        if t == DRF:  # unsigned levels
            x, w = x.abs(), w.abs()
        qw = tab_amd.QuantizeFormat(w, _mean_abs(w), t, KN, KH, KW, C)
        ths, btn = _mean_abs(x), torch.zeros(KN, dtype=torch.int32, device="cuda")
    else:
        w_ths = _mean_abs(w) if _weight_bits(t) == 2 else torch.zeros(KN, device="cuda")
        qw, btn = tab_amd.Quantize(w, w_ths, _weight_bits(t), KN, KH, KW, C)
        ths = _mean_abs(x) if _act_bits(t) == 2 else torch.zeros(N, device="cuda")
    return (x, qw, ths, btn, t, p1, p2, s1, s2, N, H, W, C, KN, KH, KW)


def prepare(case, seed):
    gen = torch.Generator("cuda").manual_seed(int(seed))
    op, N = case["op"], case["N"]
    if op in ("conv", "step"):
        api = APIS[case.get("api", "TAB_CUDA")]
        calls = [_conv_state(gen, c, case["relu"]) for c in _convs(case)]
        return lambda: [api.Conv2d(*a) for a in calls]
    if op == "quantize":
        api, bits, H, W, C = APIS[case["api"]], case["bits"], case["H"], case["W"], case["C"]
        nchw = case["layout"] == "NCHW"
        x = _randn(gen, (N, C, H, W) if nchw else (N, H, W, C))
        ths = _mean_abs(x) if bits == 2 else torch.zeros(N, device="cuda")
        if nchw:
            return lambda: api.QuantizeNCHW(x, ths, bits, N, C, H, W)
        return lambda: api.Quantize(x, ths, bits, N, H, W, C)
    if op == "linear":
        layer = tab_nn.TABLinear.from_float(_randn(gen, (case["KN"], case["C"])), case["type"])
        x = _randn(gen, (N, case["C"]))
        return lambda: layer(x)
    layout, convs = case["layout"], _convs(case)
    layers = [tab_nn.TABConv2d.from_float(_randn(gen, (KN, C, KH, KW)), t, (s1, s2), (p1, p2), data_format=layout)
              for t, _, _, _, C, KN, KH, KW, p1, p2, s1, s2 in convs]
    model = layers[0]
    if op == "chain":
        # a ternary activation's threshold between layers is a constant found beforehand: half a standard deviation of a sum
        # over the layer's taps with half of the activations zero
        ths = {i: 0.5 * math.sqrt(0.5 * c[6] * c[7] * c[4]) for i, c in enumerate(convs[:-1], start=1)}
        model = tab_nn.TABPackedChain(layers, ths if _act_bits(case["type"]) == 2 else None, data_format=layout)
    shape = (N, case["C"], case["H"], case["W"])
    x = _randn(gen, shape if layout == "NCHW" else (N, case["H"], case["W"], case["C"]))
    return lambda: model(x)


def run(state):
    return state()
