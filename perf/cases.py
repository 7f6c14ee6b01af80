"""The layers this framework is measured on: 3x3, pad 1, stride 1 forward convolutions through its
public entry points, over the sizes, operand types and calling conventions that its users meet.

Sizes are the reference's own sweep (C = K, H = W of (64, 56), (128, 28), (256, 14), (512, 7) at
N = 32 ... 128), layers of ResNet-34 and VGG-16 at serving and training batch sizes, and shapes that
fit no tile.  Three ways to call:

  dropin    convolutionForward / its descriptor form: raw filters with every call, tensors in the
            library's layouts (CHWN in, CRSK filters, KHWN out)
  prepared  filters transformed once, as a server does at start-up, then one call per batch
  nchw      prepared filters, and activations that arrive and leave as NCHW
"""
import math

import torch

import opencnn_amd as ocn

PRECISION = {"f32": ocn.F32, "f16": ocn.F16, "bf16": ocn.BF16}


def _case(name, n, c, h, w, k, operands="f32", api="dropin"):
    return {"name": name, "n": n, "c": c, "h": h, "w": w, "k": k, "operands": operands, "api": api}


def listed():
    return [
        # one image on a small layer: launches and latency, next to no arithmetic
        _case("one_image", 1, 64, 14, 14, 64),
        # small batch on the deepest layer of the sweep: few tiles, long channel sums
        _case("deep_small_batch", 32, 512, 7, 7, 512),
        # the four layers of the sweep at training batch sizes
        _case("resnet_56", 64, 64, 56, 56, 64),
        _case("resnet_28", 128, 128, 28, 28, 128),
        _case("deep_14", 128, 256, 14, 14, 256),
        _case("deep_7", 128, 512, 7, 7, 512),
        # the first layer of a network: three channels, a large image
        _case("rgb_224", 64, 3, 224, 224, 64),
        # nothing is a multiple of a tile; weights laid out once
        _case("ragged", 100, 120, 27, 29, 250, api="prepared"),
        # a server's batch on a large image: half of a 32-wide batch group
        _case("half_group", 16, 64, 56, 56, 64, api="prepared"),
        # a layer inside a network that keeps its activations in NCHW
        _case("nchw_28", 64, 128, 28, 28, 128, api="nchw"),
        # reduced-precision GEMM operands: the benchmark layer, and the heaviest layer of VGG-16
        _case("f16_deep_14", 128, 256, 14, 14, 256, operands="f16"),
        _case("bf16_vgg_28", 64, 512, 28, 28, 512, operands="bf16", api="prepared"),
    ]


def draw(rng):
    """One more layer of the same ranges; no more arithmetic and no larger tensors than the listed ones."""
    most_flops = max(work(c)["flops"] for c in listed())
    most_bytes = max(work(c)["bytes"] for c in listed())

    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    while True:
        api = rng.choice(["dropin", "dropin", "prepared", "nchw"])
        operands = rng.choice(["f32", "f32", "f32", "f16", "bf16"])
        n, c, h, k = spread(1, 128), spread(3, 512), spread(7, 224), spread(32, 512)
        if rng.random() < 0.5:  # the round numbers that networks use
            n, c, k = (1 << round(math.log2(v)) for v in (n, max(c, 8), k))
        # the drop-in call takes square images only
        w = h if api == "dropin" or rng.random() < 0.5 else max(7, min(224, spread(h / 2, h * 2)))
        case = {"n": n, "c": c, "h": h, "w": w, "k": k, "operands": operands, "api": api}
        cost = work(case)
        if cost["flops"] <= most_flops and cost["bytes"] <= most_bytes:
            return case


def prepare(case, seed):
    n, c, h, w, k = (case[key] for key in ("n", "c", "h", "w", "k"))
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    ocn.init()
    shape = (n, c, h, w) if case["api"] == "nchw" else (c, h, w, n)
    x = torch.randn(shape, device=dev, generator=gen)  # a normalised image
    if c > 3:
        x.relu_()  # what the layer before leaves
    filters = torch.randn((c, 3, 3, k), device=dev, generator=gen) * math.sqrt(2.0 / (9.0 * c))
    state = {
        "case": case,
        "x": x,
        "y": torch.empty((k, h, w, n), device=dev),
        "ws": torch.empty(ocn.workspace_bytes(c, k) // 4, device=dev),
        "filters": filters,
    }
    if case["api"] != "dropin":
        ocn.set_operand_precision(PRECISION[case["operands"]])
        ocn.filter_transform(filters, state["ws"], k, c, ocn.FILTER_CRSK, ocn.WW_MFMA)
        ocn.set_operand_precision(ocn.F32)
    if case["api"] == "nchw":
        state["x_chwn"] = torch.empty((c, h, w, n), device=dev)
        state["y_nchw"] = torch.empty((n, k, h, w), device=dev)
    return state


def run(state):
    case = state["case"]
    n, c, h, w, k = (case[key] for key in ("n", "c", "h", "w", "k"))
    precision = PRECISION[case["operands"]]
    if case["api"] == "dropin":
        if precision == ocn.F32:
            tiles = ocn.tiles_dim(w)
            ocn.convolutionForward(state["x"], h, w, state["filters"], h, w, n, k, state["y"], state["ws"],
                                   k * n * h * w, tiles, n, 4, tiles * 4, c, k, c, 3, 3, 4, 2)
        else:
            ocn.conv_forward_desc(state["x"], state["filters"], state["y"], state["ws"], n, c, h, w, k,
                                  precision=precision)
        return state["y"]
    if case["api"] == "prepared":
        ocn.conv_forward_desc(state["x"], None, state["y"], state["ws"], n, c, h, w, k, precision=precision)
        return state["y"]
    ocn.nchw_to_chwn(state["x"], state["x_chwn"], n, c, h, w)
    ocn.conv_forward_desc(state["x_chwn"], None, state["y"], state["ws"], n, c, h, w, k, precision=precision)
    ocn.khwn_to_nkhw(state["y"], state["y_nchw"], n, k, h, w)
    return state["y_nchw"]


def work(case):
    """Every input read once, the output written once; the multiplications of the sixteen products of
    Winograd's F(2x2, 3x3), which the layer's arithmetic is defined as."""
    n, c, h, w, k = (case[key] for key in ("n", "c", "h", "w", "k"))
    element = 4 if case["operands"] == "f32" else 2
    filters = 9 * c * k * 4 if case["api"] == "dropin" else 16 * c * k * element
    tiles = ((h + 1) // 2) * ((w + 1) // 2)
    return {"bytes": 4 * n * h * w * (c + k) + filters, "flops": 32 * n * tiles * c * k}


def tolerance(case):
    """Four times what the layer differs by from the direct convolution in 64 bits: 1.2e-7 (3 channels) ...
    5.8e-7 (512) with fp32 operands, 4.3e-4 ... 4.4e-4 with fp16 and 3.4e-3 ... 3.5e-3 with bf16; the largest
    difference of an element 0.9e-6 ... 4.1e-6, 1.9e-3 ... 2.5e-3 and 1.7e-2 ... 2.0e-2."""
    return {"f32": {"rel": 2.4e-6, "max": 1.6e-5},
            "f16": {"rel": 1.8e-3, "max": 1e-2},
            "bf16": {"rel": 1.4e-2, "max": 8e-2}}[case["operands"]]
