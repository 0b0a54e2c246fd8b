"""What the framework's speed is judged by: passes of ``KSLinear(algo='kernel')`` layers, forward
and training, over the sizes, types and layouts a program uses them in.

A case is a dict of plain values:

``layers``   the layers of the pass, separated by ``|``; a layer is its factors ``axbxcxd``
             separated by ``+``, the one applied first on the left
``dtype``    ``fp32``, ``fp16`` or ``e4m3`` (the layer's type: e4m3 layers return fp16)
``input``    type of the pass's input: the layer's own, or ``fp16`` for an e4m3 layer that
             quantises its input itself
``bs_last``  feature-major (features, batch) tensors instead of (batch, features)
``batch``    rows: tokens x images
``bias``     the layers have a bias
``act``      ``gelu`` after every layer but the last one (after the only one), or empty
``train``    forward and backward; the pass returns every gradient
"""
import math

import torch

from ksmm_amd import KSLinear, quantize_fp8

FP8 = torch.float8_e4m3fn
DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "e4m3": FP8}
SIZES = {"fp32": 4, "fp16": 2, "e4m3": 1}

# 128 images of 196 tokens: the batch of the published tables, and of the benchmark here
FULL = 25088

# the feed-forward blocks of a ViT-S (384 -> 1536 -> 384) and a ViT-B (768 -> 3072 -> 768)
VIT_S_UP, VIT_S_DOWN = "6x64x64x1+1x768x192x2", "6x64x256x1+1x128x128x3"
VIT_B_UP, VIT_B_DOWN = "12x64x64x1+1x1536x384x2", "12x64x256x1+1x256x256x3"


def _case(name, layers, dtype, batch, bs_last=False, bias=True, act="", train=False, input=None):
    case = {"layers": layers, "dtype": dtype, "input": input or dtype, "bs_last": bs_last, "batch": batch,
            "bias": bias, "act": act, "train": train}
    return dict(case, name=name) if name else case


def listed():
    ffn_s, ffn_b = VIT_S_UP + "|" + VIT_S_DOWN, VIT_B_UP + "|" + VIT_B_DOWN
    return [
        # a single request: the feed-forward block on the tokens of one image
        _case("ffn_s fp16 1 image", ffn_s, "fp16", 196, act="gelu"),
        # the layer of the README on a handful of columns, as a small test or a probe calls it
        _case("readme fp32 last 32", VIT_S_UP, "fp32", 32, bs_last=True),
        # the headline: one bandwidth-bound fp32 factor
        _case("48x48 d16 fp32 last", "1x48x48x16", "fp32", FULL, bs_last=True, bias=False),
        # the same in the default layout on 33 images of 197 tokens (a class token makes them odd)
        _case("48x48 d16 fp32 odd", "1x48x48x16", "fp32", 33 * 197),
        # the layer of the README at the batch it is quoted at
        _case("readme fp32 last", VIT_S_UP, "fp32", FULL, bs_last=True),
        # dense 192 x 192 blocks, feature-major rows that no vector divides
        _case("192x192 fp16 last odd", "4x192x192x1", "fp16", 33 * 197, bs_last=True),
        # serving a ViT-B feed-forward block on full batches
        _case("up_b fp16 gelu", VIT_B_UP, "fp16", FULL, act="gelu"),
        # one training step of the ViT-S feed-forward block
        _case("ffn_s fp16 train", ffn_s, "fp16", FULL, act="gelu", train=True),
        # training in fp32 on a smaller, feature-major batch (32 images)
        _case("readme fp32 last train", VIT_S_UP, "fp32", 32 * 196, bs_last=True, train=True),
        # butterfly of radix 16 on e4m3 activations that come with their scale
        _case("butterfly e4m3 last", "1x16x16x64+16x16x16x4+64x16x16x1", "e4m3", FULL, bs_last=True, bias=False),
        # 8-bit weights in a network of fp16 activations: every layer quantises what it is given
        _case("ffn_b e4m3 from fp16", ffn_b, "e4m3", 32 * 197, act="gelu", input="fp16"),
        # the largest: a wide factor of the pattern list, 73728 features
        _case("192x192 d64 fp16 wide", "6x192x192x64", "fp16", FULL, bias=False),
    ]


def _layers(case):
    return [[tuple(int(v) for v in f.split("x")) for f in layer.split("+")] for layer in case["layers"].split("|")]


def _ffn_layers(width):
    """Up- and down-projection of a feed-forward block the way those of ViT-S and ViT-B are cut."""
    n = width // 64
    k = 3 if width % 3 == 0 else 4
    return ("%dx64x64x1+1x%dx%dx2" % (n, 2 * width, width // 2),
            "%dx64x256x1+1x%dx%dx%d" % (n, width // k, width // k, k))


def _single_factor(rng):
    """One factor with the block sizes, aspect ratios and strides of the pattern list."""
    while True:
        side = rng.choice((16, 32, 48, 64, 96, 128, 192, 256, 384))
        b, c = {0: (side, side), 1: (4 * side, side), 2: (side, 4 * side)}[rng.choice((0, 0, 1, 2))]
        if rng.random() < 0.1:
            b += rng.randint(1, 15)  # the list has blocks of 449 .. 468 rows
        a, d = rng.choice((1, 1, 2, 3, 4, 6, 12, 16)), rng.choice((1, 1, 2, 3, 4, 6, 8, 16, 32, 64))
        if max(b, c) <= 1536 and 256 <= a * d * max(b, c) <= 24576:
            return "%dx%dx%dx%d" % (a, b, c, d)


def draw(rng):
    kind = rng.choice(("ffn", "layer", "factor", "factor", "factor", "butterfly"))
    dtype = rng.choice(("fp32", "fp16", "fp16", "e4m3"))
    act, bias = "", rng.random() < 0.7
    if kind == "factor":
        layers = _single_factor(rng)
    elif kind == "butterfly":
        n = rng.choice((256, 512, 1024))
        layers = {256: "1x16x16x16+16x16x16x1", 512: "1x16x16x32+16x16x16x2+32x16x16x1",
                  1024: "1x16x16x64+16x16x16x4+64x16x16x1"}[n]
    else:
        up, down = _ffn_layers(rng.choice((192, 384, 576, 768, 1024)))
        layers = up + "|" + down if kind == "ffn" else rng.choice((up, down))
        act = "gelu" if kind == "ffn" or rng.random() < 0.5 else ""
    train = dtype != "e4m3" and rng.random() < 0.35
    given = rng.choice(("fp16", "e4m3")) if dtype == "e4m3" else dtype
    batch = int(round(math.exp(rng.uniform(0.0, math.log(FULL)))))
    if rng.random() < 0.5:  # whole images, with or without a class token
        batch = max(1, batch // 196) * rng.choice((196, 197))
    case = _case(None, layers, dtype, min(batch, FULL), bool(rng.random() < 0.5), bias, act, train, given)
    most = _cost(listed()[-1])
    while _cost(case) > most / 2:
        case["batch"] = (case["batch"] + 1) // 2
    return case


def _cost(case):
    """Seconds a pass would take at ordinary rates: what keeps drawn cases below the largest."""
    w = work(case)
    return w["bytes"] / 4e12 + w["flops"] / (6e13 if case["dtype"] == "fp32" else 3e14)


def prepare(case, seed):
    gen = torch.Generator().manual_seed(seed)
    dev = torch.Generator(device="cuda").manual_seed(seed)
    torch.manual_seed(seed)  # the layers' own biases
    layers, modules = _layers(case), []
    for i, patterns in enumerate(layers):
        weights = [(torch.rand(p, generator=gen) * 2 - 1) / math.sqrt(p[2]) for p in patterns]
        act = case["act"] if len(layers) == 1 or i + 1 < len(layers) else ""
        modules.append(KSLinear(patterns, weights=weights, bias=case["bias"], algo="kernel", dtype=DTYPES[case["dtype"]],
                                bs_last=case["bs_last"], device="cuda", act=act or None))

    def normal(features):
        shape = (features, case["batch"]) if case["bs_last"] else (case["batch"], features)
        dtype = torch.float32 if case["dtype"] == "fp32" else torch.float16
        return torch.randn(shape, generator=dev, device="cuda", dtype=dtype)

    x, scale, grad = normal(modules[0].in_size), None, None
    if case["input"] == "e4m3":
        x, scale = quantize_fp8(x)
        scale = float(scale)
    if case["train"]:
        x.requires_grad_(True)
        grad = normal(modules[-1].out_size)
    return {"layers": modules, "x": x, "x_scale": scale, "grad": grad}


def run(state):
    layers, x = state["layers"], state["x"]
    if state["grad"] is None:
        with torch.no_grad():
            y = layers[0](x, x_scale=state["x_scale"])
            for layer in layers[1:]:
                y = layer(y)
        return y
    y = x
    for layer in layers:
        y = layer(y)
    wanted = [x] + [p for layer in layers for p in layer.parameters()]
    return [y.detach()] + list(torch.autograd.grad(y, wanted, state["grad"]))


def work(case):
    """Input, weights and biases read, result written; a training pass also reads the gradient of
    the result and writes those of the input and of the parameters, for three times the products."""
    layers = _layers(case)
    wide = SIZES["fp32" if case["dtype"] == "fp32" else "fp16"]
    a, _, c, d = layers[0][0]
    in_size = a * c * d
    outs = [p[-1][0] * p[-1][1] * p[-1][3] for p in layers]
    weights = sum(math.prod(p) for patterns in layers for p in patterns)
    x = in_size * case["batch"] * SIZES[case["input"]]
    y = outs[-1] * case["batch"] * wide
    params = weights * SIZES[case["dtype"]] + (sum(outs) * wide if case["bias"] else 0)
    times = 2 if case["train"] else 1
    return {"bytes": times * (x + y + params), "flops": (3 if case["train"] else 1) * 2 * case["batch"] * weights}


def tolerance(case):
    """About four times the difference to the same pass on float64 tensors, measured over these ranges:
    up to 6e-7 in fp32 (a sum over the full batch makes it 1e-6) and 5.6e-4 in fp16, where chains and
    gradients round several times.  An e4m3 layer that quantises the result of another layer
    turns a last-bit difference of that result into a step of e4m3 now and then: 3.5e-3."""
    if case["dtype"] == "fp32":
        return {"rel": 4e-6}
    return {"rel": 1.4e-2 if case["dtype"] == "e4m3" and "|" in case["layers"] else 2.2e-3}
