"""What the package is timed on: calls that its users make, over the range of sizes they make them at.

A case is one pass through the public operators and layers on tensors that are already on the GPU:

  infer       conv2d_gw8 without gradients (serving, evaluation)
  train       conv2d_gw8 and its gradients on float16 tensors
  amp         a Conv2dGw8 layer with float32 parameters under torch.autocast, forward and backward, as a
              training loop runs it; the activations are float16, or float32 where the layer sits on a
              residual stream that autocast has promoted
  block       Conv2dGw8 followed by LayerNorm2d under torch.autocast, forward and backward: the two layers
              of this package at the head of a ConvNeXt block
  norm_infer  layernorm_2d without gradients
  norm_train  layernorm_2d and its gradients

Sizes are those of the package's benchmark and tests (C=64 56x56 batches, the stages of the ConvNeXt-T-shaped
network, the EfficientNet-like shapes of the kernel tests) and odd ones between them.
"""

import math

import torch

from spio_amd.functional import conv2d_gw8, layernorm_2d
from spio_amd.layers import Conv2dGw8, LayerNorm2d

CL = torch.channels_last
OPS = ("infer", "train", "amp", "block", "norm_infer", "norm_train")


def _case(op, n, c, h, w, k=3, pad=None, bias=False, x="float16", input_grad=True, name=None):
    """A case; `pad` None keeps the image size (odd k)."""
    case = {
        "op": op, "n": n, "c": c, "h": h, "w": w, "k": k, "pad": k // 2 if pad is None else pad,
        "bias": bias, "x": x, "input_grad": input_grad,
    }  # fmt: skip
    return case if name is None else dict(case, name=name)


def listed():
    return [
        # one image: what a request costs when nothing is batched
        _case("infer", 1, 64, 56, 56, name="infer 1n 64c 56x56"),
        # a small ragged batch, image and channel count: no dimension is a multiple of a tile
        _case("infer", 3, 72, 49, 33, 5, bias=True, name="infer 3n 72c 49x33 5x5"),
        # early layer of an EfficientNet-like network: three groups only, large images
        _case("infer", 128, 24, 144, 144, name="infer 128n 24c 144x144"),
        # training at a per-GPU batch of 32, at the benchmark's batch of 128 and at a large batch
        _case("train", 32, 64, 56, 56, name="train 32n 64c 56x56"),
        _case("train", 128, 64, 56, 56, name="train 128n 64c 56x56"),
        _case("train", 512, 64, 56, 56, name="train 512n 64c 56x56"),
        # the large filter of ConvNeXt-like blocks
        _case("train", 256, 256, 14, 14, 7, name="train 256n 256c 14x14 7x7"),
        # late layer of an EfficientNet-like network: many channels, odd small images, 5x5
        _case("train", 128, 1392, 9, 9, 5, name="train 128n 1392c 9x9 5x5"),
        # first layer of a network: the images need no gradient
        _case("train", 32, 48, 224, 224, bias=True, input_grad=False, name="train first 32n 48c 224x224"),
        # mixed precision: third stage of the ConvNeXt-T-shaped network on its float32 residual
        # stream, and the first stage's convolution and norm on float16 activations
        _case("amp", 128, 384, 14, 14, bias=True, x="float32", name="amp 128n 384c 14x14 float32"),
        _case("block", 128, 96, 56, 56, bias=True, name="block 128n 96c 56x56"),
        # the norm alone, last stage: few pixels, many channels
        _case("norm_train", 128, 768, 7, 7, bias=True, name="norm 128n 768c 7x7"),
    ]


def _log_uniform(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def draw(rng):
    sizes = [work(c) for c in listed()]
    least = min(w["bytes"] for w in sizes)
    most = max(w["bytes"] for w in sizes)
    wide = next(w for c, w in zip(listed(), sizes) if c["k"] == 7)  # the most arithmetic of a listed case
    while True:
        op = rng.choices(OPS, weights=(5, 7, 4, 3, 1, 2))[0]
        norm = op.startswith("norm")
        k = 3 if norm else rng.choices((3, 5, 7, 1), weights=(12, 5, 3, 1))[0]
        n = round(_log_uniform(rng, 1, 512))
        c = 8 * round(_log_uniform(rng, 2, 128 if norm or op == "block" else 192))
        h = round(_log_uniform(rng, 7, 224))
        w = h if rng.random() < 0.6 else round(min(256, max(7, h * _log_uniform(rng, 0.5, 2))))
        pad = 0 if not norm and rng.random() < 0.1 else None
        amp = op in ("amp", "block")
        case = _case(
            op, n, c, h, w, k, pad, bias=op == "block" or norm or rng.random() < 0.4,
            x="float32" if op == "amp" and rng.random() < 0.5 else "float16",
            input_grad=amp or rng.random() < 0.85,
        )  # fmt: skip
        cost = work(case)
        # float32 activations under autocast cost about twice their own bytes
        if (least <= cost["bytes"] <= most / (2 if amp else 1)) and cost["flops"] <= wide["flops"]:
            return case


def _shapes(case):
    n, c, h, w, k, pad = (case[f] for f in ("n", "c", "h", "w", "k", "pad"))
    out = (n, c, h, w) if case["op"].startswith("norm") else (n, c, h + 2 * pad - k + 1, w + 2 * pad - k + 1)
    return (n, c, h, w), out


def prepare(case, seed):
    op, c, k = case["op"], case["c"], case["k"]
    in_shape, out_shape = _shapes(case)
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(shape, dtype):
        t = torch.empty(shape, device="cuda", dtype=dtype, memory_format=CL)
        return t.normal_(generator=gen)

    def uniform(shape, low, high):
        return torch.empty(shape, device="cuda", dtype=torch.float32).uniform_(low, high, generator=gen)

    bound = 1 / math.sqrt(8 * k * k)  # nn.Conv2d's initial range
    weight = uniform((c, 8, k, k), -bound, bound).contiguous(memory_format=CL)
    bias = uniform((c,), -bound, bound) if case["bias"] else None
    scale, shift = uniform((c,), 0.5, 1.5), uniform((c,), -0.5, 0.5)
    state = {"case": case, "x": normal(in_shape, getattr(torch, case["x"]))}
    if not op.endswith("infer"):
        state["x"].requires_grad_(case["input_grad"])
        state["dy"] = normal(out_shape, getattr(torch, case["x"]))
    if op in ("infer", "train"):
        state["weight"], state["bias"] = weight.half(), bias
    elif op in ("norm_infer", "norm_train"):
        state["weight"], state["bias"] = scale, shift
    if op in ("train", "norm_train"):
        state["weight"].requires_grad_()
        if state["bias"] is not None:
            state["bias"].requires_grad_()
    if op in ("amp", "block"):
        conv = Conv2dGw8(c, c, k, padding=case["pad"], groups=c // 8, bias=case["bias"], device="cuda")
        conv = conv.to(memory_format=CL)
        with torch.no_grad():
            conv.weight.copy_(weight)
            if bias is not None:
                conv.bias.copy_(bias)
        layers = [conv]
        if op == "block":
            norm = LayerNorm2d(c, eps=1e-6, device="cuda")
            with torch.no_grad():
                norm.weight.copy_(scale)
                norm.bias.copy_(shift)
            layers.append(norm)
        state["model"] = torch.nn.Sequential(*layers)
    return state


def run(state):
    case, x = state["case"], state["x"]
    op, pad = case["op"], case["pad"]
    if op in ("infer", "train"):
        y = conv2d_gw8(x, state["weight"], state["bias"], padding_y=pad, padding_x=pad, groups=case["c"] // 8)
    elif op in ("norm_infer", "norm_train"):
        y = layernorm_2d(x, state["weight"], state["bias"], 1e-6)
    if op in ("infer", "norm_infer"):
        return y
    if op in ("train", "norm_train"):
        wanted = [t for t in (x, state["weight"], state["bias"]) if t is not None and t.requires_grad]
        return [y, *torch.autograd.grad(y, wanted, state["dy"])]
    model = state["model"]
    model.zero_grad(set_to_none=True)
    x.grad = None
    with torch.autocast("cuda", dtype=torch.float16):
        y = model(x)
    y.backward(state["dy"])
    return [y.detach(), x.grad, *(p.grad for p in model.parameters())]


def work(case):
    op, c, k = case["op"], case["c"], case["k"]
    in_shape, out_shape = _shapes(case)
    size = 4 if case["x"] == "float32" else 2
    x, y = size * math.prod(in_shape), size * math.prod(out_shape)
    macs = 0 if op.startswith("norm") else math.prod(out_shape) * 8 * k * k
    weights = 0 if op.startswith("norm") else c * 8 * k * k * (4 if op in ("amp", "block") else 2)
    vectors = 4 * c * ((2 if op == "block" or op.startswith("norm") else 0) + (1 if case["bias"] and macs else 0))
    moved, flops = x + y + weights + vectors, 2 * macs
    if op.endswith("infer"):
        return {"bytes": moved, "flops": flops if macs else 10 * math.prod(in_shape)}
    # backward: the input and the output's gradient in, the gradients of the input and the parameters out
    moved += x + y + (x if case["input_grad"] else 0) + 2 * weights + vectors
    flops += 2 * macs * (2 if case["input_grad"] else 1)
    if not macs:
        flops = 30 * math.prod(in_shape)
    elif op == "block":
        flops += 30 * math.prod(out_shape)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    # Four times what the path differs from itself in float64: its results are rounded to float16 once
    # (2.1e-4 of the norm, 4.9e-4 of a value); behind a convolution whose output was rounded the norm's
    # results are off by 3.0e-4 and 1.5e-3, the latter more where a pixel's variance is small.
    return {"rel": 1.2e-3, "max": 1e-2} if case["op"] == "block" else {"rel": 8e-4, "max": 2e-3}
