"""The work a user of this package has it do, as cases that can be timed: block dropout fused into a linear layer, into a
whole MLP stack and into a convolution, through the functions that the layers call, forward and backward.

A pass is one training step of the layer or stack (forward, then every gradient the optimiser would ask for), or the
forward alone where nothing needs a gradient.  Masks are drawn on the device by the call itself, pinned by a seed, or
given.  Data has the distributions that the path meets: standard normal activations, weights of variance 1/K, images
in [0, 1), gradients of the size that a mean over the batch leaves.
"""
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "sparse-dropout_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import flash_dropout.functional as F  # noqa: E402

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _linear(m, k, n, dtype="fp16", bs=64, p=0.5, mask="drawn", grad=True):
    return dict(kind="linear", m=m, k=k, n=n, dtype=dtype, bs=bs, p=p, mask=mask, grad=grad)


def _mlp(m, dims, act, dtype="fp16", bs=64, p=0.5, first_p=None, grad_in=False):
    """dims: feature counts from the input to the output, "784-1024-10"; first_p: drop rate of the first layer's input."""
    return dict(kind="mlp", m=m, dims=dims, act=act, dtype=dtype, bs=bs, p=p, first_p=p if first_p is None else first_p,
                grad_in=grad_in)


def _conv(b, c, h, w, k, r=3, stride=1, pad=1, dtype="fp16", bs=64, p=0.5, channels_last=False):
    return dict(kind="conv", b=b, c=c, h=h, w=w, k=k, r=r, stride=stride, pad=pad, dtype=dtype, bs=bs, p=p,
                channels_last=channels_last)


def listed():
    return [
        # a small layer on a small batch: what a step costs before any arithmetic does
        dict(_linear(128, 256, 256, p=0.1), name="linear small"),
        # sampling predictions with dropout left on (no gradients): a few hundred tokens through one layer
        dict(_linear(512, 1024, 1024, "bf16", p=0.1, grad=False), name="linear forward only"),
        # classifier on flattened 32 x 32 images: three narrow layers, ReLU between, the first without dropout
        dict(_mlp(1024, "1024-1024-1024-128", "relu", first_p=0.0), name="mlp 1024 wide"),
        # classifier on 28 x 28 images: a reduction that ends inside a block, ten outputs
        dict(_mlp(4096, "784-1024-1024-10", "relu", first_p=0.0), name="mlp 784 ten classes"),
        # transformer feed-forward blocks inside a model (the input needs its gradient): 64 images of 256 patches, and
        # 32 sequences of 128 tokens; drop rates as trained with
        dict(_mlp(16384, "384-1536-384", "gelu", "bf16", p=0.1, grad_in=True), name="ffn 384-1536"),
        dict(_mlp(4096, "1024-4096-1024", "gelu", "fp16", bs=128, p=0.3, grad_in=True), name="ffn 1024-4096"),
        # one linear layer at the sizes of a square sweep; the mask given by the caller at the middle size
        dict(_linear(2048, 2048, 2048, p=0.25, mask="given"), name="linear 2048"),
        dict(_linear(4096, 4096, 4096, "bf16", bs=32, p=0.5), name="linear 4096 blocks of 32"),
        dict(_linear(8192, 8192, 8192, p=0.5), name="linear 8192"),
        # sizes nobody rounded: a batch as long as its data, features with one more appended, an odd number of outputs
        dict(_linear(3001, 1025, 777, "bf16", p=0.3), name="linear odd"),
        # a 3 x 3 convolution on 32 x 32 images, and one on 28 x 28 images, whose rows do not divide a block
        dict(_conv(128, 64, 32, 32, 128), name="conv 32x32"),
        dict(_conv(256, 32, 28, 28, 64, dtype="bf16", p=0.25), name="conv 28x28"),
    ]


# What the listed cases stand for.  No drawn case does more arithmetic than the largest listed one.
_MOST_FLOPS = 6.0 * 8192 ** 3 * 0.5
_DROP = (0.05, 0.1, 0.2, 0.25, 0.3, 0.4, 0.5, 0.6, 0.75)


def _size(rng, lo, hi, grain):
    """Spread over the logarithm of [lo, hi], a multiple of grain."""
    v = lo * (hi / lo) ** rng.random()
    return max(grain, int(v / grain + 0.5) * grain)


def draw(rng):
    kind = rng.choices(("linear", "forward", "mlp", "conv"), (9, 2, 5, 4))[0]
    dtype, p = rng.choice(("fp16", "bf16")), rng.choice(_DROP)
    while True:
        if kind in ("linear", "forward"):
            # layers are mostly multiples of 64 wide; the rest are multiples of 8 or any number at all
            grain = rng.choice((64, 64, 64, 8, 1))
            c = _linear(_size(rng, 64, 16384, rng.choice((64, 1))), _size(rng, 64, 8192, grain), _size(rng, 64, 8192, grain),
                        dtype, rng.choice((32, 64, 64, 64, 96, 128, 256)), p, rng.choice(("drawn", "drawn", "given")),
                        kind == "linear")
            most = _MOST_FLOPS if grain >= 8 else _MOST_FLOPS / 16
        elif kind == "mlp":
            m, act = _size(rng, 256, 16384, rng.choice((64, 1))), rng.choice(("relu", "gelu"))
            if rng.random() < 0.5:  # feed-forward block: out to four times the width and back
                d = _size(rng, 128, 2048, 64)
                c = _mlp(m, f"{d}-{4 * d}-{d}", act, dtype, rng.choice((32, 64, 64, 128)), p, grad_in=True)
            else:  # classifier: hidden layers of one width, any number of classes
                d = _size(rng, 128, 2048, 64)
                dims = [_size(rng, 128, 3072, rng.choice((64, 8)))] + [d] * rng.choice((1, 2, 3)) + [_size(rng, 10, 1000, 1)]
                c = _mlp(m, "-".join(map(str, dims)), act, dtype, rng.choice((64, 64, 128)), p, first_p=0.0)
            most = _MOST_FLOPS
        else:
            hw, r = rng.choice((7, 8, 14, 16, 28, 30, 32, 48, 56, 64)), rng.choice((1, 3, 3, 3, 5))
            c = _conv(_size(rng, 8, 256, 1), _size(rng, 16, 256, 8), hw, hw, _size(rng, 32, 256, 8), r,
                      rng.choice((1, 1, 1, 2)), r // 2, dtype, rng.choice((64, 64, 128)), p, rng.random() < 0.25)
            most = _MOST_FLOPS / 16
        if work(c)["flops"] <= most:
            return c


# ------------------------------------------------------------------------------------------------ inputs
def _blocks(n, bs):
    return -(-n // bs)


def _dims(case):
    return [int(v) for v in case["dims"].split("-")]


def prepare(case, seed):
    dev, dt = torch.device("cuda"), _DTYPES[case["dtype"]]
    gen = torch.Generator(dev).manual_seed(seed)

    def normal(*shape, std=1.0):
        return torch.randn(*shape, generator=gen, device=dev).mul_(std).to(dt)

    if case["kind"] == "linear":
        m, k, n, bs, p = case["m"], case["k"], case["n"], case["bs"], case["p"]
        s = dict(case=case, seed=seed, x=normal(m, k), w=normal(n, k, std=k ** -0.5), mask=None)
        if case["grad"]:
            s["dy"] = normal(m, n)
            s["x"].requires_grad_()
            s["w"].requires_grad_()
        if case["mask"] == "given":
            s["mask"] = torch.rand(_blocks(m, bs), _blocks(k, bs), generator=gen, device=dev) < p
        return s
    if case["kind"] == "mlp":
        m, dims = case["m"], _dims(case)
        x = normal(m, dims[0]) if case["grad_in"] else torch.rand(m, dims[0], generator=gen, device=dev).to(dt)
        ws = [normal(o, i, std=(1.0 if j else 2.0) * i ** -0.5).requires_grad_() for j, (i, o) in enumerate(zip(dims, dims[1:]))]
        s = dict(case=case, seed=seed, x=x.requires_grad_(case["grad_in"]), ws=ws, dy=normal(m, dims[-1]))
        s["ps"] = (case["first_p"],) + (case["p"],) * (len(ws) - 1)
        return s
    b, c, h, w, k, r = (case[v] for v in ("b", "c", "h", "w", "k", "r"))
    x = normal(b, c, h, w)
    if case["channels_last"]:
        x = x.to(memory_format=torch.channels_last)
    po, qo = _conv_out(case)
    return dict(case=case, seed=seed, x=x.requires_grad_(), w=normal(k, c, r, r, std=(c * r * r) ** -0.5).requires_grad_(),
                dy=normal(b, k, po, qo))


def _conv_out(case):
    return tuple((v + 2 * case["pad"] - case["r"]) // case["stride"] + 1 for v in (case["h"], case["w"]))


# ------------------------------------------------------------------------------------------------ one pass
def run(state):
    case = state["case"]
    if case["kind"] == "linear":
        if not case["grad"]:
            with torch.no_grad():
                return _linear_forward(state, case)
        y = _linear_forward(state, case)
        return (y, *torch.autograd.grad(y, (state["x"], state["w"]), state["dy"]))
    if case["kind"] == "mlp":
        y = F.hip_blockwise_dropout_mlp(state["x"], state["ws"], case["bs"], state["ps"], case["act"], seed=state["seed"])
        wrt = ([state["x"]] if case["grad_in"] else []) + state["ws"]
        return (y, *torch.autograd.grad(y, wrt, state["dy"]))
    y = F.blockwise_dropout_conv2d(state["x"], state["w"], case["bs"], case["p"], case["pad"], case["stride"],
                                   seed=state["seed"])
    return (y, *torch.autograd.grad(y, (state["x"], state["w"]), state["dy"]))


def _linear_forward(state, case):
    if state["mask"] is not None:
        return F.hip_blockwise_dropout_matmul_mask(state["x"], state["mask"], case["bs"], case["p"], state["w"])
    return F.hip_blockwise_dropout_matmul(state["x"], state["w"], case["bs"], case["p"], seed=state["seed"])


# ------------------------------------------------------------------------------------------------ bounds
def work(case):
    """Two bytes per element.  Dropped blocks of an input are not read; dropped blocks of its gradient are written (zeros).
    Each of the three products costs 2 flops per kept element of the masked matrix and column."""
    if case["kind"] == "linear":
        m, k, n, keep = case["m"], case["k"], case["n"], 1.0 - case["p"]
        if not case["grad"]:
            return {"bytes": 2.0 * (m * k * keep + n * k + m * n), "flops": 2.0 * m * k * n * keep}
        return {"bytes": 2.0 * (m * k * keep + n * k + 2 * m * n + m * k + n * k), "flops": 6.0 * m * k * n * keep}
    if case["kind"] == "mlp":
        m, dims = case["m"], _dims(case)
        size = m * dims[0] * (1.0 - case["first_p"]) + 2 * m * dims[-1] + (m * dims[0] if case["grad_in"] else 0)
        flops = 0.0
        for j, (i, o) in enumerate(zip(dims, dims[1:])):
            size += 2 * i * o
            products = 3 if (j or case["grad_in"]) else 2
            flops += 2.0 * products * m * i * o * (1.0 - (case["p"] if j else case["first_p"]))
        return {"bytes": 2.0 * size, "flops": flops}
    b, c, h, w, k, r, keep = (*(case[v] for v in ("b", "c", "h", "w", "k", "r")), 1.0 - case["p"])
    po, qo = _conv_out(case)
    return {"bytes": 2.0 * (2 * b * c * h * w + 2 * k * c * r * r + 2 * b * k * po * qo),
            "flops": 6.0 * b * po * qo * c * r * r * k * keep}


def tolerance(case):
    """Sums are in fp32 and rounded once per product, so two correct results differ by the last bit of the element type
    here and there: 2^-11 (fp16) or 2^-8 (bf16) of a value at most per rounding.  A stack rounds at every hidden layer and
    a convolution's input gradient may round the terms of its sum, so a few such roundings add up."""
    return {"rel": 1e-2, "max": 0.1} if case["dtype"] == "bf16" else {"rel": 2e-3, "max": 0.02}
