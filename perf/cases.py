"""The work that training code has the "vk" device do, as cases to measure: what goes in, one pass through the
public entry points (ordinary PyTorch calls on vk tensors, autograd, torch_vulkan.dequant_int8_linear), what
the pass cannot do without, and what a float64 evaluation of the same inputs gives.

The kinds of case are the layers of a diffusion transformer or UNet trained with low-rank adapters: linear
layers (trained, frozen under a LoRA, int8), the conditioning projection, fused attention over tokens and
over a text context, layer_norm, a convolution block, and one whole DiT block.  Token counts are those of
image aspect buckets (an H / 16 x W / 16 grid is rarely a multiple of 64), dimensions those of this
repository's tests and benchmark (512 and 2048 wide blocks, heads of 40 to 128, 77-token contexts, 320 to
512 channels) and generic ones around them."""

import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "torch-vulkan_amd"))
import torch_vulkan  # noqa: E402

VK = torch.device("vk")
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
SIZE = {"bf16": 2, "f16": 2, "f32": 4}


def listed():
    return [
        # AdaLN conditioning: SiLU and a projection of one vector per image; launches and latency
        {"name": "modulation", "kind": "modulation", "dtype": "bf16", "batch": 2, "dim": 512},
        # a trained linear layer over the tokens of an odd aspect bucket (60 x 67), both directions
        {"name": "linear_bf16", "kind": "linear", "dtype": "bf16", "tokens": 4020, "fin": 2048, "fout": 2048},
        # the same in full precision (a small model or a stage kept in fp32)
        {"name": "linear_f32", "kind": "linear", "dtype": "f32", "tokens": 1024, "fin": 1024, "fout": 2048},
        # a frozen linear under a rank-16 adapter: the MLP's first layer of a 2048-wide block
        {"name": "lora_f16", "kind": "lora", "dtype": "f16", "tokens": 1024, "fin": 2048, "fout": 8192, "rank": 16},
        # int8 weights, the tokens of two images at once
        {"name": "int8_bf16", "kind": "int8", "dtype": "bf16", "tokens": 2 * 1560, "fin": 2048, "fout": 8192},
        # self-attention of a 512 px image, the repository's benchmark shape
        {"name": "attn_bf16", "kind": "attention", "dtype": "bf16", "batch": 1, "heads": 16, "q": 1024, "k": 1024, "dim": 128},
        # self-attention of a UNet's first level over a 63 x 64 latent, two images
        {"name": "attn_long_f16", "kind": "attention", "dtype": "f16", "batch": 2, "heads": 8, "q": 4032, "k": 4032, "dim": 64},
        # cross-attention to a 77-token text context, a UNet level with heads of 80
        {"name": "attn_cross_f16", "kind": "attention", "dtype": "f16", "batch": 2, "heads": 8, "q": 1024, "k": 77, "dim": 80},
        # self-attention in full precision, large enough for the default policy to take the fused kernels
        {"name": "attn_f32", "kind": "attention", "dtype": "f32", "batch": 1, "heads": 16, "q": 2080, "k": 2080, "dim": 64},
        # layer_norm with affine parameters, both directions
        {"name": "norm_bf16", "kind": "norm", "dtype": "bf16", "rows": 4020, "dim": 2048},
        # group_norm, SiLU and a 3 x 3 convolution on the latent of a 768 px image, both directions
        {"name": "resnet_bf16", "kind": "resnet", "dtype": "bf16", "batch": 1, "cin": 320, "cout": 512, "h": 96, "w": 96},
        # one whole DiT block with rank-16 adapters on its four linears: output and every gradient
        {"name": "block_bf16", "kind": "block", "dtype": "bf16", "tokens": 1024, "heads": 16},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A feature dimension: mostly multiples of 64, some of 8, now and then any (patch embeddings)."""
    step = rng.choice((64, 64, 64, 64, 64, 64, 8, 8, 8, 1))
    return max(lo, _log(rng, lo, hi) // step * step)


# Work of a drawn case in bf16 flops: full-precision flops count sixteenfold (the cards' matrix rates).
def _cost(case):
    return work(case)["flops"] * (16 if case["dtype"] == "f32" else 1)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(("modulation", "linear", "linear", "lora", "int8", "attention", "attention", "attention", "norm",
                           "resnet", "block"))
        half = rng.choice(("bf16", "f16"))
        any3 = rng.choice(("bf16", "f16", "f32"))
        if kind == "modulation":
            c = {"dtype": half, "batch": rng.randint(1, 16), "dim": _width(rng, 256, 3072)}
        elif kind == "linear":
            c = {"dtype": any3, "tokens": _log(rng, 64, 8192), "fin": _width(rng, 64, 8192), "fout": _width(rng, 64, 8192)}
        elif kind == "lora":
            c = {"dtype": half, "tokens": _log(rng, 64, 4096), "fin": 64 * _log(rng, 5, 128), "fout": 64 * _log(rng, 5, 128),
                 "rank": rng.choice((4, 8, 16, 32, 64, 128))}
        elif kind == "int8":
            c = {"dtype": half, "tokens": _log(rng, 1, 8192), "fin": 64 * _log(rng, 5, 128), "fout": 64 * _log(rng, 5, 128)}
        elif kind == "attention":
            q = _log(rng, 64, 4096)
            c = {"dtype": any3, "batch": rng.randint(1, 4), "heads": rng.randint(1, 24), "q": q,
                 "k": rng.choice((q, q, rng.randint(8, 512))), "dim": rng.choice((40, 64, 64, 80, 96, 128, 128))}
        elif kind == "norm":
            c = {"dtype": any3, "rows": _log(rng, 16, 16384), "dim": _width(rng, 64, 4096)}
        elif kind == "resnet":
            c = {"dtype": half, "batch": rng.randint(1, 2), "cin": 64 * rng.randint(2, 10), "cout": 64 * rng.randint(2, 10),
                 "h": 4 * rng.randint(4, 32), "w": 4 * rng.randint(4, 32)}
        else:
            c = {"dtype": "bf16", "tokens": _log(rng, 64, 1100), "heads": rng.randint(2, 16)}
        c = {"kind": kind, **c}
        if _cost(c) <= most:
            return c


# ---- inputs ---------------------------------------------------------------------------------------------------
def _inputs(case, seed):
    """Everything a pass reads, on the CPU in the case's dtype, from the seed alone: activations and output
    gradients ~ N(0, 1), weights ~ N(0, 0.02), norm weights around 1."""
    g = torch.Generator().manual_seed(seed)
    dt = DTYPES[case["dtype"]]

    def r(*shape, scale=1.0, mean=0.0):
        return torch.randn(shape, generator=g).mul_(scale).add_(mean).to(dt)

    kind = case["kind"]
    if kind == "modulation":
        n, d = case["batch"], case["dim"]
        return {"c": r(n, d), "w": r(6 * d, d, scale=0.02), "b": r(6 * d, scale=0.02), "g": r(n, 6 * d)}
    if kind in ("linear", "lora", "int8"):
        m, i, o = case["tokens"], case["fin"], case["fout"]
        t = {"x": r(m, i), "b": r(o, scale=0.02)}
        if kind == "int8":
            t["q"] = torch.randint(-127, 128, (o, i), generator=g, dtype=torch.int8)
            t["scale"] = (torch.rand((o, (i + 63) // 64), generator=g) * 2e-4 + 1e-4).to(torch.bfloat16)
            return t
        t.update(w=r(o, i, scale=0.02), g=r(m, o))
        if kind == "lora":
            t.update(A=r(case["rank"], i, scale=0.02), B=r(o, case["rank"], scale=0.01))
        return t
    if kind == "attention":  # token-major, as a model's projections leave them
        n, h, d = case["batch"], case["heads"], case["dim"]
        return {"q": r(n, case["q"], h, d), "k": r(n, case["k"], h, d), "v": r(n, case["k"], h, d), "g": r(n, case["q"], h, d)}
    if kind == "norm":
        m, d = case["rows"], case["dim"]
        return {"x": r(m, d, mean=0.5), "w": r(d, scale=0.1, mean=1.0), "b": r(d, scale=0.1), "g": r(m, d)}
    if kind == "resnet":
        n, i, o, h, w = case["batch"], case["cin"], case["cout"], case["h"], case["w"]
        return {"x": r(n, i, h, w, mean=0.2), "nw": r(i, scale=0.1, mean=1.0), "nb": r(i, scale=0.1),
                "w": r(o, i, 3, 3, scale=0.02), "b": r(o, scale=0.02), "g": r(n, o, h, w)}
    d, m = 128 * case["heads"], case["tokens"]  # a DiT block, AdaLN-conditioned, MLP ratio 4, rank-16 adapters
    t = {"x": r(1, m, d), "c": r(1, d), "g": r(1, m, d), "ada_w": r(6 * d, d, scale=0.02), "ada_b": r(6 * d, scale=0.02)}
    for name, i, o in (("qkv", d, 3 * d), ("proj", d, d), ("fc1", d, 4 * d), ("fc2", 4 * d, d)):
        t.update({name + "_w": r(o, i, scale=0.02), name + "_b": r(o, scale=0.02), name + "_A": r(16, i, scale=0.02),
                  name + "_B": r(o, 16, scale=0.01)})
    return t


# What is trained: the inputs whose gradients a pass returns.
def _wrt(case, names):
    return {"modulation": ("c", "w", "b"), "linear": ("x", "w", "b"), "lora": ("x", "A", "B"), "int8": (), "attention": ("q", "k", "v"),
            "norm": ("x", "w", "b"), "resnet": ("x", "nw", "nb", "w", "b"),
            "block": ("x",) + tuple(sorted(n for n in names if n.endswith(("_A", "_B"))))}[case["kind"]]


# ---- the layers -------------------------------------------------------------------------------------------------
def _block(t, heads):
    def lora(x, n):
        return F.linear(x, t[n + "_w"], t[n + "_b"]) + F.linear(F.linear(x, t[n + "_A"]), t[n + "_B"])

    x, (n, m, d) = t["x"], t["x"].shape
    sh1, sc1, g1, sh2, sc2, g2 = F.linear(F.silu(t["c"]), t["ada_w"], t["ada_b"]).unsqueeze(1).chunk(6, dim=-1)
    h = F.layer_norm(x, (d,), eps=1e-6) * (1 + sc1) + sh1
    q, k, v = lora(h, "qkv").view(n, m, 3, heads, d // heads).unbind(2)
    a = F.scaled_dot_product_attention(q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2))
    x = x + g1 * lora(a.transpose(1, 2).reshape(n, m, d), "proj")
    h = F.layer_norm(x, (d,), eps=1e-6) * (1 + sc2) + sh2
    return x + g2 * lora(F.gelu(lora(h, "fc1"), approximate="tanh"), "fc2")


def _forward(case, t):
    kind = case["kind"]
    if kind == "modulation":
        return F.linear(F.silu(t["c"]), t["w"], t["b"])
    if kind == "linear":
        return F.linear(t["x"], t["w"], t["b"])
    if kind == "lora":
        return F.linear(t["x"], t["w"], t["b"]) + F.linear(F.linear(t["x"], t["A"]), t["B"])
    if kind == "attention":
        q, k, v = (t[n].transpose(1, 2) for n in "qkv")
        return F.scaled_dot_product_attention(q, k, v).transpose(1, 2)
    if kind == "norm":
        return F.layer_norm(t["x"], (case["dim"],), t["w"], t["b"], 1e-5)
    if kind == "resnet":
        return F.conv2d(F.silu(F.group_norm(t["x"], 32, t["nw"], t["nb"], 1e-5)), t["w"], t["b"], padding=1)
    return _block(t, case["heads"])


def prepare(case, seed):
    torch_vulkan.set_inline_backward()  # as a training loop on this device does once, on its own thread
    t = {k: v.to(VK) for k, v in _inputs(case, seed).items()}
    wrt = _wrt(case, t)
    for n in wrt:
        t[n].requires_grad_(True)
    return {"case": case, "t": t, "wrt": wrt}


def run(state):
    case, t, wrt = state["case"], state["t"], state["wrt"]
    if case["kind"] == "int8":
        return {"y": torch_vulkan.dequant_int8_linear(t["x"], t["q"], t["scale"], t["b"])}
    y = _forward(case, t)
    grads = torch.autograd.grad(y, [t[n] for n in wrt], t["g"])
    return {"y": y.detach(), **{"d" + n: d for n, d in zip(wrt, grads)}}


def exact(case, seed):
    t = {k: v.double() for k, v in _inputs(case, seed).items()}
    if case["kind"] == "int8":
        # the weight that the layer defines is the product rounded once to the activations' dtype
        s = t["scale"].repeat_interleave(64, dim=1)[:, : case["fin"]]
        return {"y": F.linear(t["x"], (t["q"] * s).to(DTYPES[case["dtype"]]).double(), t["b"])}
    wrt = _wrt(case, t)
    if case["kind"] == "attention":  # head by head: the score matrices of all heads at once are gigabytes
        out = {"y": torch.empty_like(t["q"]), **{"d" + n: torch.empty_like(t[n]) for n in wrt}}
        for n in range(case["batch"]):
            for h in range(case["heads"]):
                q, k, v = (t[m][n, :, h].clone().requires_grad_(True) for m in "qkv")
                y = torch.softmax(q @ k.t() / math.sqrt(case["dim"]), dim=-1) @ v
                grads = torch.autograd.grad(y, (q, k, v), t["g"][n, :, h])
                for m, d in zip(("y", "dq", "dk", "dv"), (y.detach(), *grads)):
                    out[m][n, :, h] = d
        return out
    for n in wrt:
        t[n].requires_grad_(True)
    y = _forward(case, t)
    grads = torch.autograd.grad(y, [t[n] for n in wrt], t["g"])
    return {"y": y.detach(), **{"d" + n: d for n, d in zip(wrt, grads)}}


# ---- what a pass cannot do without --------------------------------------------------------------------------------
def work(case):
    kind, e = case["kind"], SIZE[case["dtype"]]
    if kind == "modulation":
        n, d = case["batch"], case["dim"]
        return {"bytes": e * 2 * (6 * d * d + 6 * d + n * d + n * 6 * d), "flops": 3 * 2 * n * 6 * d * d}
    if kind in ("linear", "lora", "int8"):
        m, i, o = case["tokens"], case["fin"], case["fout"]
        if kind == "int8":
            return {"bytes": e * (m * i + m * o + o) + i * o + 2 * o * ((i + 63) // 64), "flops": 2 * m * i * o}
        if kind == "linear":
            return {"bytes": e * (2 * m * i + 2 * i * o + 2 * m * o + 2 * o), "flops": 3 * 2 * m * i * o}
        k = case["rank"]
        return {"bytes": e * (2 * m * i + i * o + 2 * m * o + o + 2 * k * (i + o)),
                "flops": 2 * 2 * m * i * o + 3 * 2 * m * k * (i + o)}
    if kind == "attention":
        n, h, q, k, d = (case[x] for x in ("batch", "heads", "q", "k", "dim"))
        # forward two products; backward four and the scores again
        return {"bytes": e * n * h * d * (4 * q + 4 * k), "flops": 7 * 2 * n * h * q * k * d}
    if kind == "norm":
        m, d = case["rows"], case["dim"]
        return {"bytes": e * (4 * m * d + 4 * d), "flops": 20 * m * d}
    if kind == "resnet":
        n, i, o, hw = case["batch"], case["cin"], case["cout"], case["h"] * case["w"]
        return {"bytes": e * (2 * n * hw * (i + o) + 2 * 9 * i * o + 4 * i + 2 * o), "flops": 3 * 2 * 9 * n * hw * i * o}
    m, d, k = case["tokens"], 128 * case["heads"], 16
    io = ((d, 3 * d), (d, d), (d, 4 * d), (4 * d, d))
    flops = 2 * 6 * d * d + sum(2 * 2 * m * i * o + 3 * 2 * m * k * (i + o) for i, o in io) + 7 * 2 * m * m * d
    weights = 6 * d * d + sum(i * o + o + 2 * k * (i + o) for i, o in io)
    return {"bytes": e * (4 * m * d + weights), "flops": flops}


# What another correct implementation at the same precision may differ by: about four times the distance from
# the float64 values measured per kind (one rounding per stored value in the case's dtype; softmax weights and
# score gradients rounded once more in 16-bit attention; every intermediate of a block).
_REL = {"bf16": 1e-2, "f16": 2e-3, "f32": 1e-5}


def tolerance(case):
    if case["kind"] == "block":
        return {"rel": 3e-2}
    return {"rel": _REL[case["dtype"]]}
