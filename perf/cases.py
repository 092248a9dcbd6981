"""What the low-precision path is measured on: calls of the public operators as a training or a
serving program makes them, with the sizes, types and options that such programs use.

Five kinds of case:

  linear    one ``gemm_fp8`` / ``gemm_fp4`` layer. Serving: the weight is quantized once and kept, the
            activation is quantized on each call. Training: the weight is a 16-bit parameter, forward and
            backward run, both gradients come back.
  experts   one ``grouped_gemm_fp8`` / ``grouped_gemm_fp4`` bank of MoE experts, serving or training alike;
            the experts' token counts are uneven ("zipf", two of them empty) or even.
  moe       a whole expert layer: permute by router choice, first grouped product, gated activation fused
            into the second, unpermute; forward and backward.
  quantize  the stand-alone quantizers with the matching de-quantizer.
"""

import math
import os
import random  # noqa: F401  (draw() takes a random.Random)
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("primus-turbo_amd"))  # the package of the tree that is the working folder

import primus_turbo.pytorch as turbo  # noqa: E402
from primus_turbo.pytorch.core.low_precision import (  # noqa: E402
    Float4QuantConfig,
    Float8QuantConfig,
    Format,
    ScaleDtype,
    ScalingGranularity,
)
from primus_turbo.pytorch.core.quantized_tensor import create_quantized_weight  # noqa: E402

_G = ScalingGranularity
_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_SIZE = {"bf16": 2, "f16": 2, "f32": 4}
#: bytes of one quantized element with its share of the scales
_CODE = {"tensorwise": 1.0, "rowwise": 1.0, "blockwise": 1.0, "mxfp8": 1 + 1 / 32, "mxfp4": 0.5 + 1 / 32}


def _linear(name, recipe, tokens, n, k, train, **more):
    return dict(dict(name=name, kind="linear", recipe=recipe, tokens=tokens, n=n, k=k, train=train, dtype="bf16",
                     hybrid=False, main_grad=False), **more)


def _experts(name, recipe, groups, tokens, n, k, train, spread, **more):
    return dict(dict(name=name, kind="experts", recipe=recipe, groups=groups, tokens=tokens, n=n, k=k, train=train,
                     spread=spread, dtype="bf16", hybrid=False), **more)


def listed():
    return [
        # a decoding step of a serving program: sixteen sequences, one token each, weight kept in FP8
        _linear("serve_linear_tensorwise_decode", "tensorwise", 16, 4096, 4096, False),
        # a short prompt of odd length through the widest projection, block scales
        _linear("serve_linear_blockwise_prompt", "blockwise", 777, 4096, 7168, False),
        # prefill of a long batch through an FP4 up-projection
        _linear("serve_linear_mxfp4_prefill", "mxfp4", 4096, 28672, 8192, False),
        # decoding with experts: thirty-two sequences of eight choices each, spread over thirty-two experts
        _experts("serve_experts_blockwise_decode", "blockwise", 32, 256, 4096, 7168, False, "zipf"),
        # the default recipe in training, weight gradients added into the optimizer's fp32 buffer
        _linear("train_linear_tensorwise", "tensorwise", 4096, 4096, 4096, True, main_grad=True),
        # a ragged micro-batch, output width no multiple of a tile, gradients in E5M2
        _linear("train_linear_rowwise_ragged", "rowwise", 3001, 2880, 4096, True, hybrid=True),
        # the headline product in training
        _linear("train_linear_blockwise_8192", "blockwise", 8192, 8192, 8192, True),
        # a down-projection in MXFP8
        _linear("train_linear_mxfp8", "mxfp8", 8192, 7168, 2048, True),
        # the headline expert bank: gate and up projections of thirty-two experts
        _experts("train_experts_blockwise", "blockwise", 32, 32768, 4096, 7168, True, "zipf"),
        # the matching down-projection in FP4 on a quarter of the tokens, evenly routed
        _experts("train_experts_mxfp4_down", "mxfp4", 32, 8192, 7168, 2048, True, "even"),
        # a whole expert layer on a small micro-batch
        dict(name="train_moe_layer_mxfp8", kind="moe", recipe="mxfp8", tokens=1024, topk=8, experts=32, hidden=4096,
             inter=2048, dtype="bf16"),
        # the stand-alone tensorwise cast and its inverse
        dict(name="quantize_tensorwise_4096", kind="quantize", recipe="tensorwise", rows=4096, cols=4096, direction="row",
             dtype="bf16"),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of ``step`` between ``lo`` and ``hi``, spread evenly over its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi // step * step, max(-(-lo // step) * step, round(v / step) * step)))


def draw(rng):
    kind = rng.choice(["serve_linear", "serve_linear", "serve_experts", "train_linear", "train_linear", "train_experts", "moe",
                       "quantize"])
    while True:
        if kind in ("serve_linear", "train_linear"):
            recipe = rng.choice(["tensorwise", "rowwise", "blockwise", "mxfp8", "mxfp4"])
            train = kind == "train_linear"
            n, k = _log(rng, 512, 16384, 32), _log(rng, 512, 16384, 32)
            tokens = _log(rng, 128, 16384) if train else _log(rng, 1, 8192)
            if recipe == "mxfp4":  # this recipe takes token counts in steps of its block
                tokens = -(-tokens // 32) * 32
            flops = 2 * tokens * n * k * (3 if train else 1)
            if n * k > 1 << 27 or flops > 3e12:
                continue
            c = _linear(None, recipe, tokens, n, k, train, dtype=rng.choice(["bf16", "bf16", "f16"]),
                        hybrid=train and recipe != "mxfp4" and rng.random() < 0.5,
                        main_grad=train and recipe in ("tensorwise", "mxfp8", "mxfp4") and rng.random() < 0.5)
        elif kind in ("serve_experts", "train_experts"):
            recipe = rng.choice(["rowwise", "blockwise", "mxfp8", "mxfp4"])
            train = kind == "train_experts"
            groups = rng.choice([4, 8, 16, 32, 64])
            n, k = _log(rng, 512, 7168, 128), _log(rng, 512, 7168, 128)
            tokens = _log(rng, 512, 32768) if train else _log(rng, 8, 8192)
            if groups * n * k > 1 << 30 or 2 * tokens * n * k * (3 if train else 1) > 3e12:
                continue
            c = _experts(None, recipe, groups, tokens, n, k, train, rng.choice(["zipf", "even"]),
                         hybrid=train and recipe != "mxfp4" and rng.random() < 0.5)
        elif kind == "moe":
            experts = rng.choice([8, 16, 32, 64])
            hidden, inter = _log(rng, 1024, 7168, 128), _log(rng, 512, 2048, 128)
            tokens, topk = _log(rng, 64, 4096), rng.choice([2, 4, 6, 8])
            if experts * hidden * inter > 1 << 28 or 18 * tokens * topk * hidden * inter > 3e12:
                continue
            c = dict(name=None, kind="moe", recipe=rng.choice(["blockwise", "mxfp8", "mxfp4"]), tokens=tokens, topk=topk,
                     experts=experts, hidden=hidden, inter=inter, dtype="bf16")
        else:
            recipe = rng.choice(["tensorwise", "rowwise", "blockwise", "mxfp8", "mxfp4"])
            rows, cols = _log(rng, 16, 32768), _log(rng, 256, 16384, 32)
            if recipe == "mxfp4":
                rows = -(-rows // 32) * 32
            ways = {"tensorwise": ["row"], "rowwise": ["row", "column"]}.get(recipe, ["row", "both"])
            if rows * cols > 1 << 28:
                continue
            c = dict(name=None, kind="quantize", recipe=recipe, rows=rows, cols=cols, direction=rng.choice(ways),
                     dtype=rng.choice(["bf16", "bf16", "f16", "f32"]))
        del c["name"]
        return c


def _config(recipe, hybrid=False):
    if recipe == "mxfp4":
        return Float4QuantConfig()
    more = {"blockwise": dict(block_size=128), "mxfp8": dict(block_size=32, scale_dtype=ScaleDtype.E8M0)}.get(recipe, {})
    gran = {"tensorwise": _G.TENSORWISE, "rowwise": _G.ROWWISE, "blockwise": _G.BLOCKWISE, "mxfp8": _G.MX_BLOCKWISE}[recipe]
    return Float8QuantConfig(format=Format.HYBRID if hybrid else Format.E4M3, granularity=gran, **more)


def _code_dtype(recipe):
    return turbo.float4_e2m1fn_x2 if recipe == "mxfp4" else turbo.float8_e4m3


def group_lens(groups, total, spread, seed):
    """Tokens of each expert: "even", or about 1 / rank^1.2 in a random order with two experts idle."""
    rng = np.random.default_rng(seed)
    w = np.ones(groups)
    if spread == "zipf":
        w = rng.permutation((1.0 + np.arange(groups)) ** -1.2)
        w[rng.choice(groups, 2, replace=False)] = 0
    lens = np.floor(w / w.sum() * total).astype(np.int64)
    rest = int(total - lens.sum())
    lens[np.argsort(-w, kind="stable")[:rest]] += 1
    lens[int(np.argmax(w))] += total - int(lens.sum())
    return lens


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = _DTYPES[case["dtype"]]

    def randn(*shape, std=1.0, dtype=dt):
        return torch.randn(shape, generator=gen, device="cuda", dtype=dtype).mul_(std)

    s = {"case": case}
    if case["kind"] == "quantize":
        s["x"] = randn(case["rows"], case["cols"])
        return s
    s["config"] = _config(case["recipe"], case.get("hybrid", False))
    if case["kind"] == "moe":
        t, e, h, f = case["tokens"], case["experts"], case["hidden"], case["inter"]
        s["x"] = randn(t, h).requires_grad_(True)
        s["w1"] = randn(e, 2 * f, h, std=h ** -0.5).requires_grad_(True)
        s["w2"] = randn(e, h, f, std=f ** -0.5).requires_grad_(True)
        # a router: scores with a bias for each expert, the best of them chosen, their weights normalised
        scores = torch.randn(t, e, generator=gen, device="cuda") + 0.5 * torch.randn(e, generator=gen, device="cuda")
        best, s["topk_idx"] = scores.topk(case["topk"], dim=1)
        s["probs"] = best.softmax(1).requires_grad_(True)
        s["grad"] = randn(t, h, std=1e-2)
        return s
    n, k = case["n"], case["k"]
    lead = ()
    if case["kind"] == "experts":
        lead = (case["groups"],)
        s["lens"] = torch.from_numpy(group_lens(case["groups"], case["tokens"], case["spread"], seed)).cuda()
    s["x"] = randn(case["tokens"], k).requires_grad_(case["train"])
    w = randn(*lead, n, k, std=k ** -0.5)
    if case["train"]:
        s["w"] = torch.nn.Parameter(w)
        if case.get("main_grad"):
            s["w"].main_grad = torch.zeros(w.shape, dtype=torch.float32, device="cuda")
            s["w"].grad_added_to_main_grad = False
        s["grad"] = randn(case["tokens"], n, std=1e-2)
    else:
        s["w"] = create_quantized_weight(w, _code_dtype(case["recipe"]), s["config"])[0]
    return s


def _run_linear(s, case):
    op = turbo.ops.gemm_fp4 if case["recipe"] == "mxfp4" else turbo.ops.gemm_fp8
    if not case["train"]:
        with torch.no_grad():
            return op(s["x"], s["w"], trans_b=True, config=s["config"])
    out = op(s["x"], s["w"], trans_b=True, config=s["config"],
             fuse_bgrad_accum_pattern="megatron" if case["main_grad"] else None)
    gx, gw = torch.autograd.grad(out, (s["x"], s["w"]), s["grad"])
    return out.detach(), gx, s["w"].main_grad if case["main_grad"] else gw


def _run_experts(s, case):
    op = turbo.ops.grouped_gemm_fp4 if case["recipe"] == "mxfp4" else turbo.ops.grouped_gemm_fp8
    if not case["train"]:
        with torch.no_grad():
            return op(s["x"], s["w"], s["lens"], trans_b=True, config=s["config"])
    out = op(s["x"], s["w"], s["lens"], trans_b=True, config=s["config"])
    return (out.detach(), *torch.autograd.grad(out, (s["x"], s["w"]), s["grad"]))


def _run_moe(s, case):
    first, second = ((turbo.ops.grouped_gemm_fp4, turbo.ops.glu_grouped_gemm_fp4) if case["recipe"] == "mxfp4"
                     else (turbo.ops.grouped_gemm_fp8, turbo.ops.glu_grouped_gemm_fp8))
    pad = 128
    px, row_map, lens, _, dispatched, _, pprobs = turbo.ops.moe_permute(
        s["x"], s["topk_idx"], num_local_experts=case["experts"], num_topk=case["topk"], pad_multiple=pad,
        probs=s["probs"], probs_layout="topk")
    h = first(px, s["w1"], lens, trans_b=True, config=s["config"])
    y = second(h, pprobs, s["w2"], lens, trans_b=True, config=s["config"], act_type="silu")
    out, _ = turbo.ops.moe_unpermute(y, row_map, dispatched, restore_shape=s["x"].shape,
                                     num_local_experts=case["experts"], pad_multiple=pad)
    return (out.detach(), *torch.autograd.grad(out, (s["x"], s["w1"], s["w2"], s["probs"]), s["grad"]))


def _run_quantize(s, case):
    x, recipe, way, hp = s["x"], case["recipe"], case["direction"], s["x"].dtype
    fp4 = recipe == "mxfp4"
    gran = _config(recipe).granularity
    kw = {"blockwise": dict(block_size=128), "mxfp8": dict(block_size=32), "mxfp4": dict(block_size=32)}.get(recipe, {})
    axis = {} if recipe == "tensorwise" else dict(axis=0 if way == "column" else 1)
    if way == "both":
        codes = (turbo.ops.quantize_fp4_with_trans if fp4 else turbo.ops.quantize_fp8_with_trans)(
            x, _code_dtype(recipe), gran, **kw)
    else:
        codes = (turbo.ops.quantize_fp4 if fp4 else turbo.ops.quantize_fp8)(x, _code_dtype(recipe), gran, **kw, **axis)
    back = (turbo.ops.dequantize_fp4 if fp4 else turbo.ops.dequantize_fp8)(codes[0], hp, gran, scale_inv=codes[1], **kw, **axis)
    if gran == _G.MX_BLOCKWISE:  # packed codes and exponents are bytes
        codes = tuple(c.view(torch.uint8) for c in codes)
    return (*codes, back)


def run(state):
    case = state["case"]
    return {"linear": _run_linear, "experts": _run_experts, "moe": _run_moe, "quantize": _run_quantize}[case["kind"]](state, case)


def work(case):
    hp, code = _SIZE[case["dtype"]], _CODE[case["recipe"]]
    if case["kind"] == "quantize":
        one = case["rows"] * case["cols"]
        # the input once, each direction's codes once, the de-quantizer's codes once and its output once
        return {"bytes": one * (hp + code * (2 if case["direction"] == "both" else 1) + code + hp), "flops": 0}
    if case["kind"] == "moe":
        rows, h, f = case["tokens"] * case["topk"], case["hidden"], case["inter"]
        weights = 3 * case["experts"] * h * f
        # tokens, gradients and their counterparts once; weights and their gradients once; the rows of both
        # products are the path's own intermediates
        return {"bytes": hp * (4 * case["tokens"] * h + 2 * weights), "flops": 3 * 2 * rows * 3 * h * f}
    t, n, k = case["tokens"], case["n"], case["k"]
    g = case.get("groups", 1)
    if case["kind"] == "experts" and not case["train"]:
        g = sum(1 for v in group_lens(g, t, case["spread"], 0) if v)  # idle experts' weights stay where they are
    if case["train"]:
        grad_w = 8 if case.get("main_grad") else hp
        return {"bytes": hp * (2 * t * k + 2 * t * n + g * n * k) + grad_w * g * n * k, "flops": 6 * t * n * k}
    return {"bytes": hp * (t * k + t * n) + code * g * n * k, "flops": 2 * t * n * k}


def tolerance(case):
    """Quantizers give the same bytes. Products: about four times what the path differs from itself when
    the reduction axes are permuted (fp32 sums in another order, up to 2.7e-4 and one unit in the last
    place of the 16-bit result); an expert layer quantizes what its first product rounded differently
    (up to 2.5e-4, 0.048 at the largest)."""
    if case["kind"] == "quantize":
        return "exact"
    return {"rel": 1e-3, "max": 0.2 if case["kind"] == "moe" else 0.031}
