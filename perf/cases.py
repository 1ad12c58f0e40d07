"""The work that users of this framework have it do, as cases that can be timed and compared.

Sizes are those of the models the framework serves -- LLaMA-7B and 13B, CLIP ViT-L/14, Whisper
large -- through the public operator interface (``adrastea_amd.GpuKernels``), with the views a
model's forward pass makes: weights ``[N, K]`` handed over as their permuted view, heads as views
of ``[tokens, width]`` tensors.  A program keeps its weights, their views, its operator options and
its activation buffers from call to call; the views of activations are made at the call, as the
tensors behind them change from layer to layer.
"""
import math

import torch

from adrastea_amd import (GpuKernels, MatmulLoad, MatmulMask, MatmulOptions, MatmulStore, TensorView)

BLOCK = 32  # weights per scale of the u8 format

# (width, inner width of the MLP) of the decoder-only models, (heads, head dimension) of attention
LLAMA_7B = (4096, 11008)
LLAMA_13B = (5120, 13824)
MLP_SIZES = ((768, 3072), (1024, 4096), (1280, 5120))   # CLIP text, CLIP vision, Whisper large
HEADS = ((32, 128), (40, 128), (12, 64), (16, 64), (20, 64))


def listed():
    return [
        # The query/key/value projection of CLIP's text encoder on one prompt of 77 positions: the
        # smallest product a model issues, where the call itself and the launch are the time.
        {"name": "clip_text_qkv", "kind": "product", "rows": 77, "k": 768, "n": 2304, "store": "bias"},
        # The MLP of CLIP's vision tower on a batch of eight images of 257 positions (2056 rows, no
        # multiple of a tile), with the activation and the residual fused into the stores.
        {"name": "clip_vision_mlp", "kind": "mlp", "rows": 2056, "width": 1024, "inner": 4096,
         "activation": "quick_gelu"},
        # The five products of a LLaMA-7B layer over a prompt of 2048 tokens, fp16 weights: the
        # largest work, bound by the matrix cores.
        {"name": "llama7b_prefill_f16", "kind": "layer", "weights": "f16", "rows": 2048, "width": 4096,
         "inner": 11008},
        # The same layer for one generated token: every weight is read for one row.
        {"name": "llama7b_token_f16", "kind": "layer", "weights": "f16", "rows": 1, "width": 4096,
         "inner": 11008},
        # The layer over a prompt with u8 weights, dequantised inside the products.
        {"name": "llama7b_prefill_u8", "kind": "layer", "weights": "u8", "rows": 2048, "width": 4096,
         "inner": 11008},
        # One generated token with u8 weights: the usual way to serve one user.
        {"name": "llama7b_token_u8", "kind": "layer", "weights": "u8", "rows": 1, "width": 4096,
         "inner": 11008},
        # Sixteen sequences that generate together with u8 weights.
        {"name": "llama7b_batch16_u8", "kind": "layer", "weights": "u8", "rows": 16, "width": 4096,
         "inner": 11008},
        # Attention of a LLaMA-7B layer over 2048 tokens as the three calls the model makes: masked and
        # scaled scores, softmax in place, product with the values.
        {"name": "llama7b_attention_calls", "kind": "attention_calls", "heads": 32, "d": 128, "m": 2048,
         "n": 2048, "causal": True},
        # The same attention as the one fused call.
        {"name": "llama7b_attention", "kind": "attention", "heads": 32, "d": 128, "m": 2048, "n": 2048,
         "causal": True},
        # One generated token against a context of 2047 keys (odd, as it grows by one with each token).
        {"name": "llama7b_token_attention", "kind": "attention", "heads": 32, "d": 128, "m": 1, "n": 2047,
         "causal": False},
        # Self-attention of Whisper's encoder over 1500 frames (head dimension 64, no mask, ragged).
        {"name": "whisper_encoder_attention", "kind": "attention", "heads": 20, "d": 64, "m": 1500,
         "n": 1500, "causal": False},
        # A checkpoint's matrix turned into the u8 format, back, and the loss of it measured on the
        # device: what loading a model with u8 weights does for each of its matrices.
        {"name": "checkpoint_u8", "kind": "checkpoint", "rows": 11008, "cols": 4096},
    ]


def _spread(rng, low, high):
    """An integer of [low, high], even over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))))


def draw(rng):
    kind = rng.choice(("product", "mlp", "layer", "layer", "layer", "attention_calls", "attention",
                       "attention", "attention", "checkpoint"))
    if kind == "product":
        k, inner = rng.choice(MLP_SIZES)
        return {"kind": kind, "rows": _spread(rng, 1, 2056), "k": k, "n": rng.choice((k, 3 * k, inner)),
                "store": rng.choice(("bias", "identity", "scale"))}
    if kind == "mlp":
        width, inner = rng.choice(MLP_SIZES)
        return {"kind": kind, "rows": _spread(rng, 16, 2056), "width": width, "inner": inner,
                "activation": rng.choice(("quick_gelu", "gelu"))}
    if kind == "layer":
        width, inner = rng.choice((LLAMA_7B, LLAMA_13B))
        # (a 13B layer has 1.57 times the weights of a 7B layer)
        return {"kind": kind, "weights": rng.choice(("f16", "u8")),
                "rows": _spread(rng, 1, 2048 if (width, inner) == LLAMA_7B else 1280),
                "width": width, "inner": inner}
    if kind == "checkpoint":
        width, inner = rng.choice((LLAMA_7B,) + MLP_SIZES)
        rows, cols = rng.choice(((width, width), (inner, width), (width, inner)))
        return {"kind": kind, "rows": rows - rng.choice((0, 0, 1, 3)), "cols": cols}
    heads, d = rng.choice(HEADS)
    most = 2048 if heads * d <= 4096 else 1600
    shape = rng.choice(("self", "causal", "few"))
    if shape == "few":    # a few query rows against a longer context: generation, cross attention
        return {"kind": kind, "heads": heads, "d": d, "m": _spread(rng, 1, 448), "n": _spread(rng, 64, most),
                "causal": False}
    s = _spread(rng, 64, most)
    return {"kind": kind, "heads": heads, "d": d, "m": s, "n": s, "causal": shape == "causal"}


# ---- inputs ----------------------------------------------------------------------------------

def _layer_shapes(width, inner):
    """(name, K, N) of the products of one layer; the gate and up projections have one shape."""
    return (("qkv", width, 3 * width), ("o", width, width), ("gate", width, inner),
            ("up", width, inner), ("down", inner, width))


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    s = {"case": case, "kernels": GpuKernels()}

    def normal(*shape, std=1.0):
        return torch.randn(*shape, dtype=torch.float16, device="cuda", generator=g) * std

    def zeros(*shape):  # (the reference's tensors start at zero as well)
        return torch.zeros(*shape, dtype=torch.float16, device="cuda")

    def weight(n, k):
        t = normal(n, k, std=1.0 / math.sqrt(k))
        return TensorView.of(t).permute([1, 0])

    kind = case["kind"]
    if kind == "product":
        rows, k, n = case["rows"], case["k"], case["n"]
        s["x"], s["out"], s["w"] = normal(rows, k), zeros(rows, n), weight(n, k)
        store = {"identity": MatmulStore.Identity(), "scale": MatmulStore.Scale(0.125),
                 "bias": MatmulStore.BetaBias(0.0, TensorView.of(normal(n, std=0.1)))}[case["store"]]
        s["options"] = MatmulOptions.new().store(store)
    elif kind == "mlp":
        rows, width, inner = case["rows"], case["width"], case["inner"]
        s["x"], s["hidden"], s["residual"] = normal(rows, width), zeros(rows, inner), normal(rows, width)
        s["up"], s["down"] = weight(inner, width), weight(width, inner)
        bias = TensorView.of(normal(inner, std=0.1))
        s["up_options"] = MatmulOptions.new().store(
            MatmulStore.QuickGeluBias(bias) if case["activation"] == "quick_gelu"
            else MatmulStore.BetaGeluBias(0.0, bias))
        s["down_options"] = MatmulOptions.new().store(
            MatmulStore.BetaBias(1.0, TensorView.of(normal(width, std=0.1))))
    elif kind == "layer":
        rows = case["rows"]
        s["x"] = {}
        for name, k, n in _layer_shapes(case["width"], case["inner"]):
            if k not in s["x"]:
                s["x"][k] = normal(rows, k)
            if case["weights"] == "f16":
                s[name] = weight(n, k)
            else:
                q = torch.randint(0, 256, (n, k), dtype=torch.uint8, device="cuda", generator=g)
                scales = torch.rand(n, k // BLOCK, device="cuda", generator=g) * 0.019 + 0.001
                s[name] = (q, scales.half())
            # (the attention output and the MLP output are added to the residual stream with fp16
            # weights; the u8 products have no such store)
            s[name + "_out"] = normal(rows, n) if name in ("o", "down") else zeros(rows, n)
        s["options"], s["add"] = MatmulOptions.new(), MatmulOptions.new().store(MatmulStore.Add())
    elif kind in ("attention", "attention_calls"):
        heads, d, m, n = case["heads"], case["d"], case["m"], case["n"]
        s["q"], s["k"], s["v"] = normal(m, heads * d), normal(n, heads * d), normal(n, heads * d)
        s["out"] = zeros(m, heads * d)
        s["scale"] = 1.0 / math.sqrt(d)
        s["mask"] = MatmulMask.CAUSAL if case["causal"] else MatmulMask.NONE
        if kind == "attention_calls":
            s["scores"] = zeros(heads, m, n)
            # LLaMA and CLIP scale the scores, Whisper (20 heads) both operands
            if heads == 20:
                scores = MatmulOptions.new().load(MatmulLoad.Scale(d ** -0.25))
            else:
                scores = MatmulOptions.new().store(MatmulStore.Scale(s["scale"]))
            s["score_options"] = scores.mask(s["mask"])
            s["options"] = MatmulOptions.new()
    elif kind == "checkpoint":
        rows, cols = case["rows"], case["cols"]
        s["w"] = normal(rows, cols, std=1.0 / math.sqrt(cols))
        s["q"] = torch.zeros(rows, cols, dtype=torch.uint8, device="cuda")
        s["scales"], s["back"] = zeros(rows, cols // BLOCK), zeros(rows, cols)
        s["stats"] = torch.zeros(3, dtype=torch.float32, device="cuda")
    else:
        raise ValueError(kind)
    return s


def _heads(t, heads, d):
    """The [heads, tokens, d] view of a [tokens, heads * d] tensor."""
    return TensorView.of(t).shape_cast([t.shape[0], heads, d]).permute([1, 0, 2])


def run(s):
    case, k, view = s["case"], s["kernels"], TensorView.of
    kind = case["kind"]
    if kind == "product":
        k.matmul_f16(view(s["out"]), view(s["x"]), s["w"], s["options"])
        return s["out"]
    if kind == "mlp":
        k.matmul_f16(view(s["hidden"]), view(s["x"]), s["up"], s["up_options"])
        k.matmul_f16(view(s["residual"]), view(s["hidden"]), s["down"], s["down_options"])
        return s["hidden"], s["residual"]
    if kind == "layer":
        outs = []
        for name, width, _ in _layer_shapes(case["width"], case["inner"]):
            x, out = s["x"][width], s[name + "_out"]
            if case["weights"] == "u8":
                q, scales = s[name]
                k.matmul_nt_fp16u8(out, x, q, scales, BLOCK)
            else:
                k.matmul_f16(view(out), view(x), s[name],
                             s["add"] if name in ("o", "down") else s["options"])
            outs.append(out)
        return outs
    if kind == "checkpoint":
        k.quantize_absmax_uint8(s["q"], s["scales"], s["w"])
        k.dequantize_absmax_uint8(s["back"], s["scales"], s["q"])
        s["stats"].zero_()
        k.error_stats_f16(view(s["stats"]), view(s["back"]), view(s["w"]))
        return s["q"], s["scales"], s["back"], s["stats"]
    heads, d = case["heads"], case["d"]
    q, key, value, out = (_heads(s[t], heads, d) for t in ("q", "k", "v", "out"))
    if kind == "attention":
        k.attention_f16(out, q, key, value, s["scale"], 1.0, s["mask"])
        return s["out"]
    scores = view(s["scores"])
    k.matmul_f16(scores, q, key.permute([0, 2, 1]), s["score_options"])
    k.softmax_rows_inplace(scores, 1.0)
    k.matmul_f16(out, scores, value, s["options"])
    return s["scores"], s["out"]


# ---- what a pass cannot do without ---------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "product":
        rows, k, n = case["rows"], case["k"], case["n"]
        return {"bytes": 2 * (rows * k + k * n + rows * n), "flops": 2 * rows * k * n}
    if kind == "mlp":
        rows, width, inner = case["rows"], case["width"], case["inner"]
        # up: x, weights, hidden; down: hidden, weights, the residual read and written
        return {"bytes": 2 * (3 * rows * width + 2 * rows * inner + 2 * width * inner),
                "flops": 4 * rows * width * inner}
    if kind == "layer":
        rows, nbytes, flops = case["rows"], 0, 0
        for name, k, n in _layer_shapes(case["width"], case["inner"]):
            f16 = case["weights"] == "f16"
            nbytes += 2 * k * n if f16 else k * n + 2 * k * n // BLOCK
            nbytes += 2 * rows * (k + n * (2 if f16 and name in ("o", "down") else 1))
            flops += 2 * rows * k * n
        return {"bytes": nbytes, "flops": flops}
    if kind == "checkpoint":
        weights = case["rows"] * case["cols"]
        # quantise 2 -> 1 byte, dequantise 1 -> 2, statistics of 2 + 2, and the scales twice
        return {"bytes": 10 * weights + 4 * weights // BLOCK, "flops": 0}
    heads, d, m, n = case["heads"], case["d"], case["m"], case["n"]
    operands = 2 * heads * d * (2 * m + 2 * n)
    pairs = m * n - (m * (m - 1) // 2 if case["causal"] else 0)  # (causal cases are square)
    if kind == "attention":
        return {"bytes": operands, "flops": 4 * heads * d * pairs}
    # three calls: scores written, read and written again, read; the product with the values knows no mask
    return {"bytes": operands + 4 * 2 * heads * m * n, "flops": 2 * heads * d * (pairs + m * n)}


def tolerance(case):
    """Measured against the same operations in 32- and 64-bit arithmetic, times four.  fp16 results
    that differ only in the order of their 32-bit sums are 2.5e-5 to 6.6e-5 apart (some land on the other
    side of a rounding); u8 products round their weights to fp16 or do not, by the number of rows,
    and fused attention rounds its probabilities and not its scores: 3.2e-4 for either."""
    if case["kind"] == "checkpoint":
        # bytes, scales and restored weights are exact; the means are sums of 32-bit atomics
        return {"rel": 2e-6, "differ": 0.0}
    if case["kind"] == "attention" or case.get("weights") == "u8":
        return {"rel": 1.3e-3}
    return {"rel": 3e-4}
