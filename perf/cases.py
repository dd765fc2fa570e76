"""Workloads of the BitLinear W1.58A8 path, each as a user's program calls it through the Python binding.

`listed()` names the standing workloads, `draw(rng)` gives further ones of the same kinds and ranges, `prepare` makes what
a program holds before the call (inputs, a layer or decoder with its weights), `run` is one pass through the public entry
points, `work` the bytes and operations no implementation can do without, `tolerance` how far another correct
implementation's results may lie from these.

Kinds: `linear` one BitLinear forward; `multi` several layers on one input (q/k/v, gate/up); `decode` a token step of a
decoder stack enqueued launch by launch; `replay` the recorded step; `batch` requests of different lengths through the
inference backend; `quantize` f32 weights to packed ternary ones; `load` a GGUF ternary tensor from host memory into a layer
and the layer's packed bytes back to the host; `activations` the per-tensor dynamic activation quantiser.
"""
import math
import os
import struct
import sys

import torch

# the package lies in the tree this file is used with: the working folder, which need not be this file's own
sys.path.insert(1, os.path.join(os.getcwd(), "bitnet-mlx.rs_amd", "python"))

import bitnet_hip as bh  # noqa: E402

LARGEST_MACS = 8192 * 13824 * 2560  # multiply-adds of the largest listed product; no drawn one has more
STACK_BYTES = 521_011_200  # packed weights of the 30-block stack; no drawn stack has more


def listed():
    return [
        # one token through one attention projection: the smallest call a program makes, launch and host latency only
        {"name": "linear_1x2560_2560", "kind": "linear", "batch": 0, "tokens": 1, "k": 2560, "n": 2560, "norm": False,
         "residual": False, "bias": False},
        # one token through a layer large enough for the memory to be the limit (the output head of a large model)
        {"name": "linear_1x16384_32768", "kind": "linear", "batch": 0, "tokens": 1, "k": 16384, "n": 32768, "norm": False,
         "residual": False, "bias": False},
        # sixteen concurrent sequences, one token each, through the FFN's down projection with the residual added
        {"name": "linear_16x6912_2560", "kind": "linear", "batch": 0, "tokens": 16, "k": 6912, "n": 2560, "norm": False,
         "residual": True, "bias": False},
        # three prompts of 111 tokens as a [b, s, in] tensor, widths that are no multiple of a tile, bias and norm
        {"name": "linear_3x111x3200_8640", "kind": "linear", "batch": 3, "tokens": 111, "k": 3200, "n": 8640, "norm": True,
         "residual": False, "bias": True},
        # a long prompt through the down projection
        {"name": "linear_2048x6912_2560", "kind": "linear", "batch": 0, "tokens": 2048, "k": 6912, "n": 2560, "norm": False,
         "residual": True, "bias": False},
        # several long prompts at once through gate and up: the largest product
        {"name": "multi_8192x2560_6912_6912", "kind": "multi", "tokens": 8192, "k": 2560, "n1": 6912, "n2": 6912, "n3": 0,
         "norm": True},
        # a generation loop: one token through the whole stack, recorded once and replayed
        {"name": "replay_stack30_b1", "kind": "replay", "layers": 30, "hidden": 2560, "ffn": 6912, "q_heads": 20,
         "kv_heads": 5, "head_dim": 128, "tokens": 1},
        # eight sequences decoding together, the step enqueued as it comes (no recording)
        {"name": "decode_stack30_b8", "kind": "decode", "layers": 30, "hidden": 2560, "ffn": 6912, "q_heads": 20,
         "kv_heads": 5, "head_dim": 128, "tokens": 8},
        # a serving loop: twelve requests of one to six rows in one execute_batch
        {"name": "batch_stack30_12_requests", "kind": "batch", "layers": 30, "hidden": 2560, "ffn": 6912, "q_heads": 20,
         "kv_heads": 5, "head_dim": 128, "requests": 12, "rows": 6},
        # converting a checkpoint: one f32 FFN matrix to packed ternary weights and their scale
        {"name": "quantize_6912x2560_absmean", "kind": "quantize", "n": 6912, "k": 2560, "method": "absmean"},
        # loading a model file: one GGUF ternary tensor from host memory, re-tiled, and read back for saving
        {"name": "load_gguf_6912x2560", "kind": "load", "n": 6912, "k": 2560, "in_out": False},
        # quantising the activations of a prompt with one moving-average scale for the tensor
        {"name": "activations_2048x2560_int8", "kind": "activations", "rows": 2048, "cols": 2560, "bits8": True},
    ]


# ---- drawing ----------------------------------------------------------------------------------------

def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    """A feature count: mostly multiples of 64 to 256 as models have them, some multiples of 4, a few odd ones."""
    v = _log_int(rng, lo, hi)
    unit = rng.choice((256, 256, 128, 64, 64, 4, 1))
    return max(unit, v // unit * unit)


def _draw_stack(rng, tokens):
    head_dim = rng.choice((64, 128))
    kv_heads = rng.randint(1, 8)
    q_heads = kv_heads * rng.randint(1, max(1, 4096 // (head_dim * kv_heads)))
    hidden = q_heads * head_dim
    while hidden < 512:
        q_heads, hidden = q_heads + kv_heads, hidden + kv_heads * head_dim
    ffn = max(64, int(hidden * rng.uniform(2.0, 4.0)) // 64 * 64)
    per_layer = (2 * hidden * hidden + 2 * hidden * kv_heads * head_dim + 3 * hidden * ffn) // 4
    layers = _log_int(rng, 2, max(2, min(40, STACK_BYTES // per_layer)))
    return {"layers": layers, "hidden": hidden, "ffn": ffn, "q_heads": q_heads, "kv_heads": kv_heads, "head_dim": head_dim,
            **tokens}


def draw(rng):
    kind = rng.choices(("linear", "multi", "decode", "replay", "batch", "quantize", "load", "activations"),
                       weights=(9, 4, 3, 3, 1, 2, 1, 2))[0]
    if kind == "linear":
        tokens, k, n = _log_int(rng, 1, 8192), _width(rng, 256, 16384), _width(rng, 256, 32768)
        while tokens * n * k > LARGEST_MACS // 2:
            tokens = max(1, tokens // 2)
        batch = rng.randint(1, 4) if tokens <= 2048 and rng.random() < 0.3 else 0
        return {"kind": kind, "batch": batch, "tokens": tokens, "k": k, "n": n, "norm": rng.random() < 0.5,
                "residual": rng.random() < 0.4, "bias": rng.random() < 0.2}
    if kind == "multi":
        tokens, k, n1 = _log_int(rng, 1, 8192), _width(rng, 256, 8192), _width(rng, 256, 14336)
        n2 = n1 if rng.random() < 0.5 else max(64, n1 // 4 // 64 * 64)
        n3 = n2 if n2 != n1 else 0
        while tokens * (n1 + n2 + n3) * k > LARGEST_MACS // 2:
            tokens = max(1, tokens // 2)
        return {"kind": kind, "tokens": tokens, "k": k, "n1": n1, "n2": n2, "n3": n3, "norm": rng.random() < 0.8}
    if kind in ("decode", "replay"):
        return {"kind": kind, **_draw_stack(rng, {"tokens": _log_int(rng, 1, 64)})}
    if kind == "batch":
        return {"kind": kind, **_draw_stack(rng, {"requests": _log_int(rng, 2, 24), "rows": _log_int(rng, 1, 8)})}
    if kind == "quantize":
        return {"kind": kind, "n": _width(rng, 256, 14336), "k": _width(rng, 256, 8192),
                "method": rng.choice(("absmean", "reference"))}
    if kind == "load":
        return {"kind": kind, "n": _width(rng, 256, 14336), "k": _width(rng, 256, 8192), "in_out": rng.random() < 0.3}
    return {"kind": kind, "rows": _log_int(rng, 1, 4096), "cols": _width(rng, 256, 8192), "bits8": rng.random() < 0.6}


# ---- inputs -----------------------------------------------------------------------------------------

def _activations(gen, *shape):
    """Rows ~ N(0, 1) with one value in a hundred twenty times as large."""
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    return torch.where(torch.rand(shape, generator=gen, device="cuda") < 0.01, x * 20.0, x)


def _packed(gen, count):
    """`count` ternary weights, a third of each value, as packed bytes (codes 0, 1, 2; four to a byte)."""
    codes = torch.randint(0, 3, ((count + 3) // 4, 4), generator=gen, device="cuda", dtype=torch.uint8)
    return (codes[:, 0] | (codes[:, 1] << 2) | (codes[:, 2] << 4) | (codes[:, 3] << 6)).contiguous()


def _layer(gen, k, n, bias=False):
    layer = bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n, use_bias=bias))
    layer.set_quantized_weights(_packed(gen, n * k), 0.016)
    if bias:
        layer.update_bias(torch.randn((n,), generator=gen, device="cuda") * 0.1)
    return layer


def _stack(gen, case, max_tokens):
    dec = bh.DecoderProjections(case["layers"], case["hidden"], case["ffn"], case["q_heads"], case["kv_heads"],
                                case["head_dim"], max_tokens=max_tokens)
    for layer in range(case["layers"]):
        for p in range(7):
            n, k = dec.proj_shape(p)
            dec.projection(layer, p).set_quantized_weights(_packed(gen, n * k), 0.016)
        for which in (0, 1):
            dec.set_norm(layer, which, 1.0 + 0.1 * torch.randn((case["hidden"],), generator=gen, device="cuda"))
    return dec


def _request_rows(case):
    """Rows of each request of a `batch` case: 1 .. rows in turn, so that short and long ones follow each other."""
    return [1 + (5 * i) % case["rows"] for i in range(case["requests"])]


def prepare(case, seed):
    bh.init(0)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind = case["kind"]
    if kind in ("linear", "multi"):
        k = case["k"]
        gamma = 1.0 + 0.1 * torch.randn((k,), generator=gen, device="cuda") if case["norm"] else None
        if kind == "multi":
            layers = [_layer(gen, k, n) for n in (case["n1"], case["n2"], case["n3"]) if n]
            return {"kind": kind, "layers": layers, "x": _activations(gen, case["tokens"], k), "gamma": gamma}
        lead = (case["batch"], case["tokens"]) if case["batch"] else (case["tokens"],)
        layer = _layer(gen, k, case["n"], case["bias"])
        residual = torch.randn(lead + (case["n"],), generator=gen, device="cuda") if case["residual"] else None
        return {"kind": kind, "layer": layer, "x": _activations(gen, *lead, k), "gamma": gamma, "residual": residual}
    if kind in ("decode", "replay"):
        dec = _stack(gen, case, case["tokens"])
        x = torch.randn((case["tokens"], case["hidden"]), generator=gen, device="cuda")
        return {"kind": kind, "dec": dec, "x": x, "graph": dec.record(x) if kind == "replay" else None}
    if kind == "batch":
        rows = _request_rows(case)
        backend = bh.create_backend("hip:0")
        backend.optimize_model(_stack(gen, case, 64))
        return {"kind": kind, "backend": backend,
                "inputs": [torch.randn((r, case["hidden"]), generator=gen, device="cuda") for r in rows]}
    if kind == "quantize":
        w = torch.randn((case["n"], case["k"]), generator=gen, device="cuda") * 0.02
        return {"kind": kind, "w": w, "quantizer": bh.BitNetWeightQuantizer() if case["method"] == "reference" else None}
    if kind == "load":
        n, k = case["n"], case["k"]
        header = torch.frombuffer(bytearray(struct.pack("<ff", 0.016, 0.0)), dtype=torch.uint8)
        data = torch.cat([header, _packed(gen, n * k).cpu()])
        return {"kind": kind, "data": data, "layout": bh.LAYOUT_IN_OUT if case["in_out"] else bh.LAYOUT_OUT_IN,
                "layer": bh.BitLinear(bh.BitLinearConfig(in_features=k, out_features=n))}
    precision = bh.QuantizationPrecision.EightBit if case["bits8"] else bh.QuantizationPrecision.OneFiveFiveBit
    quantizer = bh.create_activation_quantizer(bh.ActivationQuantizationConfig(precision=precision))
    return {"kind": kind, "quantizer": quantizer, "x": _activations(gen, case["rows"], case["cols"])}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["layer"].forward(state["x"], gamma=state["gamma"], residual=state["residual"])
    if kind == "multi":
        return bh.forward_multi(state["layers"], state["x"], gamma=state["gamma"])
    if kind == "decode":
        return state["dec"].decode(state["x"])
    if kind == "replay":
        return state["graph"].replay()
    if kind == "batch":
        return state["backend"].execute_batch(state["inputs"])
    if kind == "quantize":
        if state["quantizer"] is not None:
            r = state["quantizer"].quantize(state["w"])
            return {"values": r.values, "packed": r.packed, "scale": r.scales}
        packed, scale, _ = bh.quantize_weights(state["w"])
        return {"packed": packed, "scale": scale}
    if kind == "load":
        state["layer"].load_gguf_ternary(state["data"], layout=state["layout"])
        packed, scale = state["layer"].get_quantized_weights()
        return {"packed": packed, "scale": scale}
    r = state["quantizer"].quantize_dynamic(state["x"])
    return {"values": r.values, "scale": r.scales}


# ---- what a pass cannot do without ------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind in ("linear", "multi"):
        m = case["tokens"] * max(1, case.get("batch", 0))
        k = case["k"]
        n = case["n"] if kind == "linear" else case["n1"] + case["n2"] + case["n3"]
        extra = 4 * k * case["norm"] + 4 * m * n * case.get("residual", False) + 4 * n * case.get("bias", False)
        return {"bytes": 4 * m * k + n * k // 4 + 4 * m * n + extra, "flops": 2 * m * n * k}
    if kind in ("decode", "replay", "batch"):
        m = sum(_request_rows(case)) if kind == "batch" else case["tokens"]
        h, kv = case["hidden"], case["kv_heads"] * case["head_dim"]
        weights = case["layers"] * (2 * h * h + 2 * h * kv + 3 * h * case["ffn"])
        return {"bytes": weights // 4 + 8 * case["layers"] * h + 8 * m * h, "flops": 2 * m * weights}
    if kind == "quantize":
        nk = case["n"] * case["k"]
        return {"bytes": 4 * nk + nk // 4 + (nk if case["method"] == "reference" else 0), "flops": 2 * nk}
    if kind == "load":
        return {"bytes": 2 * ((case["n"] * case["k"] + 3) // 4), "flops": 0}
    count = case["rows"] * case["cols"]
    return {"bytes": 5 * count, "flops": 2 * count}


def tolerance(case):
    """Whole numbers (int8 values, packed bytes) are the same; f32 results agree as 32-bit arithmetic does."""
    return {"rel": 1e-5, "differ": 0.0}
