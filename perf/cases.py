"""The work that this library is used for, as cases that can be timed: weight syncs, checkpoint conversion in both
directions, quantization-aware training steps and activation quantization, from one decode token up to whole layers of
experts.

`listed()` names the cases, `draw(rng)` makes more of the same ranges, `prepare(case, seed)` builds what a program holds
before the call, `run(state)` is one pass through the public entry points.  Shapes are those of the repository's
benchmark configurations and tests, or generic.
"""

from __future__ import annotations

import math
import os
from argparse import Namespace

import torch

from miles_amd import launch
from miles_amd.kernels.quant import fake_quant as fq
from miles_amd.kernels.quant.fp8_act_quant import act_quant, fp8_simulate_qat
from miles_amd.kernels.quant.int4_fake import fake_int4_quant_cuda, pack_layer
from miles_amd.megatron_to_hf.processors.quantizer_nvfp4 import quantize_nvfp4
from miles_amd.tools.convert_hf_to_fp8 import quant_fp8
from miles_amd.tools.convert_kimi_int4_to_bf16 import _dequantize_tensor
from miles_amd.tools.convert_mxfp4_to_fp8 import cast_e2m1fn_to_e4m3fn
from miles_amd.tools.fp8_cast_bf16 import weight_dequant
from miles_amd.utils.mxfp4 import dequantize_mxfp4, quantize_mxfp4
from miles_amd.utils.mxfp8 import mxfp8_quantize, requantize_fp8_block_to_mxfp8
from miles_amd.utils.nvfp4_fake_qat import NVFP4_FAKE_QAT_FLAG, maybe_fake_quantize_nvfp4_weight_tensors
from miles_amd.weight_update.updater import WeightUpdater

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}
FAKE_QUANT = {"fp8": fq.fake_quant_fp8, "fp4": fq.fake_quant_fp4, "kv": fq.fake_quant_compressed_kv}


def listed():
    return [
        # One generated token's hidden state on its way into an FP8 matrix product: the smallest call, launch and host cost.
        {"name": "act_token", "op": "act_quant", "rows": 1, "cols": 7168, "block": 128, "pow2": True, "dtype": "bf16"},
        # Quantization-aware training, activations of a packed batch, forward and backward.
        {"name": "train_fake_fp8", "op": "fake_quant", "kind": "fp8", "rows": 32768, "cols": 2560, "dtype": "bf16"},
        # The compressed key/value stream of an odd number of tokens, simulated FP8, forward and backward.
        {"name": "train_kv_simulate", "op": "simulate", "rows": 4099, "cols": 512, "block": 64, "dtype": "bf16"},
        # NVFP4 quantization-aware training: the weights of a grouped linear layer (the sixteen experts of one of eight
        # ranks, Qwen3-30B-A3B) in front of its matrix product, forward and backward.
        {"name": "qat_nvfp4", "op": "qat_nvfp4", "count": 16, "rows": 1536, "cols": 2048, "four_over_six": False,
         "dtype": "bf16"},
        # The same with Four Over Six block scaling and a few large experts (DeepSeek-V3-shaped).
        {"name": "qat_nvfp4_four_over_six", "op": "qat_nvfp4", "count": 4, "rows": 4096, "cols": 7168,
         "four_over_six": True, "dtype": "bf16"},
        # A trainer's FP8 weight sync: three decoder layers of Qwen3-4B, fused QKV and gate/up as the trainer stores them.
        {"name": "sync_fp8_dense", "op": "sync_dense", "layers": 3, "hidden": 2560, "heads": 32, "groups": 8, "ffn": 9728},
        # MXFP8 sync of Qwen3-30B-A3B's experts (many small matrices) into packed transport payloads: the largest case.
        {"name": "sync_mxfp8_experts", "op": "sync_moe", "quant": "mxfp8", "layers": 2, "experts": 128, "hidden": 2048,
         "ffn": 768},
        # INT4 sync of Kimi-K2-shaped experts (few large matrices) into packed transport payloads.
        {"name": "sync_int4_experts", "op": "sync_moe", "quant": "int4", "layers": 1, "experts": 16, "hidden": 7168,
         "ffn": 2048},
        # Checkpoint conversion to NVFP4, a stack of DeepSeek-V3-shaped experts with a global scale each.
        {"name": "convert_nvfp4_stack", "op": "nvfp4_stack", "count": 32, "rows": 2048, "cols": 7168,
         "four_over_six": False, "dtype": "bf16"},
        # Checkpoint conversion to FP8 128x128 of matrices whose sides are no multiple of anything.
        {"name": "convert_fp8_ragged", "op": "convert", "method": "fp8_block", "count": 12, "rows": 1545, "cols": 2563,
         "dtype": "bf16"},
        # Checkpoint conversion to MXFP8 of a checkpoint kept in fp32.
        {"name": "convert_mxfp8_fp32", "op": "convert", "method": "mxfp8", "count": 12, "rows": 2560, "cols": 4096,
         "dtype": "fp32"},
        # An FP8 checkpoint's layer back to bf16.
        {"name": "decode_fp8", "op": "decode", "kind": "fp8_bf16", "count": 24, "rows": 2048, "cols": 7168},
    ]


# ---- drawn cases ---------------------------------------------------------------------------------------------------
MAX_ELEMENTS = 1 << 27          # of a drawn case outside the syncs (a sync: four times that); the largest listed has 2^30.2


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _multiple(rng, low, high, unit):
    """A multiple of `unit`, its logarithm spread over the range."""
    return max(1, _log(rng, low, high) // unit) * unit


def _fit(case, limit=MAX_ELEMENTS):
    """Halve the largest count of a drawn case until it costs no more than it may."""
    while case.get("count", 1) * case["rows"] * case["cols"] > limit:
        if case.get("count", 1) > 1:
            case["count"] //= 2
        else:
            case["rows"] = max(1, case["rows"] // 2)
    return case


def draw(rng):
    op = rng.choice(["act_quant", "fake_quant", "simulate", "qat_nvfp4", "qat_int4", "sync_dense", "sync_moe",
                     "nvfp4_stack", "convert", "convert", "convert", "decode", "decode"])
    any_dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
    half = rng.choice(["bf16", "bf16", "fp16"])
    if op == "act_quant":
        block = rng.choice([32, 64, 128, 128])
        return _fit({"op": op, "rows": _log(rng, 1, 16384), "cols": _multiple(rng, block, 16384, block), "block": block,
                     "pow2": rng.random() < 0.5, "dtype": half})
    if op == "fake_quant":
        return _fit({"op": op, "kind": rng.choice(["fp8", "fp4", "kv"]), "rows": _log(rng, 1, 16384),
                     "cols": _multiple(rng, 64, 16384, 32), "dtype": any_dtype})
    if op == "simulate":
        return _fit({"op": op, "rows": _log(rng, 16, 32768), "cols": _multiple(rng, 128, 2048, 64), "block": 64, "dtype": half})
    if op == "qat_nvfp4":
        return _fit({"op": op, "count": _log(rng, 1, 24), "rows": _log(rng, 16, 8192), "cols": _multiple(rng, 64, 8192, 16),
                     "four_over_six": rng.random() < 0.4, "dtype": half})
    if op == "qat_int4":
        group = rng.choice([32, 64, 128])
        return _fit({"op": op, "rows": _log(rng, 16, 16384), "cols": _multiple(rng, 128, 16384, group), "group": group,
                     "symmetric": rng.random() < 0.7, "dtype": any_dtype})
    if op == "sync_dense":
        groups = rng.choice([1, 2, 4, 8])
        return {"op": op, "layers": rng.randint(1, 3), "hidden": _multiple(rng, 512, 4096, 64), "heads": groups * rng.choice([2, 4, 8]),
                "groups": groups, "ffn": _multiple(rng, 512, 10240, 64)}
    if op == "sync_moe":
        case = {"op": op, "quant": rng.choice(["mxfp8", "int4", "int4_asym", "mxfp4"]), "layers": rng.randint(1, 2), "experts": _log(rng, 4, 128),
                "hidden": _multiple(rng, 512, 7168, 128), "ffn": _multiple(rng, 256, 2048, 128)}
        while case["layers"] * case["experts"] * case["hidden"] * case["ffn"] * 3 > 4 * MAX_ELEMENTS:
            case["experts"] //= 2
        return case
    if op == "nvfp4_stack":
        return _fit({"op": op, "count": _log(rng, 1, 64), "rows": _log(rng, 64, 7168), "cols": _multiple(rng, 64, 7168, 16),
                     "four_over_six": rng.random() < 0.3, "dtype": any_dtype})
    if op == "convert":
        method = rng.choice(["fp8_block", "fp8_block", "fp8_channel", "fp8_tensor", "mxfp8", "mxfp8", "int4", "int4_asym", "mxfp4"])
        rows, cols = _log(rng, 64, 8192), _log(rng, 256, 16384)
        if method.startswith("fp8"):
            cols = cols if rng.random() < 0.3 else max(64, cols // 64 * 64)          # odd widths among them
        elif method.startswith("int4"):
            cols = max(128, cols // 128 * 128)
            rows = max(8, rows // 8 * 8) if method == "int4_asym" else rows
        else:
            cols = max(32, cols // 32 * 32)
        return _fit({"op": op, "method": method, "count": _log(rng, 1, 16), "rows": rows, "cols": cols, "dtype": any_dtype})
    kind = rng.choice(["fp8_bf16", "int4_bf16", "mxfp4_bf16", "mxfp4_fp8", "fp8_mxfp8"])
    unit = 128 if kind == "mxfp4_fp8" else 1
    rows, cols = _multiple(rng, 128, 8192, unit), _multiple(rng, 256, 8192, 128)
    if kind == "fp8_bf16" and rng.random() < 0.3:
        cols += rng.randint(1, 127)
    return _fit({"op": "decode", "kind": kind, "count": _log(rng, 1, 32), "rows": rows, "cols": cols})


# ---- inputs --------------------------------------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _weight(g, shape, dtype=torch.bfloat16, std=0.02):
    """N(0, std) with one entry in a thousand twenty times as large."""
    x = torch.randn(shape, generator=g, device="cuda")
    x *= torch.where(torch.rand(shape, generator=g, device="cuda") < 0.001, 20.0 * std, std)
    return x.to(dtype)


def _activation(g, shape, dtype):
    """Tokens of very different magnitude: N(0, 1) scaled by a log-normal factor per row."""
    x = torch.randn(shape, generator=g, device="cuda")
    x *= torch.exp(torch.randn((shape[0], 1), generator=g, device="cuda"))
    return x.to(dtype)


# ---- one builder per operation: seed -> the pass as a callable ---------------------------------------------------------
def _prepare_act_quant(c, g):
    x = _activation(g, (c["rows"], c["cols"]), DTYPES[c["dtype"]])
    block, fmt = c["block"], "ue8m0" if c["pow2"] else None
    return lambda: act_quant(x, block, fmt)


def _forward_backward(f, x, gy):
    """A training step's share: the forward, and the gradient through it."""
    x.requires_grad_(True)

    def step():
        y = f(x)
        return y, torch.autograd.grad(y, x, gy)[0]

    return step


def _prepare_fake_quant(c, g):
    shape, dtype = (c["rows"], c["cols"]), DTYPES[c["dtype"]]
    return _forward_backward(FAKE_QUANT[c["kind"]], _activation(g, shape, dtype), _activation(g, shape, dtype))


def _prepare_simulate(c, g):
    shape, dtype, block = (c["rows"], c["cols"]), DTYPES[c["dtype"]], c["block"]
    return _forward_backward(lambda x: fp8_simulate_qat(x, block), _activation(g, shape, dtype), _activation(g, shape, dtype))


def _block_scaling(c):
    """The value of the environment variable by which a program selects Four Over Six or plain block scaling."""
    return "weights" if c["four_over_six"] else "none"


def _prepare_qat_nvfp4(c, g):
    shape, dtype = (c["rows"], c["cols"]), DTYPES[c["dtype"]]
    weights = [_weight(g, shape, dtype).requires_grad_(True) for _ in range(c["count"])]
    gys = [_activation(g, shape, dtype) for _ in range(c["count"])]
    mode = _block_scaling(c)

    def step():
        os.environ["NVTE_NVFP4_4OVER6"], os.environ[NVFP4_FAKE_QAT_FLAG] = mode, "1"
        ys = maybe_fake_quantize_nvfp4_weight_tensors(weights)
        return ys, torch.autograd.grad(ys, weights, gys)

    return step


def _prepare_qat_int4(c, g):
    x, block, sym = _weight(g, (c["rows"], c["cols"]), DTYPES[c["dtype"]]), (1, c["group"]), c["symmetric"]

    def call():
        out, scale, zero = fake_int4_quant_cuda(x, block, sym)
        return (out, scale) if sym else (out, scale, zero)        # the symmetric form leaves `zero` unwritten

    return call


def _sync(args, weights, model_name, quantization_config, packed, basenames=None):
    """A trainer's updater after its first sync: the plan is recorded.  Every bucket keeps an arena of its own, so that
    the buckets of one sync can be returned together."""
    sent = []
    updater = WeightUpdater(args, weights_getter=lambda: weights, model_name=model_name, quantization_config=quantization_config,
                            send_bucket=sent.append, packed_weight_basenames=basenames, packed_buckets=packed, plan_arenas=None)
    updater.update_weights()

    def call():
        sent.clear()
        updater.update_weights()
        if packed:
            return [bucket.get_flattened_tensor() for bucket in sent]
        return [tensor for bucket in sent for _name, tensor in bucket]

    return call


def _args(c, heads, groups):
    return Namespace(hidden_size=c["hidden"], num_attention_heads=heads, num_query_groups=groups, kv_channels=128, vocab_size=1024,
                     num_layers=c["layers"], update_weight_buffer_size=512 * 1024**2, q_lora_rank=None)


def _prepare_sync_dense(c, g):
    h, ffn, heads, groups = c["hidden"], c["ffn"], c["heads"], c["groups"]
    one = lambda n: torch.ones(n, device="cuda", dtype=torch.bfloat16)  # noqa: E731
    w = {"module.module.embedding.word_embeddings.weight": _weight(g, (1024, h))}       # handed on as it is
    for i in range(c["layers"]):
        at = f"module.module.decoder.layers.{i}."
        w[at + "self_attention.linear_qkv.layer_norm_weight"] = one(h)
        w[at + "self_attention.linear_qkv.weight"] = _weight(g, ((heads + 2 * groups) * 128, h))
        w[at + "self_attention.q_layernorm.weight"] = one(128)
        w[at + "self_attention.k_layernorm.weight"] = one(128)
        w[at + "self_attention.linear_proj.weight"] = _weight(g, (h, heads * 128))
        w[at + "mlp.linear_fc1.layer_norm_weight"] = one(h)
        w[at + "mlp.linear_fc1.weight"] = _weight(g, (2 * ffn, h))
        w[at + "mlp.linear_fc2.weight"] = _weight(g, (h, ffn))
    w["module.module.decoder.final_layernorm.weight"] = one(h)
    config = {"quant_method": "fp8", "activation_scheme": "dynamic", "fmt": "e4m3", "weight_block_size": [128, 128]}
    return _sync(_args(c, heads, groups), w, "qwen3", config, packed=False)


def _pack_quantized(symmetric):
    return {"quant_method": "compressed-tensors", "format": "pack-quantized", "config_groups": {"group_0": {"weights": {
        "group_size": 128, "symmetric": symmetric, "num_bits": 4, "type": "int"}}}}


MOE_QUANT = {
    "mxfp8": ("qwen3moe", {"quant_method": "mxfp8"}),
    "int4": ("kimi_k2", _pack_quantized(True)),
    "int4_asym": ("kimi_k2", _pack_quantized(False)),
    "mxfp4": ("kimi_k2", {"quant_method": "compressed-tensors", "format": "mxfp4-pack-quantized", "config_groups": {
        "group_0": {"weights": {"group_size": 32, "symmetric": True, "num_bits": 4, "type": "float",
                                "scale_dtype": "torch.uint8"}}}}),
}


def _prepare_sync_moe(c, g):
    name, config = MOE_QUANT[c["quant"]]
    w, basenames = {}, set()
    for layer in range(c["layers"]):
        for e in range(c["experts"]):
            at = f"module.module.decoder.layers.{layer}.mlp.experts."
            w[at + f"linear_fc1.weight{e}"] = _weight(g, (2 * c["ffn"], c["hidden"]))
            w[at + f"linear_fc2.weight{e}"] = _weight(g, (c["hidden"], c["ffn"]))
            basenames.update(f"model.layers.{layer}.mlp.experts.{e}.{p}_proj" for p in ("gate", "up", "down"))
    return _sync(_args(c, 32, 4), w, name, config, packed=True, basenames=None if c["quant"] == "mxfp8" else basenames)


def _prepare_nvfp4_stack(c, g):
    stack = torch.stack([_weight(g, (c["rows"], c["cols"]), DTYPES[c["dtype"]]) for _ in range(c["count"])])
    mode = _block_scaling(c)

    def call():
        os.environ["NVTE_NVFP4_4OVER6"] = mode
        with launch.deferred():
            return quantize_nvfp4(stack)

    return call


CONVERT = {
    "fp8_block": lambda w: quant_fp8(w, "block", [128, 128]),
    "fp8_channel": lambda w: quant_fp8(w, "channel"),
    "fp8_tensor": lambda w: quant_fp8(w, "tensor"),
    "mxfp8": mxfp8_quantize,
    "int4": lambda w: pack_layer(w, 128, True)[:2],
    "int4_asym": lambda w: pack_layer(w, 128, False),
    "mxfp4": lambda w: quantize_mxfp4(w, 32),
}


def _deferred(function, inputs):
    """A checkpoint shard's tensors, submitted together as the converters do."""

    def call():
        with launch.deferred():
            return [function(*each) for each in inputs]

    return call


def _prepare_convert(c, g):
    return _deferred(CONVERT[c["method"]], [(_weight(g, (c["rows"], c["cols"]), DTYPES[c["dtype"]]),) for _ in range(c["count"])])


def _prepare_decode(c, g):
    """The codes and scales come from quantizing weights, as those of a checkpoint do."""
    weights = [_weight(g, (c["rows"], c["cols"])) for _ in range(c["count"])]
    if c["kind"] in ("fp8_bf16", "fp8_mxfp8"):
        back = weight_dequant if c["kind"] == "fp8_bf16" else requantize_fp8_block_to_mxfp8
        return _deferred(back, [quant_fp8(w, "block", [128, 128]) for w in weights])
    if c["kind"] == "int4_bf16":
        return _deferred(lambda p, s: _dequantize_tensor(p, s, (c["rows"], c["cols"]), 128),
                         [(p, s.float()) for p, s, _ in (pack_layer(w, 128) for w in weights)])
    pairs = [quantize_mxfp4(w, 32) for w in weights]
    if c["kind"] == "mxfp4_bf16":
        return _deferred(lambda p, s: dequantize_mxfp4(p, s, 32), pairs)
    return _deferred(cast_e2m1fn_to_e4m3fn, [(p.view(torch.int8), s) for p, s in pairs])


PREPARE = {"act_quant": _prepare_act_quant, "fake_quant": _prepare_fake_quant, "simulate": _prepare_simulate,
           "qat_nvfp4": _prepare_qat_nvfp4, "qat_int4": _prepare_qat_int4, "sync_dense": _prepare_sync_dense,
           "sync_moe": _prepare_sync_moe, "nvfp4_stack": _prepare_nvfp4_stack, "convert": _prepare_convert,
           "decode": _prepare_decode}


def prepare(case, seed):
    return {"pass": PREPARE[case["op"]](case, _generator(seed))}


def run(state):
    return state["pass"]()


# ---- what a pass cannot do without -----------------------------------------------------------------------------------
OUT_BYTES = {"fp8_block": 1 + 4 / 16384, "fp8_channel": 1, "fp8_tensor": 1, "mxfp8": 1 + 1 / 32, "int4": 0.5 + 2 / 128,
             "int4_asym": 0.5 + 3 / 128, "mxfp4": 0.5 + 1 / 32}
DECODE_BYTES = {"fp8_bf16": 1 + 4 / 16384 + 2, "int4_bf16": 0.5 + 4 / 128 + 2, "mxfp4_bf16": 0.5 + 1 / 32 + 2,
                "mxfp4_fp8": 0.5 + 1 / 32 + 1 + 4 / 16384, "fp8_mxfp8": 1 + 4 / 16384 + 1 + 1 / 32}


def work(case):
    """Every input byte read once, every output byte written once; a comparison and a product per element, and for Four
    Over Six two candidates with an error term each."""
    op = case["op"]
    if op == "sync_dense":
        h, per_head = case["hidden"], 128
        n = case["layers"] * ((2 * case["heads"] + 2 * case["groups"]) * per_head * h + 3 * case["ffn"] * h)
        return {"bytes": n * (2 + OUT_BYTES["fp8_block"]), "flops": 2 * n}
    if op == "sync_moe":
        n = case["layers"] * case["experts"] * 3 * case["ffn"] * case["hidden"]
        return {"bytes": n * (2 + OUT_BYTES[case["quant"]]), "flops": 2 * n}
    n = case.get("count", 1) * case["rows"] * case["cols"]
    if op == "decode":
        return {"bytes": n * DECODE_BYTES[case["kind"]], "flops": n}
    size = BYTES[case["dtype"]]
    if op == "act_quant":
        return {"bytes": n * (size + 1 + 4 / case["block"]), "flops": 2 * n}
    if op in ("fake_quant", "simulate"):
        return {"bytes": n * 2 * size, "flops": 3 * n}        # the backward hands the gradient on untouched
    if op == "qat_nvfp4":
        return {"bytes": n * 2 * size, "flops": (10 if case["four_over_six"] else 3) * n}
    if op == "qat_int4":
        return {"bytes": n * (2 * size + (1 if case["symmetric"] else 2) * size / case["group"]), "flops": 2 * n}
    if op == "nvfp4_stack":
        return {"bytes": n * (size + 0.5 + 1 / 16), "flops": (9 if case["four_over_six"] else 2) * n}
    return {"bytes": n * (size + OUT_BYTES[case["method"]]), "flops": 2 * n}


def tolerance(case):
    """Codes, scales and dequantized values are defined byte for byte; gradients pass through untouched."""
    return "exact"
