"""The work a user of this package gives it, as cases that can be timed.

A case is a dict of plain values; `what` says which public entry point one pass goes through:

  linear         one quantised projection applied to a batch of activations: MarlinLinearKernel.apply_weights
                 (GPTQ, AWQ, act-order, 8-bit integer codes, int8 / fp8 activations), apply_fp8_marlin_linear,
                 apply_mxfp8_marlin_linear, apply_fp4_marlin_linear
  decode_layers  the four projections (qkv, o, gate_up, down) of a few decoder layers for one decode step, recorded
                 in a HIP graph as a serving engine records its decode step; a pass is one replay
  moe            one mixture-of-experts layer: fused_marlin_moe
  load_linear    a checkpoint's projection made ready for the kernels: convert_awq_to_standard_format (AWQ),
                 MarlinLinearKernel.process_weights_after_loading
  load_experts   a checkpoint's experts made ready: process_gptq_moe_weights, process_awq_moe_weights

`m` is the number of rows (1 in the decoding of one sequence, up to thousands in a prefill), `k` and `n` the input
and output features, `group` the rows that share a scale (-1: all of them)."""
import math
from types import SimpleNamespace

import torch

from sonar_amd import fused_moe, marlin_linear, marlin_utils_fp4, marlin_utils_fp8, moe_weights
from sonar_amd.scalar_type import scalar_types

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
#: Bits of a stored weight, and of what is stored for each group and column (scales, zero points).
FORMATS = {"gptq": (4, 16), "awq": (4, 20), "act_order": (4, 16), "int8w": (8, 16), "fp8": (8, 16), "mxfp8": (8, 8),
           "mxfp4": (4, 8), "nvfp4": (4, 8), "w4a8_int8": (4, 16), "w4a8_fp8": (4, 16)}
#: The most multiply-adds and the most packed bytes of a drawn case: those of the largest listed ones.
MOST_FLOPS = 2.0 * 8192 * 4096 * 28672
MOST_BYTES = 8 * 3 * 4096 * 14336 // 2


def listed():
    return [
        # one sequence being decoded: the attention output projection of an 8B decoder, the smallest call there is
        {"name": "linear_1_row", "what": "linear", "format": "gptq", "dtype": "bf16", "group": 128, "m": 1, "k": 4096,
         "n": 4096, "bias": False},
        # the decode step of a small batch: the projections of four decoder layers, whose weights (460 MB) no cache holds
        {"name": "decode_layers_16_rows", "what": "decode_layers", "dtype": "bf16", "group": 128, "layers": 4, "m": 16,
         "hidden": 4096, "qkv": 6144, "inter": 14336},
        # a larger decode batch on the widest projection
        {"name": "linear_64_rows", "what": "linear", "format": "gptq", "dtype": "bf16", "group": 128, "m": 64,
         "k": 4096, "n": 28672, "bias": False},
        # a short prompt (or a chunk of one) on an AWQ checkpoint's qkv projection
        {"name": "awq_200_rows", "what": "linear", "format": "awq", "dtype": "fp16", "group": 128, "m": 200, "k": 4096,
         "n": 6144, "bias": False},
        # a mixed batch of decodes and a prompt, small groups, features that are no power of two, a bias
        {"name": "group32_333_rows", "what": "linear", "format": "gptq", "dtype": "bf16", "group": 32, "m": 333,
         "k": 2880, "n": 5760, "bias": True},
        # decoding on a checkpoint that was quantised with act-order
        {"name": "act_order_12_rows", "what": "linear", "format": "act_order", "dtype": "fp16", "group": 128, "m": 12,
         "k": 4096, "n": 11008, "bias": False},
        # decoding on fp8 weights, one scale a column
        {"name": "fp8_8_rows", "what": "linear", "format": "fp8", "dtype": "bf16", "group": -1, "m": 8, "k": 4096,
         "n": 11008, "bias": False},
        # a long prefill on the widest projection: the largest call
        {"name": "prefill_8192_rows", "what": "linear", "format": "gptq", "dtype": "fp16", "group": 128, "m": 8192,
         "k": 4096, "n": 28672, "bias": False},
        # a prefill with 8-bit activations, which are quantised in the call
        {"name": "w4a8_2048_rows", "what": "linear", "format": "w4a8_int8", "dtype": "fp16", "group": 128, "m": 2048,
         "k": 4096, "n": 11008, "bias": False},
        # a decode step of a Mixtral-8x7B-shaped layer
        {"name": "moe_16_tokens", "what": "moe", "format": "gptq", "dtype": "bf16", "group": 128, "tokens": 16,
         "experts": 8, "top_k": 2, "hidden": 4096, "inter": 14336, "activation": "silu", "bias": False},
        # a prefill of MXFP4 experts with the shape and activation of gpt-oss
        {"name": "moe_mxfp4_2000_tokens", "what": "moe", "format": "mxfp4", "dtype": "bf16", "group": 32,
         "tokens": 2000, "experts": 32, "top_k": 4, "hidden": 2880, "inter": 2880, "activation": "swigluoai",
         "bias": True},
        # a model being loaded: one layer's experts
        {"name": "load_experts", "what": "load_experts", "format": "gptq", "dtype": "bf16", "group": 128, "experts": 8,
         "hidden": 4096, "inter": 14336},
    ]


def _between(rng, low, high, step=1):
    """A multiple of `step`, evenly spread over the logarithm of its range."""
    return max(low, min(high, step * round(math.exp(rng.uniform(math.log(low), math.log(high))) / step)))


def draw(rng):
    what = rng.choice(["linear"] * 11 + ["decode_layers"] * 2 + ["moe"] * 4 + ["load_linear"] * 2 + ["load_experts"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if what in ("linear", "load_linear"):
        kinds = ["gptq"] * 5 + ["awq"] * 2 + ["act_order"]
        if what == "linear":
            kinds += ["int8w", "fp8", "mxfp8", "mxfp4", "nvfp4", "w4a8_int8", "w4a8_int8", "w4a8_fp8"]
        kind = rng.choice(kinds)
        group = {"int8w": 128, "fp8": -1, "mxfp8": 32, "mxfp4": 32, "nvfp4": 16, "act_order": 128, "w4a8_int8": 128,
                 "w4a8_fp8": 128}.get(kind) or rng.choice([128, 128, 128, 64, 32, -1] if kind == "gptq" else [128, 128, 64])
        if kind in ("mxfp4", "mxfp8"):
            dtype = "bf16"
        case = {"what": what, "format": kind, "dtype": dtype, "group": group, "k": _between(rng, 1024, 14336, 128),
                "n": _between(rng, 1024, 28672, 64)}
        if what == "linear":
            m = _between(rng, 1, 8192)
            case["m"] = max(1, min(m, int(MOST_FLOPS / (2.0 * case["k"] * case["n"]))))
            case["bias"] = rng.random() < 0.25
        return case
    if what == "decode_layers":
        hidden = _between(rng, 2048, 8192, 256)
        return {"what": what, "dtype": dtype, "group": 128, "layers": rng.choice([2, 3, 4]), "m": _between(rng, 1, 64),
                "hidden": hidden, "qkv": hidden + 2 * rng.choice([512, 1024]), "inter": hidden * 7 // 2}
    kind = rng.choice(["gptq", "gptq", "awq"] if what == "load_experts" else ["gptq", "gptq", "awq", "mxfp4"])
    experts = rng.choice([8, 16, 32, 64])
    hidden = _between(rng, 1024, 4096, 128)
    inter = min(_between(rng, 512, 14336, 128), MOST_BYTES * 2 // (3 * experts * hidden) // 128 * 128)
    case = {"what": what, "format": kind, "dtype": "bf16" if kind == "mxfp4" else dtype,
            "group": 32 if kind == "mxfp4" else 128, "experts": experts, "hidden": hidden, "inter": inter}
    if what == "moe":
        top_k = rng.choice([2, 2, 4, 8])
        tokens = min(_between(rng, 1, 8192), int(MOST_FLOPS / (6.0 * top_k * hidden * inter)))
        case.update(tokens=tokens, top_k=top_k, activation="silu", bias=False)
    return case


# ---------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _codes4(gen, rows, cols):
    """4-bit codes of normally distributed weights, as a quantiser with the offset 8 leaves them."""
    w = torch.randn((rows, cols), device="cuda", generator=gen, dtype=torch.float16)
    return (w * 2.6 + 8.5).floor_().clamp_(0, 15).to(torch.int32)


def _pack_rows(q, bits=4):
    """(R, C) codes -> (R * bits / 32, C) int32, consecutive rows from the low bits up (the GPTQ packing)."""
    per = 32 // bits
    q = q.view(q.shape[0] // per, per, q.shape[1])
    out = q[:, 0].clone()
    for t in range(1, per):
        out |= q[:, t] << (bits * t)
    return out


def _pack_cols(q, order=range(8)):
    """(R, C) 4-bit codes -> (R, C / 8) int32; column 8 j + t in nibble order[t]."""
    q = q.view(q.shape[0], q.shape[1] // 8, 8)
    out = q[..., 0] << (4 * order[0])
    for t in range(1, 8):
        out |= q[..., t] << (4 * order[t])
    return out


_AWQ_ORDER = (0, 4, 1, 5, 2, 6, 3, 7)


def _zero_codes(gen, rows, cols):
    return torch.randint(5, 12, (rows, cols), device="cuda", generator=gen, dtype=torch.int32)


def _scales(gen, shape, dtype):
    return (torch.rand(shape, device="cuda", generator=gen) * 9e-3 + 1e-3).to(dtype)


def _fp4_bytes(gen, rows, cols):
    """(rows, cols / 2) bytes of two float4_e2m1f codes each, of normally distributed values."""
    edges = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device="cuda", dtype=torch.float16)
    w = torch.randn((rows, cols), device="cuda", generator=gen, dtype=torch.float16) * 2
    code = torch.bucketize(w.abs(), edges, out_int32=True).to(torch.uint8) | ((w < 0).to(torch.uint8) << 3)
    return code[:, 0::2] | (code[:, 1::2] << 4)


def _exponents(gen, shape):
    return torch.randint(117, 122, shape, device="cuda", generator=gen, dtype=torch.uint8)


def _checkpoint_linear(case, gen):
    """The tensors of a GPTQ / AWQ checkpoint's projection, as they lie in its files."""
    k, n, kind, dtype = case["k"], case["n"], case["format"], DTYPES[case["dtype"]]
    groups = 1 if case["group"] == -1 else k // case["group"]
    raw = {"scales": _scales(gen, (groups, n), dtype)}
    if kind == "int8w":
        raw["qweight"] = torch.randint(-2 ** 31, 2 ** 31 - 1, (k // 4, n), device="cuda", generator=gen, dtype=torch.int32)
        raw["scales"] = raw["scales"] * 0.0625
    elif kind == "awq":
        raw["qweight"] = _pack_cols(_codes4(gen, k, n), _AWQ_ORDER)
        raw["qzeros"] = _pack_cols(_zero_codes(gen, groups, n), _AWQ_ORDER)
    else:
        raw["qweight"] = _pack_rows(_codes4(gen, k, n))
    if kind == "act_order":
        raw["g_idx"] = (torch.randperm(k, device="cuda", generator=gen) // case["group"]).to(torch.int32)
    return raw


def _linear_kernel(case):
    kind = case["format"]
    k, n = case["k"], case["n"]
    return marlin_linear.MarlinLinearKernel(marlin_linear.MPLinearLayerConfig(
        full_weight_shape=(k, n), partition_weight_shape=(k, n),
        weight_type={"awq": scalar_types.uint4, "int8w": scalar_types.uint8b128}.get(kind, scalar_types.uint4b8),
        act_type={"w4a8_int8": torch.int8, "w4a8_fp8": torch.float8_e4m3fn}.get(kind, DTYPES[case["dtype"]]),
        group_size=case["group"], zero_points=kind == "awq", has_g_idx=kind == "act_order"))


def _load_linear(case, raw):
    layer = SimpleNamespace(**raw)
    if case["format"] == "awq":
        marlin_linear.convert_awq_to_standard_format(layer)
    kernel = _linear_kernel(case)
    kernel.process_weights_after_loading(layer)
    return kernel, layer


def _linear_call(case, gen):
    """A loaded projection: the function of the activations that its user calls."""
    k, n, kind, dtype = case["k"], case["n"], case["format"], DTYPES[case["dtype"]]
    bias = (torch.randn(n, device="cuda", generator=gen) * 0.1).to(dtype) if case["bias"] else None
    if kind in ("fp8", "mxfp8", "mxfp4", "nvfp4"):
        layer = SimpleNamespace(output_size_per_partition=n, input_size_per_partition=k, params_dtype=dtype,
                                orig_dtype=dtype, bias=bias)
        if kind in ("fp8", "mxfp8"):
            layer.weight = (torch.randn((n, k), device="cuda", generator=gen) * 64).to(torch.float8_e4m3fn)
        else:
            layer.weight = _fp4_bytes(gen, n, k)
        if kind == "fp8":
            layer.weight_scale = torch.rand(n, device="cuda", generator=gen) * 3e-4 + 1e-4
            marlin_utils_fp8.prepare_fp8_layer_for_marlin(layer, size_k_first=False)
            return lambda x: marlin_utils_fp8.apply_fp8_marlin_linear(x, layer.weight, layer.weight_scale,
                                                                      layer.workspace, n, k, layer.bias)
        if kind == "mxfp8":
            layer.weight_scale = _exponents(gen, (n, k // 32)) - 6
            marlin_utils_fp8.prepare_mxfp8_layer_for_marlin(layer)
            return lambda x: marlin_utils_fp8.apply_mxfp8_marlin_linear(x, layer.weight, layer.weight_scale,
                                                                        layer.workspace, n, k, layer.bias)
        if kind == "nvfp4":
            layer.weight_scale = (torch.rand((n, k // 16), device="cuda", generator=gen) * 440 + 8).to(torch.float8_e4m3fn)
            layer.weight_global_scale = torch.full((1,), 3e-5, device="cuda")
        else:
            layer.weight_scale = _exponents(gen, (n, k // 32))
        marlin_utils_fp4.prepare_fp4_layer_for_marlin(layer)
        scale2 = layer.weight_global_scale if kind == "nvfp4" else None
        return lambda x: marlin_utils_fp4.apply_fp4_marlin_linear(x, layer.weight, layer.weight_scale, scale2,
                                                                  layer.workspace, n, k, layer.bias)
    raw = _checkpoint_linear(case, gen)
    kernel, layer = _load_linear(case, dict(raw, bias=bias))
    return lambda x: kernel.apply_weights(layer, x, layer.bias)


def _activations(gen, m, k, dtype):
    return torch.randn((m, k), device="cuda", generator=gen).to(dtype)


def _checkpoint_experts(case, gen):
    """One layer's experts as a checkpoint holds them (MXFP4: (E, N, K / 2) bytes and exponent bytes)."""
    e, hidden, inter, group = case["experts"], case["hidden"], case["inter"], case["group"]
    dtype, raw = DTYPES[case["dtype"]], {}
    for name, k, n in (("w13", hidden, 2 * inter), ("w2", inter, hidden)):
        if case["format"] == "mxfp4":
            raw[name + "_qweight"] = torch.stack([_fp4_bytes(gen, n, k) for _ in range(e)])
            raw[name + "_scales"] = _exponents(gen, (e, n, k // 32))
            continue
        pack = (lambda q: _pack_cols(q, _AWQ_ORDER)) if case["format"] == "awq" else _pack_rows
        raw[name + "_qweight"] = torch.stack([pack(_codes4(gen, k, n)) for _ in range(e)])
        raw[name + "_scales"] = _scales(gen, (e, k // group, n), dtype)
        if case["format"] == "awq":
            raw[name + "_qzeros"] = torch.stack([_pack_cols(_zero_codes(gen, k // group, n), _AWQ_ORDER) for _ in range(e)])
    return raw


def _load_experts(case, raw):
    if case["format"] == "awq":
        return moe_weights.process_awq_moe_weights(case["inter"], 4, case["group"], **raw)
    return moe_weights.process_gptq_moe_weights(case["inter"], 4, case["group"], False, **raw)


def _moe_call(case, gen):
    e, hidden, inter, dtype = case["experts"], case["hidden"], case["inter"], DTYPES[case["dtype"]]
    bias1 = bias2 = zeros1 = zeros2 = None
    if case["bias"]:
        bias1 = torch.randn((e, 2 * inter), device="cuda", generator=gen).to(dtype) * 0.1
        bias2 = torch.randn((e, hidden), device="cuda", generator=gen).to(dtype) * 0.1
    raw = _checkpoint_experts(case, gen)
    if case["format"] == "mxfp4":
        w1, w2, s1, s2, bias1, bias2 = marlin_utils_fp4.prepare_moe_mxfp4_layer_for_marlin(
            SimpleNamespace(params_dtype=dtype), raw["w13_qweight"], raw["w2_qweight"], raw["w13_scales"],
            raw["w2_scales"], bias1, bias2)
        wtype = scalar_types.float4_e2m1f
    else:
        w = _load_experts(case, raw)
        w1, w2, s1, s2, zeros1, zeros2 = w.w1, w.w2, w.w1_scale, w.w2_scale, w.w1_zeros, w.w2_zeros
        wtype = scalar_types.uint4 if case["format"] == "awq" else scalar_types.uint4b8
    x = _activations(gen, case["tokens"], hidden, dtype)
    logits = torch.randn((case["tokens"], e), device="cuda", generator=gen)
    weights, ids = torch.topk(torch.softmax(logits, dim=1), case["top_k"], dim=1)
    weights, ids = weights.contiguous(), ids.to(torch.int32)
    return lambda: fused_moe.fused_marlin_moe(x, w1, w2, bias1, bias2, s1, s2, weights, ids, wtype.id,
                                              activation=case["activation"], w1_zeros=zeros1, w2_zeros=zeros2)


def _decode_layers(case, gen):
    """The projections of a few decoder layers in one graph; each reads its own activations."""
    m, hidden, inter, dtype = case["m"], case["hidden"], case["inter"], DTYPES[case["dtype"]]
    calls = []
    for _ in range(case["layers"]):
        for k, n in ((hidden, case["qkv"]), (hidden, hidden), (hidden, 2 * inter), (inter, hidden)):
            one = _linear_call(dict(case, format="gptq", k=k, n=n, bias=False), gen)
            calls.append((one, _activations(gen, m, k, dtype)))
    for one, x in calls:   # a graph is recorded after a step that was run once
        one(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = [one(x) for one, x in calls]
    return graph, out, calls


# ---------------------------------------------------------------- the five functions
def prepare(case, seed):
    gen = _generator(seed)
    what = case["what"]
    if what == "linear":
        return case, _linear_call(case, gen), _activations(gen, case["m"], case["k"], DTYPES[case["dtype"]])
    if what == "decode_layers":
        return case, _decode_layers(case, gen), None
    if what == "moe":
        return case, _moe_call(case, gen), None
    return case, (_checkpoint_linear if what == "load_linear" else _checkpoint_experts)(case, gen), None


def run(state):
    case, held, x = state
    what = case["what"]
    if what == "linear":
        return held(x)
    if what == "decode_layers":
        graph, out, _ = held
        graph.replay()
        return out
    if what == "moe":
        return held()
    if what == "load_linear":
        _, layer = _load_linear(case, held)
        return [t for t in (layer.qweight, layer.scales, getattr(layer, "qzeros", None), getattr(layer, "g_idx", None),
                            getattr(layer, "g_idx_sort_indices", None)) if t is not None and t.numel() > 0]
    w = _load_experts(case, held)
    return [t for t in (w.w1, w.w2, w.w1_scale, w.w2_scale, w.w1_zeros, w.w2_zeros) if t is not None]


def _weight_bytes(case, k, n):
    bits, group_bits = FORMATS[case.get("format", "gptq")]
    groups = 1 if case["group"] == -1 else k // case["group"]
    return (k * n * bits + groups * n * group_bits) / 8


def work(case):
    what = case["what"]
    if what == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        order = 8 * k if case["format"] == "act_order" else 0
        return {"bytes": _weight_bytes(case, k, n) + 2 * m * k + 2 * m * n + order, "flops": 2.0 * m * k * n}
    if what == "decode_layers":
        m, hidden, inter = case["m"], case["hidden"], case["inter"]
        shapes = ((hidden, case["qkv"]), (hidden, hidden), (hidden, 2 * inter), (inter, hidden))
        return {"bytes": case["layers"] * sum(_weight_bytes(case, k, n) + 2 * m * (k + n) for k, n in shapes),
                "flops": case["layers"] * sum(2.0 * m * k * n for k, n in shapes)}
    if what == "load_linear":
        return {"bytes": 2 * _weight_bytes(case, case["k"], case["n"]), "flops": 0}
    hidden, inter, experts = case["hidden"], case["inter"], case["experts"]
    each = _weight_bytes(case, hidden, 2 * inter) + _weight_bytes(case, inter, hidden)
    if what == "load_experts":
        return {"bytes": 2 * experts * each, "flops": 0}
    tokens, top_k = case["tokens"], case["top_k"]
    touched = experts * (1 - (1 - top_k / experts) ** tokens)   # experts that a token is routed to, on average
    return {"bytes": touched * each + 2 * 2 * tokens * hidden + 8 * tokens * top_k,
            "flops": 6.0 * tokens * top_k * hidden * inter}


def tolerance(case):
    if case["what"].startswith("load"):
        return "exact"   # packed codes, and scales and zero points in another order
    # sums are in fp32; what differs between correct implementations is where a weight, a partial result or the
    # output is rounded to 16 bits
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3}
