"""What this framework is timed on: the linear layers of a quantised decoder, called as a model calls them.

Five forms of call, each over the sizes it is used at:

  linear   ``W2A8Linear.forward``: one 2-bit layer, from one decode token to a prompt of thousands of tokens (the
           activation quantisation and the GEMM, plus the bias where the layer has one).
  block    the linears of one decoder block for a batch of decode tokens: query / key / value share one quantised
           activation and one grouped launch, gate / up another, the two output projections run alone.
  grouped  many independent few-row GEMMs in one launch on activations that are quantised already: the decode sweep
           of the benchmark, 1..32 rows on each of the Llama-3-8B linear shapes.
  linear4  ``W4A8Linear.forward``: the same layer with 4-bit weights.
  linear16 ``W2A16Linear.forward``: 2-bit weights, activations left in fp16 / bf16.

A case's ``rows`` are token rows (M), ``n`` the layer's outputs, ``k`` its inputs, ``group`` the scale group along k,
``mode`` the weight levels ("sym": one zero-point for all, "asym": one per group), ``dtype`` the type of activations and
outputs.  Weights are normal draws quantised by the framework, activations normal draws in which one channel in a
thousand is twenty times larger, as trained models have them.
"""
import math

import torch

from slimkernels_amd import torch as ops
from slimkernels_amd import workloads

DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16}
HIDDEN, KV, FFN = 4096, 1024, 14336          # the Llama-3-8B linears of the "block" and "grouped" forms
MAX_ROWS = {"linear": 4096, "linear4": 2048, "linear16": 1024}
MAX_WEIGHTS = 28672 * 8192


def _linear(name, rows, n, k, group=128, mode="sym", dtype="float16", bias=False, kind="linear"):
    return {"name": name, "kind": kind, "rows": rows, "n": n, "k": k, "group": group, "mode": mode, "dtype": dtype,
            "bias": bias}


def listed():
    return [
        # one user's next token through the attention output projection: the smallest call, launch latency and host work
        _linear("decode_1_attention_out", 1, 4096, 4096),
        # four users' next tokens through all seven linears of one decoder block
        {"name": "decode_4_block", "kind": "block", "rows": 4, "group": 128, "mode": "sym", "dtype": "float16"},
        # the benchmark's decode sweep: 24 GEMMs of 1..32 rows in one launch
        {"name": "decode_sweep_grouped", "kind": "grouped", "rows": 32, "group": 128, "mode": "sym", "dtype": "float16"},
        # one token through the feed-forward matrix of a 70B-class model, small groups, bf16
        _linear("decode_1_ffn70b", 1, 28672, 8192, group=64, dtype="bfloat16"),
        # a full decode batch, per-group zero-points, a width that no tile divides, a layer with a bias
        _linear("batch_77_asym_bias", 77, 11008, 4096, mode="asym", bias=True),
        # a large decode batch (or a short prompt) through the 70B-class matrix
        _linear("batch_128_ffn70b", 128, 28672, 8192, group=64, dtype="bfloat16"),
        # a prompt of 512 tokens through the long reduction of the down projection
        _linear("prefill_512_down", 512, 4096, 14336),
        # a prompt of 4096 tokens through gate / up: the throughput of the matrix cores
        _linear("prefill_4096_gate", 4096, 14336, 4096),
        # 2048 tokens through the 70B-class matrix in groups of 64: the largest call
        _linear("prefill_2048_ffn70b", 2048, 28672, 8192, group=64, dtype="bfloat16"),
        # a 4-bit layer on a prompt of an odd length
        _linear("w4_prefill_1000_gate", 1000, 14336, 4096, kind="linear4"),
        # the weight-only layer: one decode token in bf16, and a prompt that no tile divides
        _linear("weight_only_decode_1", 1, 14336, 4096, dtype="bfloat16", kind="linear16"),
        _linear("weight_only_prompt_300", 300, 4096, 14336, kind="linear16"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["block", "grouped", "linear4", "linear4", "linear16", "linear16"])
    group = rng.choice([64, 128, 128, 128, 256])
    dtype = rng.choice(list(DTYPES))
    if kind in ("block", "grouped"):
        return {"kind": kind, "rows": _log_int(rng, 1, 32), "group": group, "mode": rng.choice(["sym", "sym", "asym"]),
                "dtype": dtype}
    if kind == "linear4" and group == 256:
        group = 128
    k = _log_int(rng, 1024, 28672) // 256 * 256
    if kind == "linear" and group == 64:
        k += 64 * rng.randrange(4)                     # an odd number of 64-element steps now and then
    n = _log_int(rng, 1000, min(28672, MAX_WEIGHTS // k))
    if rng.random() < 0.7:
        n = n // 8 * 8                                 # mostly whole 16-byte rows, sometimes any width
    # a fifth of the calls are one decode token, the others spread over every row count
    rows = 1 if rng.random() < 0.2 else _log_int(rng, 2, MAX_ROWS[kind])
    rows = max(1, min(rows, 2048 * MAX_WEIGHTS // (n * k) // (1 if kind == "linear" else 8)))
    return {"kind": kind, "rows": rows, "n": n, "k": k, "group": group, "mode": rng.choice(["sym", "sym", "asym"]),
            "dtype": dtype, "bias": rng.random() < 0.25}


def _activation(rows, k, dtype, gen):
    x = torch.randn((rows, k), generator=gen, device="cuda")
    hot = torch.randperm(k, generator=gen, device="cuda")[: max(1, k // 1000)]
    x[:, hot] *= 20.0
    return x.to(DTYPES[dtype])


def _layer(cls, case, n, k, gen):
    dtype = DTYPES[case["dtype"]]
    weight = torch.randn((n, k), generator=gen, device="cuda", dtype=torch.float16) * 0.02
    bias = torch.randn((n,), generator=gen, device="cuda").to(dtype) if case.get("bias") else None
    return cls.from_float(weight, case["group"], case["mode"], bias=bias, out_dtype=dtype)


def _grouped_shapes(case):
    """(rows, n, k) of the grouped form: every row count of the sweep up to the case's, on each linear shape."""
    rows = [m for m in workloads.DECODE_M if m < case["rows"]] + [case["rows"]]
    return [(m, n, k) for (n, k) in workloads.LLAMA8B_LINEARS.values() for m in rows]


BLOCK_LAYERS = {"q": (HIDDEN, HIDDEN), "k": (KV, HIDDEN), "v": (KV, HIDDEN), "o": (HIDDEN, HIDDEN),
                "gate": (FFN, HIDDEN), "up": (FFN, HIDDEN), "down": (HIDDEN, FFN)}


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind = case["kind"]
    state = {"case": case}
    if kind == "block":
        state["w"] = {name: _layer(ops.W2A8Linear, case, n, k, gen).weight for name, (n, k) in BLOCK_LAYERS.items()}
        # what the norms, the attention and the gating of the block hand to its linears
        for name in ("x_attn", "x_out", "x_ffn"):
            state[name] = _activation(case["rows"], HIDDEN, case["dtype"], gen)
        state["x_down"] = _activation(case["rows"], FFN, case["dtype"], gen)
    elif kind == "grouped":
        problems = []
        for rows, n, k in _grouped_shapes(case):
            w = _layer(ops.W2A8Linear, case, n, k, gen).weight
            qa = ops.quantize_act_int8(_activation(rows, k, case["dtype"], gen), case["group"])
            problems.append((qa, w, torch.empty((rows, n), dtype=DTYPES[case["dtype"]], device="cuda")))
        state["problems"] = problems
    else:
        cls = {"linear": ops.W2A8Linear, "linear4": ops.W4A8Linear, "linear16": ops.W2A16Linear}[kind]
        state["layer"] = _layer(cls, case, case["n"], case["k"], gen)
        state["x"] = _activation(case["rows"], case["k"], case["dtype"], gen)
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "block":
        w, group, dtype = state["w"], case["group"], DTYPES[case["dtype"]]
        qa = ops.quantize_act_int8(state["x_attn"], group)
        q, k, v = ops.w2a8_gemm_grouped([(qa, w["q"]), (qa, w["k"]), (qa, w["v"])], dtype)
        o = ops.w2a8_gemm(ops.quantize_act_int8(state["x_out"], group), w["o"], dtype)
        qa = ops.quantize_act_int8(state["x_ffn"], group)
        gate, up = ops.w2a8_gemm_grouped([(qa, w["gate"]), (qa, w["up"])], dtype)
        down = ops.w2a8_gemm(ops.quantize_act_int8(state["x_down"], group), w["down"], dtype)
        return {"q": q, "k": k, "v": v, "o": o, "gate": gate, "up": up, "down": down}
    if case["kind"] == "grouped":
        return ops.w2a8_gemm_grouped(state["problems"], DTYPES[case["dtype"]])
    with torch.no_grad():
        return state["layer"](state["x"])


def work(case):
    kind, group = case["kind"], case["group"]
    if kind == "block":
        gemms = [(case["rows"], n, k) for n, k in BLOCK_LAYERS.values()]
    elif kind == "grouped":
        gemms = _grouped_shapes(case)
    else:
        gemms = [(case["rows"], case["n"], case["k"])]
    weight_bits = 4 if kind == "linear4" else 2
    bytes_, flops = 0, 0
    for rows, n, k in gemms:
        bytes_ += n * k * weight_bits // 8 + 2 * n * (k // group) + 2 * rows * n
        if case["mode"] == "asym":
            bytes_ += n * (k // group) * weight_bits // 8
        if kind == "grouped":
            bytes_ += rows * k + 4 * rows             # int8 activations and their token scales
        elif kind != "block":
            bytes_ += 2 * rows * k
        flops += 2 * rows * n * k
    if kind == "block":
        bytes_ += 2 * case["rows"] * (3 * HIDDEN + FFN)   # the four activations of the block, each read once
    if case.get("bias"):
        bytes_ += 2 * case["n"]
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    # The integer sums are exact, the scaled sums are 32-bit: what is left is the rounding of the outputs (half an ULP:
    # measured against a float64 evaluation of the same integers and scales: 2.1e-4 for fp16, 2.9e-4 with a bias, which
    # rounds once more, 1.7e-3 for bf16).
    return {"rel": 8e-4} if case["dtype"] == "float16" else {"rel": 7e-3}


def _levels(case, n, k, gen):
    """The layer of ``_layer`` in float64: its dequantised weight [n, k] and its bias, by the definition of the
    quantiser (float32 levels, ties to even, scales stored in fp16), in plain torch."""
    weight = torch.randn((n, k), generator=gen, device="cuda", dtype=torch.float16) * 0.02
    bias = torch.randn((n,), generator=gen, device="cuda").to(DTYPES[case["dtype"]]) if case.get("bias") else None
    top = 15 if case["kind"] == "linear4" else 3
    w = weight.float().reshape(n, k // case["group"], case["group"])
    if case["mode"] == "sym":
        zero = torch.full_like(w[:, :, :1], (top + 1) // 2)      # also the divisor of the scale
        scale = w.abs().amax(2, keepdim=True).clamp_min(1e-9) / zero[0, 0]
    else:
        low = w.amin(2, keepdim=True)
        scale = (w.amax(2, keepdim=True) - low).clamp_min(1e-9) / torch.full_like(low, top)
        zero = torch.round(-low / scale).clamp_(0, top)
    codes = torch.round(w / scale).add_(zero).clamp_(0, top)
    return (codes.sub_(zero).double() * scale.half().double()).reshape(n, k), bias


def _quantised(x):
    """The activation as the int8 path sees it, in float64: per-token scale, ties to even.  (Tensor divisors here and
    above: torch turns a division by a Python number into a product with its rounded reciprocal.)"""
    x = x.float()
    amax = x.abs().amax(1, keepdim=True).clamp_min(1e-9)
    scale = amax / torch.full_like(amax, 127.0)
    return torch.round(x / scale).clamp_(-127, 127).double() * scale.double()


def exact(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind, rows, dtype = case["kind"], case["rows"], case["dtype"]
    if kind == "block":
        w = {name: _levels(case, n, k, gen)[0] for name, (n, k) in BLOCK_LAYERS.items()}
        x_attn, x_out, x_ffn = (_quantised(_activation(rows, HIDDEN, dtype, gen)) for _ in range(3))
        x_down = _quantised(_activation(rows, FFN, dtype, gen))
        inputs = {"q": x_attn, "k": x_attn, "v": x_attn, "o": x_out, "gate": x_ffn, "up": x_ffn, "down": x_down}
        return {name: x @ w[name].t() for name, x in inputs.items()}
    if kind == "grouped":
        outs = []
        for m, n, k in _grouped_shapes(case):
            w, _ = _levels(case, n, k, gen)
            outs.append(_quantised(_activation(m, k, dtype, gen)) @ w.t())
        return outs
    w, bias = _levels(case, case["n"], case["k"], gen)
    x = _activation(rows, case["k"], dtype, gen)
    y = (x.double() if kind == "linear16" else _quantised(x)) @ w.t()
    return y if bias is None else y + bias.double()
