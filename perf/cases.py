"""The work this library is used for, as cases that can be timed and compared.

A case is a dict of plain values.  `kind` names what a program does with the library:

    linear     one eager forward of a frozen linear (a projection called on its own)
    layer      forward and input gradient of one frozen linear, eager, fp32 compute (the layer's default cell)
    decode     the gated feed-forward blocks of a few transformer layers for the rows of one decode step, captured once
               into a HIP graph and replayed per step, as a serving loop keeps it
    moe_decode one frozen-expert layer for the tokens of one decode step: routing, expert projections, combination; eager
    train      a fine-tune step through a frozen base: forward with the adapter's branch added in the store and input
               gradient with the adapter's gradient added, eager
    moe_train  one frozen-expert layer over a training batch: routing, forward, backward down to the tokens and the router
    quantise   a dense fp32 weight turned into packed int4 and into per-channel int8 storage (loading a checkpoint)

Weights are quantised by the library from N(0, 0.02), activations are N(0, 1), gradients N(0, 1e-3), expert ids uniform.
`storage`: int4 (groups of 128), int8 (per-channel scales), int8_tensor (one scale), bf16 (stored undequantised)."""
import math

import torch

from caif_amd import torch_ops as T

DTYPES = {"f32": T.F32, "f16": T.F16, "bf16": T.BF16}
GROUP = 128


def listed():
    return [
        # the smallest call: one token through one small projection (an expert's size), where launch and host path count
        {"name": "linear-int8-1", "kind": "linear", "storage": "int8", "compute": "bf16", "m": 1, "n": 1408, "k": 2048},
        # 100 rows (a short prompt, or a large decode batch) through a square int4 projection: few tiles for the chip
        {"name": "linear-int4-100", "kind": "linear", "storage": "int4", "compute": "bf16", "m": 100, "n": 4096, "k": 4096},
        # prefill of a 2048-token prompt, the up projection of a 7B feed-forward block
        {"name": "linear-int4-2048", "kind": "linear", "storage": "int4", "compute": "bf16", "m": 2048, "n": 11008, "k": 4096},
        # a ragged prompt in fp16 through int8 codes, the up projection of an 8B feed-forward block
        {"name": "linear-int8-999", "kind": "linear", "storage": "int8", "compute": "f16", "m": 999, "n": 14336, "k": 4096},
        # the default cell of the layer: fp32 compute, 16 rows, forward and input gradient
        {"name": "layer-int8-16", "kind": "layer", "storage": "int8", "compute": "f32", "m": 16, "n": 4096, "k": 4096},
        # single-token decode through int4 and batched decode through int8 and int4 feed-forward blocks
        {"name": "decode-int4-1", "kind": "decode", "storage": "int4", "compute": "bf16", "m": 1, "n": 14336, "k": 4096},
        {"name": "decode-int8-1", "kind": "decode", "storage": "int8", "compute": "bf16", "m": 1, "n": 14336, "k": 4096},
        {"name": "decode-int4-16", "kind": "decode", "storage": "int4", "compute": "bf16", "m": 16, "n": 14336, "k": 4096},
        # a decode step of 16 tokens through 64 small experts, six per token
        {"name": "moe-decode-16", "kind": "moe_decode", "storage": "int8", "compute": "bf16", "m": 16, "n": 1408, "k": 2048,
         "experts": 64, "top_k": 6},
        # adapter fine-tuning over an int4 base, 4096 tokens
        {"name": "train-int4-4096", "kind": "train", "storage": "int4", "compute": "bf16", "m": 4096, "n": 11008, "k": 4096},
        # fine-tuning through frozen int8 experts, 4096 tokens, six of 64 experts per token
        {"name": "moe-train-4096", "kind": "moe_train", "storage": "int8", "compute": "bf16", "m": 4096, "n": 1408, "k": 2048,
         "experts": 64, "top_k": 6},
        # loading one dense weight into both storage forms
        {"name": "quantise-4096", "kind": "quantise", "storage": "both", "compute": "f32", "m": 1, "n": 14336, "k": 4096},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _multiple(rng, lo, hi, step):
    return max(lo, min(hi, _log_int(rng, lo, hi) // step * step))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "layer", "decode", "decode", "moe_decode", "train", "moe_train", "quantise"])
    if kind == "linear":
        storage = rng.choice(["int4", "int4", "int8", "int8", "int8_tensor", "bf16"])
        compute = "bf16" if storage == "bf16" else rng.choice(["bf16", "f16"])
        return {"kind": kind, "storage": storage, "compute": compute, "m": _log_int(rng, 1, 4096),
                "n": _multiple(rng, 512, 14336, 64), "k": _multiple(rng, 512, 4096, 128)}
    if kind == "layer":
        return {"kind": kind, "storage": rng.choice(["int4", "int8"]), "compute": "f32", "m": _log_int(rng, 1, 256),
                "n": _multiple(rng, 512, 8192, 64), "k": _multiple(rng, 512, 4096, 128)}
    if kind == "decode":
        return {"kind": kind, "storage": rng.choice(["int4", "int8"]), "compute": rng.choice(["bf16", "bf16", "f16"]),
                "m": _log_int(rng, 1, 32), "n": _multiple(rng, 2048, 14336, 256), "k": _multiple(rng, 1024, 4096, 256)}
    if kind == "train":
        storage = rng.choice(["int4", "int8", "bf16"])
        return {"kind": kind, "storage": storage, "compute": "bf16", "m": _log_int(rng, 128, 4096),
                "n": _multiple(rng, 1024, 11008, 64), "k": _multiple(rng, 1024, 4096, 128)}
    if kind == "quantise":
        return {"kind": kind, "storage": "both", "compute": "f32", "m": 1, "n": _multiple(rng, 512, 14336, 64),
                "k": _multiple(rng, 512, 4096, 128)}
    # expert layers: the packed buffer holds m * top_k rows
    most = 64 if kind == "moe_decode" else 4096
    return {"kind": kind, "storage": rng.choice(["int8", "int8", "int4"]), "compute": "bf16",
            "m": _log_int(rng, 1 if kind == "moe_decode" else 256, most), "n": _multiple(rng, 512, 1408, 128),
            "k": _multiple(rng, 512, 2048, 256), "experts": rng.choice([8, 16, 33, 64]), "top_k": rng.choice([2, 4, 6])}


# ------------------------------------------------------------------------------------------------ what a program holds
def _normal(gen, shape, std, dtype=torch.float32):
    return torch.empty(shape, device="cuda").normal_(0, std, generator=gen).to(dtype)


def _weight(gen, storage, n, k):
    if storage == "int4":
        packed, scales = T.quantize_int4_per_group(_normal(gen, (n, k), 0.02), GROUP)
        return T.FrozenWeight(packed, T.W_INT4_GROUP, scales, n, k, 1, GROUP)
    if storage == "bf16":
        return T.FrozenWeight(_normal(gen, (n, k), 0.02, torch.bfloat16).reshape(-1), T.W_BF16, None, n, k)
    codes, scales = T.quantize_int8(_normal(gen, (k, n), 0.02), per_channel=storage == "int8")
    return T.FrozenWeight(codes.reshape(-1), T.W_INT8, scales, n, k, n if storage == "int8" else 1)


def _bank(gen, storage, experts, n, k):
    return T.GroupedFrozenWeights([_weight(gen, storage, n, k) for _ in range(experts)])


def _ffn(x, layers, compute):
    for gate, up, down in layers:
        g = T.qlinear_forward(x, gate, compute, compute)
        u = T.qlinear_forward(x, up, compute, compute)
        x = T.qlinear_forward(T.silu_multiply(g, u), down, compute, compute)
    return x


DECODE_LAYERS = 2


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, storage, m, n, k = case["kind"], case["storage"], case["m"], case["n"], case["k"]
    compute = DTYPES[case["compute"]]
    dtype = T.TORCH_DTYPE[compute]
    s = {"kind": kind, "compute": compute}
    if kind == "quantise":
        s["w_int4"], s["w_int8"] = _normal(gen, (n, k), 0.02), _normal(gen, (k, n), 0.02)
        return s
    s["x"] = _normal(gen, (m, k), 1, dtype)
    if kind in ("linear", "layer", "train"):
        s["w"] = _weight(gen, storage, n, k)
        s["dy"] = _normal(gen, (m, n), 1e-3, dtype)
        if kind == "train":        # what the adapter's own small products contribute
            s["branch"], s["branch_grad"] = _normal(gen, (m, n), 1e-2, dtype), _normal(gen, (m, k), 1e-4, dtype)
        return s
    if kind == "decode":
        layers = [(_weight(gen, storage, n, k), _weight(gen, storage, n, k), _weight(gen, storage, k, n))
                  for _ in range(DECODE_LAYERS)]
        s["layers"] = layers       # the weights that the captured graph reads
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            _ffn(s["x"], layers, compute)
        torch.cuda.current_stream().wait_stream(stream)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["y"] = _ffn(s["x"], layers, compute)
        return s
    experts, top_k = case["experts"], case["top_k"]
    s["gate"], s["up"] = _bank(gen, storage, experts, n, k), _bank(gen, storage, experts, n, k)
    s["down"] = _bank(gen, storage, experts, k, n)
    s["experts"] = experts
    s["ids"] = torch.randint(0, experts, (m, top_k), device="cuda", generator=gen, dtype=torch.int32)
    s["weights"] = torch.softmax(_normal(gen, (m, top_k), 1), dim=1).to(dtype)
    s["dy"] = _normal(gen, (m, k), 1e-3, dtype)
    return s


# ------------------------------------------------------------------------------------------------ one pass
def _moe_forward(s):
    c, x, ids = s["compute"], s["x"], s["ids"]
    dmap, offsets = T.moe_build_dispatch_map(ids, s["experts"])
    rows = ids.numel()
    packed = T.moe_dispatch(x, ids, dmap, offsets, rows)
    up = T.qlinear_grouped_forward(packed, offsets, s["up"], c, c)
    gate = T.qlinear_grouped_forward(packed, offsets, s["gate"], c, c)
    out = T.qlinear_grouped_forward(T.silu_multiply(gate, up), offsets, s["down"], c, c)
    y = T.moe_combine(out, ids, s["weights"], dmap, offsets)
    return y, dmap, offsets, up, gate, out


def run(s):
    kind, c = s["kind"], s["compute"]
    if kind == "linear":
        return T.qlinear_forward(s["x"], s["w"], c, c)
    if kind == "layer":
        return T.qlinear_forward(s["x"], s["w"], c), T.qlinear_backward_input(s["dy"], s["w"], c)
    if kind == "train":
        return (T.qlinear_forward(s["x"], s["w"], c, c, addend=s["branch"]),
                T.qlinear_backward_input(s["dy"], s["w"], c, c, addend=s["branch_grad"]))
    if kind == "decode":
        s["graph"].replay()
        return s["y"]
    if kind == "quantise":
        return T.quantize_int4_per_group(s["w_int4"], GROUP) + T.quantize_int8(s["w_int8"], per_channel=True)
    if kind == "moe_decode":
        y, dmap, offsets = _moe_forward(s)[:3]
        return y, dmap, offsets
    y, dmap, offsets, up, gate, out = _moe_forward(s)
    ids, rows = s["ids"], s["ids"].numel()
    grad_weights = T.moe_combine_backward_grad_weights(s["dy"], out, ids, dmap, offsets)
    grad_out = T.moe_combine_backward_grad_expert(s["dy"], ids, s["weights"], dmap, offsets, rows)
    grad_hidden = T.qlinear_grouped_backward_input(grad_out, offsets, s["down"], c, c)
    grad_gate, grad_up = T.swiglu_backward(gate, up, grad_hidden)
    grad_in = T.qlinear_grouped_backward_input(grad_up, offsets, s["up"], c, c)
    grad_in = T.qlinear_grouped_backward_input(grad_gate, offsets, s["gate"], c, c, addend=grad_in)
    grad_x = T.moe_dispatch_backward(grad_in, ids, dmap, offsets)
    return y, dmap, offsets, grad_x, grad_weights


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _weight_bytes(storage, n, k):
    if storage == "int4":
        return n * k / 2 + n * k / GROUP * 2
    if storage == "bf16":
        return n * k * 2
    return n * k + (n * 4 if storage == "int8" else 4)


def work(case):
    kind, storage, m, n, k = case["kind"], case["storage"], case["m"], case["n"], case["k"]
    e = 4 if case["compute"] == "f32" else 2
    w = _weight_bytes(storage, n, k)
    gemm = 2.0 * m * n * k
    if kind == "linear":
        return {"bytes": w + m * (n + k) * e, "flops": gemm}
    if kind == "layer":
        return {"bytes": 2 * (w + m * (n + k) * e), "flops": 2 * gemm}
    if kind == "train":
        return {"bytes": 2 * w + 3 * m * (n + k) * e, "flops": 2 * gemm}
    if kind == "decode":       # the activations between the projections of a block need not leave the chip
        return {"bytes": DECODE_LAYERS * 3 * w + 2 * m * k * e, "flops": DECODE_LAYERS * 3 * gemm}
    if kind == "quantise":
        return {"bytes": 8 * n * k + _weight_bytes("int4", n, k) + _weight_bytes("int8", n, k), "flops": 2.0 * n * k}
    experts, rows = case["experts"], m * case["top_k"]
    touched = experts * (1 - (1 - 1 / experts) ** rows)      # uniform ids
    tokens, ids = m * k * e, rows * 4
    if kind == "moe_decode":
        return {"bytes": 3 * touched * w + 2 * tokens + 2 * ids + rows * e, "flops": 3 * 2.0 * rows * n * k}
    # what the backward reads of the forward (gate, up, expert results) is written and read once more
    kept = 2 * rows * (2 * n + k) * e
    return {"bytes": 6 * touched * w + 4 * tokens + 2 * ids + 3 * rows * e + kept, "flops": 6 * 2.0 * rows * n * k}


# Measured against the same path in 64 bits on the quantised weights (2-norm of the difference over that of the result, and
# the largest difference over the rms or the value), times about four.  bf16: one projection 2.4e-3 / 1.1e-2 (the results'
# own rounding 1.7e-3, the weight's the rest), with an addend 2.9e-3 / 1.4e-2, an expert layer 4.3e-3 / 2.0e-2 forward and
# 5.6e-3 / 3.4e-2 with its gradients, six projections in a row 7.8e-3 / 3.4e-2.  f16 carries three bits more: an eighth.
# fp32 compute: 5.6e-7 / 2.5e-6 with int8 digits or pieces of bf16, sums of up to 8192 products in fp32.
BF16_TOLERANCE = {"linear": (1e-2, 0.045), "train": (1.2e-2, 0.055), "decode": (0.03, 0.14), "moe_decode": (1.7e-2, 0.08),
                  "moe_train": (2.2e-2, 0.14)}


def tolerance(case):
    if case["kind"] == "quantise":
        return "exact"
    if case["compute"] == "f32":
        return {"rel": 4e-6, "max": 2e-5}
    rel, most = BF16_TOLERANCE[case["kind"]]
    part = 8 if case["compute"] == "f16" else 1
    return {"rel": rel / part, "max": most / part}
