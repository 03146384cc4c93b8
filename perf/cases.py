"""The calls that decide what a program built on ``mojo_amd`` feels: one dict per case, through the package's public entry points.

A case names an entry point (``op``), the weight encoding, the lhs rows ``m`` (tokens in flight), the matrix (``n`` x ``k``; ``hidden`` /
``ffn`` / ``kv`` where a whole transformer layer is meant) and the lhs type.  Weights are N(0, 0.02) and activations N(0, 1), packed by the
package's own quantisers, as in the benchmark and the tests.
"""
import math

import torch

from mojo_amd import (QuantizationConfig, QuantizationEncoding as QE, dequantize, qmatmul, qmatmul_grouped, qmatmul_repacked,
                      qmatmul_rmsnorm, qmatmul_swiglu, quantize, quantize_gptq, repack_weights)

ENCODINGS = ("Q4_K", "Q4_0", "Q5_K", "Q6_K", "GPTQ")
LHS = {"f32": torch.float32, "bf16": torch.bfloat16}
EPS = 1e-5
# (N, K): the projections and vocabularies that the benchmark, its sweeps and the tests use
SHAPES = ((1024, 4096), (4096, 4096), (6144, 4096), (14336, 4096), (4096, 14336), (11008, 4096), (4096, 11008), (5120, 5120),
          (8192, 8192), (32000, 4096), (3584, 18944), (28672, 8192), (8192, 28672))
LAYERS = ((4096, 14336, 1024), (4096, 11008, 4096), (5120, 13824, 5120), (2048, 5632, 256))  # hidden, ffn, k / v rows
MOST = 2048 * 14336 * 4096  # multiply-adds of the largest listed product


def listed():
    return [
        # the smallest call of a decode step: one token through a k or v projection; latency
        {"name": "kv_q4k_1", "op": "matmul", "enc": "Q4_K", "m": 1, "n": 1024, "k": 4096, "lhs": "f32"},
        # one token through the seven projections of a layer, called one by one (the benchmark's step)
        {"name": "layer_q4k_1", "op": "layer", "enc": "Q4_K", "m": 1, "hidden": 4096, "ffn": 14336, "kv": 1024, "lhs": "f32"},
        # the last product of every token: the vocabulary, which mixed checkpoints store in six bits
        {"name": "vocabulary_q6k_1", "op": "matmul", "enc": "Q6_K", "m": 1, "n": 128256, "k": 4096, "lhs": "f32"},
        # one token through the largest projection of a GPTQ checkpoint, bf16 activations
        {"name": "up_gptq_1", "op": "matmul", "enc": "GPTQ", "m": 1, "n": 14336, "k": 4096, "lhs": "bf16", "group": 128},
        # four sequences decoded together, through the entry points that fuse q | k | v and the gated MLP
        {"name": "block_q4k_4", "op": "block", "enc": "Q4_K", "m": 4, "hidden": 4096, "ffn": 14336, "kv": 1024, "lhs": "bf16"},
        # sixteen sequences decoded together
        {"name": "up_q40_16", "op": "matmul", "enc": "Q4_0", "m": 16, "n": 14336, "k": 4096, "lhs": "f32"},
        # a short prompt, or a batch that is no multiple of anything, on a matrix of another model
        {"name": "up_q5k_33", "op": "matmul", "enc": "Q5_K", "m": 33, "n": 11008, "k": 4096, "lhs": "bf16"},
        # a chunk of a prompt (chunked prefill) through a whole layer
        {"name": "layer_q4k_200", "op": "layer", "enc": "Q4_K", "m": 200, "hidden": 4096, "ffn": 14336, "kv": 1024, "lhs": "bf16"},
        # a prompt on an act-order GPTQ checkpoint
        {"name": "up_gptq_order_400", "op": "matmul", "enc": "GPTQ", "m": 400, "n": 14336, "k": 4096, "lhs": "bf16", "group": 128, "order": True},
        # a prompt through the down projection, which mixed checkpoints store in six bits
        {"name": "down_q6k_500", "op": "matmul", "enc": "Q6_K", "m": 500, "n": 4096, "k": 14336, "lhs": "bf16"},
        # a long prompt: compute-bound
        {"name": "prefill_q4k_2048", "op": "matmul", "enc": "Q4_K", "m": 2048, "n": 14336, "k": 4096, "lhs": "bf16"},
        # a matrix unpacked for a consumer that takes plain bf16
        {"name": "dequantize_q4k", "op": "dequantize", "enc": "Q4_K", "n": 14336, "k": 4096, "out": "bf16"},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    op = rng.choices(("matmul", "layer", "block", "rmsnorm", "repacked", "dequantize", "quantize"), (62, 10, 8, 5, 5, 5, 5))[0]
    enc = rng.choice(ENCODINGS if op != "block" else ENCODINGS[:4])
    c = {"op": op, "enc": enc}
    if op in ("layer", "block"):
        c["hidden"], c["ffn"], c["kv"] = rng.choice(LAYERS)
        size = sum(n * k for n, k in _projections(c))
        c["m"] = _log(rng, 1, min(512, MOST // size // (2 if enc == "Q6_K" else 1)))
    else:
        if rng.random() < 0.5:
            c["n"], c["k"] = rng.choice(SHAPES)
        else:  # any matrix: rows in eights, K in blocks of the encoding
            step = {"Q4_0": 32, "GPTQ": 128}.get(enc, 256) if op != "repacked" else 256
            c["n"], c["k"] = 8 * _log(rng, 64, 4096), step * max(1, _log(rng, 512, 14336) // step)
        if op not in ("dequantize", "quantize"):
            most = max(1, min(2048, MOST // (c["n"] * c["k"]) // (2 if enc == "Q6_K" else 1)))
            c["m"] = _log(rng, 1, most)
        elif c["n"] * c["k"] > 14336 * 4096:
            c["n"], c["k"] = 14336, 4096
    if op == "dequantize":
        c["out"] = rng.choice(("f32", "bf16"))
    elif op != "quantize":
        c["lhs"] = rng.choice(("f32", "bf16"))
    if op in ("matmul", "rmsnorm") and rng.random() < 0.2:
        c["out"] = "bf16"
    if enc == "GPTQ":
        c["group"] = rng.choice((128, 128, 128, 32)) if op != "repacked" else 128
        if op == "matmul" and rng.random() < 0.3 and c["n"] * c["k"] <= 14336 * 4096:
            c["order"], c["m"] = True, min(c["m"], _log(rng, 1, 400))
    return c


def _projections(case):
    h, f, kv = case["hidden"], case["ffn"], case["kv"]
    return ((h, h), (kv, h), (kv, h), (h, h), (f, h), (f, h), (h, f))  # q, k, v, o, gate, up, down


def _normal(gen, rows, cols, scale=1.0, dtype=torch.float32):
    return torch.empty((rows, cols), device="cuda").normal_(0.0, scale, generator=gen).to(dtype)


def _weights(case, gen, n, k):
    """(config, rhs tensors) of one matrix, as a loaded checkpoint has them."""
    w = _normal(gen, n, k, 0.02)
    if case["enc"] != "GPTQ":
        return None, (quantize(QE[case["enc"]], w),)
    group, order = case["group"], case.get("order", False)
    qweight, scales, qzeros, g_idx = quantize_gptq(w, QuantizationConfig("gptq", 4, group, False, True))
    if not order:
        return QuantizationConfig("gptq", 4, group, False, True), (qweight, scales, qzeros)
    g_idx = g_idx[torch.randperm(k, device="cuda", generator=gen)].contiguous()  # act-order: every group has its columns anywhere in K
    return QuantizationConfig("gptq", 4, group, True, True), (qweight, scales, qzeros, g_idx)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = {"case": case}
    if case["op"] == "quantize":
        state["x"] = _normal(gen, case["n"], case["k"], 0.02)
        return state
    if case["op"] in ("layer", "block"):
        state["weights"] = [_weights(case, gen, n, k) for n, k in _projections(case)]
        dtype = LHS[case["lhs"]]
        # what enters the attention projections, o, the MLP and (called one by one) down
        state["lhs"] = [_normal(gen, case["m"], k, 1.0, dtype) for k in (case["hidden"], case["hidden"], case["hidden"], case["ffn"])]
        return state
    state["config"], state["rhs"] = _weights(case, gen, case["n"], case["k"])
    if case["op"] == "repacked":
        state["packed"] = repack_weights(QE[case["enc"]], state["config"], *state["rhs"])
    if case["op"] != "dequantize":
        state["lhs"] = _normal(gen, case["m"], case["k"], 1.0, LHS[case["lhs"]])
    if case["op"] == "rmsnorm":
        state["gamma"] = 1.0 + 0.1 * _normal(gen, 1, case["k"])[0]
    return state


def run(state):
    case = state["case"]
    op, enc = case["op"], QE[case["enc"]]
    if op == "matmul":
        return qmatmul(enc, state["config"], state["lhs"], *state["rhs"], out_dtype=LHS[case.get("out", "f32")])
    if op == "layer":
        return [qmatmul(enc, config, state["lhs"][i], *rhs) for i, (config, rhs) in zip((0, 0, 0, 1, 2, 2, 3), state["weights"])]
    if op == "block":
        w = [rhs[0] for _, rhs in state["weights"]]
        q, k, v = qmatmul_grouped(enc, state["lhs"][0], w[:3])
        o = qmatmul(enc, None, state["lhs"][1], w[3])
        hidden = qmatmul_swiglu(enc, state["lhs"][2], w[4], w[5])
        return [q, k, v, o, qmatmul(enc, None, hidden, w[6])]
    if op == "rmsnorm":
        return qmatmul_rmsnorm(enc, state["config"], state["lhs"], state["gamma"], EPS, *state["rhs"], out_dtype=LHS[case.get("out", "f32")])
    if op == "repacked":
        return qmatmul_repacked(state["lhs"], state["packed"])
    if op == "dequantize":
        return dequantize(enc, *state["rhs"], config=state["config"], dtype=LHS[case["out"]])
    if enc == QE.GPTQ:
        return quantize_gptq(state["x"], QuantizationConfig("gptq", 4, case["group"], False, True))
    return quantize(enc, state["x"])


def _packed_bytes(case, n, k):
    if case["enc"] == "GPTQ":
        groups = k // case["group"]
        return n * k // 2 + groups * n * 2 + groups * n // 2 + (4 * k if case.get("order") or case["op"] == "quantize" else 0)
    return n * QE[case["enc"]].packed_row_bytes(k)


def work(case):
    op = case["op"]
    if op == "quantize":
        return {"bytes": 4 * case["n"] * case["k"] + _packed_bytes(case, case["n"], case["k"]), "flops": 0}
    if op == "dequantize":
        return {"bytes": (2 if case["out"] == "bf16" else 4) * case["n"] * case["k"] + _packed_bytes(case, case["n"], case["k"]), "flops": 0}
    m, el = case["m"], 4 if case["lhs"] == "f32" else 2
    if op in ("layer", "block"):
        shapes = _projections(case)
        outs = [n for n, _ in shapes] if op == "layer" else [n for n, _ in shapes[:4]] + [case["hidden"]]
        ins = 3 * case["hidden"] + (case["ffn"] if op == "layer" else 0)
        return {"bytes": sum(_packed_bytes(case, n, k) for n, k in shapes) + m * (el * ins + 4 * sum(outs)),
                "flops": 2 * m * sum(n * k for n, k in shapes)}
    n, k = case["n"], case["k"]
    return {"bytes": _packed_bytes(case, n, k) + m * (el * k + (2 if case.get("out") == "bf16" else 4) * n) + (4 * k if op == "rmsnorm" else 0),
            "flops": 2 * m * n * k}


def tolerance(case):
    if case["op"] in ("dequantize", "quantize"):
        return "exact"
    if case.get("out") == "bf16":
        return {"rel": 5e-3, "max": 2e-2}  # two results that round to neighbouring bf16 values
    if case["op"] == "rmsnorm" and (case["lhs"] == "bf16" or case["enc"] == "Q4_0"):
        return {"rel": 2e-3, "max": 1e-2}  # a normalised value on a rounding boundary (bf16, or a code of the Q8_0 lhs)
    if case["op"] == "block" and case["enc"] == "Q4_0":
        return {"rel": 2e-3, "max": 1e-2}  # likewise: the lhs of down is quantised from a computed value
    return {"rel": 2e-5, "max": 1e-3}  # integer codes and exact products, sums in 32 bits
