"""What a user of this library has it do, as measurable cases: single-row and batched projections, the dense SwiGLU
FFN from one decode row to a prefill chunk, the MoE block, a decoder step replayed from a graph, and the host-buffer
product that a CPU graph node makes.  Weights come from the library's seeded synthetic recipe (uniform quants and
scales, fp16 block scales in [0.001, 0.01)), activations and router logits are N(0, 1).
"""
import math

import numpy as np
import torch

from densecore_amd import decode_step, ops

# bytes of 256 weights of a row
_BLOCK = {"q4_k": 144, "q5_k": 176, "q6_k": 210, "q8_0": 272}
_TYPE = {"q4_k": ops.GGML_TYPE_Q4_K, "q5_k": ops.GGML_TYPE_Q5_K, "q6_k": ops.GGML_TYPE_Q6_K, "q8_0": ops.GGML_TYPE_Q8_0}

# The dense FFN is the 4096 -> 14336 -> 4096 block that the benchmark is quoted on, the MoE block the 256-expert
# top-8 2048 x 512 one with a shared expert, the projections those of the same two models.
_LISTED = [
    # one attention projection of a small model, one token: a launch and little else
    {"name": "gemv 2048x2048 n1", "op": "mul_mat", "type": "q4_k", "rows": 2048, "cols": 2048, "n": 1},
    # the same node called from a CPU graph: host row in, host row out
    {"name": "host gemv 4096x4096 n1", "op": "mul_mat_host", "type": "q4_k", "rows": 4096, "cols": 4096, "n": 1},
    # dense FFN, one sequence decoding
    {"name": "ffn n1", "op": "ffn", "type": "q4_k", "down_type": "q4_k", "hidden": 4096, "inter": 14336, "n": 1},
    # dense FFN, thirteen sequences decoding together (an odd batch); Q6_K down as Q4_K_M files have it for half the layers
    {"name": "ffn q6 down n13", "op": "ffn", "type": "q4_k", "down_type": "q6_k", "hidden": 4096, "inter": 14336, "n": 13},
    # dense FFN, a large decode batch or a short prompt
    {"name": "ffn n50", "op": "ffn", "type": "q4_k", "down_type": "q4_k", "hidden": 4096, "inter": 14336, "n": 50},
    # dense FFN, a ragged prompt
    {"name": "ffn n391", "op": "ffn", "type": "q4_k", "down_type": "q4_k", "hidden": 4096, "inter": 14336, "n": 391},
    # dense FFN, a full prefill chunk
    {"name": "ffn n2048", "op": "ffn", "type": "q4_k", "down_type": "q4_k", "hidden": 4096, "inter": 14336, "n": 2048},
    # the output projection of a 128256-token vocabulary (Q6_K in Q4_K_M files), three sequences decoding
    {"name": "vocab q6 n3", "op": "mul_mat", "type": "q6_k", "rows": 128256, "cols": 4096, "n": 3},
    # a Q5_K projection at a prefill width (Q5_K_M files), ragged rows and tokens
    {"name": "mul_mat q5 n1000", "op": "mul_mat", "type": "q5_k", "rows": 6152, "cols": 4096, "n": 1000},
    # eight MoE decoder layers, one token, replayed from a HIP graph as a serving loop does
    {"name": "moe step n1", "op": "step", "layers": 8, "hidden": 2048, "inter": 512, "experts": 256, "top_k": 8, "n": 1},
    # MoE block, a decode batch
    {"name": "moe n24", "op": "moe", "type": "q4_k", "down_type": "q4_k", "hidden": 2048, "inter": 512, "experts": 256,
     "top_k": 8, "shared": True, "n": 24},
    # MoE block, a prefill chunk
    {"name": "moe n1500", "op": "moe", "type": "q4_k", "down_type": "q4_k", "hidden": 2048, "inter": 512, "experts": 256,
     "top_k": 8, "shared": True, "n": 1500},
]
_MOST = 2.0 * 3 * 4096 * 14336 * 2048  # operations of the largest listed case


def listed():
    return [dict(c) for c in _LISTED]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _blocks(rng, lo, hi):
    """A row length: a multiple of 256 spread over the logarithm of [lo, hi]."""
    return 256 * max(1, _log_int(rng, lo // 256, hi // 256))


def _draw(rng):
    op = rng.choice(("mul_mat", "mul_mat", "mul_mat_host", "ffn", "ffn", "ffn", "moe", "moe", "step"))
    if op == "mul_mat":
        vocab = rng.random() < 0.2
        rows = rng.randint(32000, 128256) if vocab else _log_int(rng, 512, 16384)
        return {"op": op, "type": rng.choice(("q4_k", "q4_k", "q5_k", "q6_k", "q8_0")), "rows": rows,
                "cols": _blocks(rng, 1024, 5120 if vocab else 14336), "n": _log_int(rng, 1, 32 if vocab else 2048)}
    if op == "mul_mat_host":
        return {"op": op, "type": rng.choice(("q4_k", "q5_k", "q6_k")), "rows": _log_int(rng, 512, 14336),
                "cols": _blocks(rng, 1024, 8192), "n": _log_int(rng, 1, 48)}
    if op == "ffn":
        hidden = _blocks(rng, 1024, 5120)
        return {"op": op, "type": rng.choice(("q4_k", "q4_k", "q5_k", "q6_k")), "down_type": rng.choice(("q4_k", "q4_k", "q5_k", "q6_k")),
                "hidden": hidden, "inter": _blocks(rng, 2 * hidden, min(4 * hidden, 14336)), "n": _log_int(rng, 1, 2048)}
    if op == "moe":
        experts = rng.choice((8, 16, 64, 128, 256))
        return {"op": op, "type": rng.choice(("q4_k", "q4_k", "q5_k", "q6_k")), "down_type": rng.choice(("q4_k", "q5_k", "q6_k")),
                "hidden": _blocks(rng, 1024, 4096), "inter": _blocks(rng, 256, 1024), "experts": experts,
                "top_k": rng.choice((2, 4, 6, 8)), "shared": rng.random() < 0.5, "n": _log_int(rng, 1, 2048)}
    return {"op": op, "layers": rng.randint(2, 8), "hidden": rng.choice((1024, 2048, 2048, 2560)), "inter": rng.choice((256, 512, 768)),
            "experts": rng.choice((32, 64, 128, 256)), "top_k": rng.choice((4, 8)), "n": _log_int(rng, 1, 16)}


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        if w["flops"] <= _MOST and w["bytes"] <= 1.5e9:
            return c


def _weight(seed, tag, rows, cols, experts=1, kind="q4_k"):
    return ops.Q4KWeight.synthetic((seed * 1000003 + tag) & 0x7FFFFFFFFFFFFFFF, rows, cols, experts, _TYPE[kind])


def _silu(op, n):
    """The SiLU form the graph asks for: the polynomial in a dense FFN; in a MoE block exact up to four tokens, the polynomial above."""
    if op == "ffn":
        return ops.SILU_FAST_FMA
    return ops.SILU_EXACT if n <= 4 else ops.SILU_FAST


def prepare(case, seed):
    op, n = case["op"], case["n"]
    state = {"case": case}
    if op == "mul_mat_host":
        state["w"] = _weight(seed, 1, case["rows"], case["cols"], kind=case["type"])
        state["x"] = np.random.default_rng(seed).standard_normal((n, case["cols"]), dtype=np.float32)
        return state
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(shape, device="cuda", dtype=torch.float32, generator=gen)

    if op == "mul_mat":
        state["w"] = _weight(seed, 1, case["rows"], case["cols"], kind=case["type"])
        state["x"] = normal(n, case["cols"])
    elif op == "ffn":
        h, i = case["hidden"], case["inter"]
        state["w"] = (_weight(seed, 1, i, h, kind=case["type"]), _weight(seed, 2, i, h, kind=case["type"]), _weight(seed, 3, h, i, kind=case["down_type"]))
        state["x"] = normal(n, h)
    elif op == "moe":
        h, i, e = case["hidden"], case["inter"], case["experts"]
        state["w"] = (_weight(seed, 1, i, h, e, case["type"]), _weight(seed, 2, i, h, e, case["type"]), _weight(seed, 3, h, i, e, case["down_type"]))
        state["shared"] = None
        if case["shared"]:
            state["shared"] = (_weight(seed, 4, i, h, kind=case["type"]), _weight(seed, 5, i, h, kind=case["type"]),
                               _weight(seed, 6, h, i, kind=case["down_type"]), normal(h) * h ** -0.5)
        state["x"], state["logits"] = normal(n, h), normal(n, e)
    else:
        cfg = decode_step.StepConfig(n_layers=case["layers"], hidden=case["hidden"], n_experts=case["experts"], inter=case["inter"],
                                     top_k=case["top_k"], n_q=case["hidden"], seed=seed, synthetic_logits=True)
        step = decode_step.DecodeStep(cfg, n)
        state["x"] = normal(n, case["hidden"])
        step.run(state["x"])
        step.capture()
        state["step"] = step
    return state


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "mul_mat_host":
        return ops.mul_mat_host(state["w"], state["x"])
    if op == "mul_mat":
        return ops.mul_mat(state["w"], state["x"])
    if op == "ffn":
        return ops.ffn_swiglu(*state["w"], state["x"], _silu(op, case["n"]))
    if op == "moe":
        y, ids, weights = ops.moe_layer(*state["w"], state["x"], state["logits"], case["top_k"], shared=state["shared"], silu=_silu(op, case["n"]))
        return {"y": y, "ids": ids, "weights": weights}
    step = state["step"]
    step.x.copy_(state["x"])
    return {"y": step.replay(), "ids": step.ids, "weights": step.wts}


def _matrix(rows, cols, kind):
    return rows * (cols // 256) * _BLOCK[kind]


def work(case):
    op, n = case["op"], case["n"]
    if op in ("mul_mat", "mul_mat_host"):
        return {"bytes": _matrix(case["rows"], case["cols"], case["type"]) + 4.0 * n * (case["rows"] + case["cols"]),
                "flops": 2.0 * n * case["rows"] * case["cols"]}
    h, i = case["hidden"], case["inter"]
    if op == "ffn":
        return {"bytes": 2.0 * _matrix(i, h, case["type"]) + _matrix(h, i, case["down_type"]) + 8.0 * n * h, "flops": 6.0 * n * h * i}
    e, k = case["experts"], case["top_k"]
    touched = e * (1.0 - (1.0 - k / e) ** n)  # distinct experts of n tokens that route uniformly
    shared = 1 if case.get("shared", True) else 0
    kind, down = case.get("type", "q4_k"), case.get("down_type", "q4_k")
    block = (touched + shared) * (2.0 * _matrix(i, h, kind) + _matrix(h, i, down))
    flops = 6.0 * n * h * i * (k + shared)
    if op == "moe":
        return {"bytes": block + 4.0 * n * (2 * h + e + 2 * k), "flops": flops}
    qkv = h + 2 * 256
    layer = block + _matrix(qkv, h, "q4_k") + _matrix(h, h, "q4_k") + 4.0 * e * h + 8.0 * n * k
    return {"bytes": case["layers"] * layer + 8.0 * n * h, "flops": case["layers"] * (flops + 2.0 * n * h * (qkv + h + e))}


def tolerance(case):
    # Measured as the same rows through the library's kernels for other widths, which sum in another order, and stated as
    # four times that: a single product differs by the order of its fp32 sums alone (1.6e-7, largest 7.8e-7); behind a
    # second quantizer (FFN, MoE block) a last-bit difference of a hidden value now and then moves its 8-bit code by one
    # (5e-5, largest 1e-3).
    return {"rel": 7e-7, "max": 4e-6} if case["op"] in ("mul_mat", "mul_mat_host") else {"rel": 2e-4, "max": 4e-3}
