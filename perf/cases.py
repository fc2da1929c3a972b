"""What this framework's speed is measured on: calls of prepared tensor-ring operators.

A case is one pass through the public entry points (a prepared operator's call, its fused
epilogues, the SwiGLU pair, the elementwise consumers), over the shapes, ranks and element
types of the repository's benchmarks: 1920 -> 2880 in fp16 and fp32, the Llama-3-8B
projections and the Qwen3.8-27B layer shapes in bf16, at ring ranks 8, 12 (zero-padded to 16)
and 16. Token counts run from one (decode) through small and ordinary batches to a prefill of
2048, ragged ones among them. The operator has a forward direction only.
"""
from __future__ import annotations

import math
import os
import sys
from pathlib import Path

# kernel arguments in host memory, as a latency-bound program of this framework sets it before
# HIP initialises (bench.py does)
os.environ.setdefault("HIP_FORCE_DEV_KERNARG", "0")
sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "kernel-task_amd"))

import torch  # noqa: E402
import torch.nn.functional as F  # noqa: E402

from factorized_inference import TRSpec, prepare_optimized  # noqa: E402
from factorized_inference.tr_kernel import consume_silu_mul, forward_swiglu  # noqa: E402

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}

# name: (input modes, output modes), the benchmarks' layers
SHAPES = {
    "base": ((8, 12, 20), (12, 10, 24)),          # 1920 -> 2880
    "llama_up": ((16, 16, 16), (16, 28, 32)),     # 4096 -> 14336 (gate and up)
    "llama_down": ((16, 28, 32), (16, 16, 16)),   # 14336 -> 4096
    "qwen_gate_up": ((20, 16, 16), (16, 34, 32)),  # 5120 -> 17408
    "qwen_down": ((34, 32, 16), (16, 16, 20)),    # 17408 -> 5120
    "qwen_qgate": ((20, 16, 16), (16, 24, 32)),   # 5120 -> 12288
    "qwen_kv": ((20, 16, 16), (8, 8, 16)),        # 5120 -> 1024
    "qwen_o": ((24, 16, 16), (16, 16, 20)),       # 6144 -> 5120
    "qwen_qkvz": ((20, 16, 16), (16, 32, 32)),    # 5120 -> 16384
}
# (shape, rank, dtype) of single operators as the benchmarks run them
OPERATORS = [("base", 8, "f16"), ("base", 16, "f16"), ("base", 8, "f32"),
             ("llama_up", 8, "bf16"), ("llama_down", 16, "bf16")] + [
    (s, r, "bf16") for s in ("qwen_gate_up", "qwen_down", "qwen_qgate", "qwen_kv", "qwen_o",
                             "qwen_qkvz") for r in (8, 12, 16)]
MAX_TOKENS = 2048


def op(name, shape, rank, dtype, tokens, call="plain"):
    return {"name": name, "kind": "op", "shape": shape, "rank": rank, "dtype": dtype,
            "tokens": tokens, "call": call}


def listed():
    return [
        # decode, one sequence: the benchmark's headline, bound by the launch
        op("base_r8_f16_t1", "base", 8, "f16", 1),
        # decode of a small batch
        op("base_r8_f16_t32", "base", 8, "f16", 32),
        op("base_r16_f16_t32", "base", 16, "f16", 32),
        # a prefill of ragged length
        op("base_r8_f16_t1023", "base", 8, "f16", 1023),
        # fp32, an evaluation batch
        op("base_r8_f32_t100", "base", 8, "f32", 100),
        # decode through the largest down projection, the residual fused into the store
        op("llama_down_r16_bf16_t1_add", "llama_down", 16, "bf16", 1, "add"),
        # the benchmark's largest token count on it
        op("llama_down_r16_bf16_t256", "llama_down", 16, "bf16", 256),
        # a serving batch through a wide attention projection
        op("qwen_qgate_r16_bf16_t128", "qwen_qgate", 16, "bf16", 128),
        # a rank without kernels of its own (zero-padded), ragged prompt, narrow outputs
        op("qwen_kv_r12_bf16_t300", "qwen_kv", 12, "bf16", 300),
        # prefill through the largest layer
        op("qwen_down_r16_bf16_t2048", "qwen_down", 16, "bf16", 2048),
        # a whole SwiGLU MLP block with its residual (gate and up in one launch, then down)
        {"name": "llama_mlp_bf16_t64", "kind": "mlp", "tokens": 64, "dtype": "bf16"},
        # the standalone consumer over fp32 outputs held from elsewhere, prefill-sized
        {"name": "silu_mul_bf16_t2048", "kind": "silu_mul", "tokens": 2048, "dtype": "bf16"},
    ]


def _tokens(rng, most=MAX_TOKENS):
    return int(round(math.exp(rng.uniform(0.0, math.log(most)))))


def draw(rng):
    kind = rng.choice(["op"] * 8 + ["mlp", "silu_mul"])
    if kind == "op":
        shape, rank, dtype = rng.choice(OPERATORS)
        return {"kind": "op", "shape": shape, "rank": rank, "dtype": dtype,
                "tokens": _tokens(rng),
                "call": rng.choice(["plain", "plain", "add", "silu_mul", "f32"])}
    if kind == "mlp":  # two operators: fewer tokens keep it within the largest listed case
        return {"kind": "mlp", "tokens": _tokens(rng, 1024), "dtype": "bf16"}
    return {"kind": "silu_mul", "tokens": _tokens(rng), "dtype": rng.choice(["f16", "bf16", "f32"])}


# ---- inputs, from the seed alone -------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _cores(g, shape, rank, dtype):
    """Cores of variance 1 / (rank * input mode), which gives the weight variance 1 / in."""
    ins, outs = SHAPES[shape]
    return [(torch.randn(rank, o, i, rank, generator=g, device="cuda") / math.sqrt(rank * i)
             ).to(dtype) for i, o in zip(ins, outs)]


def _features(shape):
    ins, outs = SHAPES[shape]
    return math.prod(ins), math.prod(outs)


def _inputs(case, seed):
    g, t, dt = _gen(seed), case["tokens"], DTYPES[case["dtype"]]
    randn = lambda n, dtype: torch.randn(t, n, generator=g, device="cuda").to(dtype)  # noqa: E731
    if case["kind"] == "silu_mul":
        n = _features("llama_up")[1]
        return {"g": randn(n, torch.float32), "u": randn(n, torch.float32)}
    if case["kind"] == "mlp":
        n = _features("llama_up")[0]
        return {"x": randn(n, dt), "h": randn(n, dt), "gate": _cores(g, "llama_up", 8, dt),
                "up": _cores(g, "llama_up", 8, dt), "down": _cores(g, "llama_down", 16, dt)}
    n_in, n_out = _features(case["shape"])
    made = {"x": randn(n_in, dt), "cores": _cores(g, case["shape"], case["rank"], dt)}
    if case["call"] in ("add", "silu_mul"):
        # the residual in the operator's type, the gate in fp32 as accumulate() returns it
        made["aux"] = randn(n_out, dt if case["call"] == "add" else torch.float32)
    return made


def _spec(shape, rank):
    return TRSpec(*SHAPES[shape], rank)


def prepare(case, seed):
    made = _inputs(case, seed)
    state = {"kind": case["kind"], "call": case.get("call"), "dtype": DTYPES[case["dtype"]]}
    if case["kind"] == "silu_mul":
        return state | made
    if case["kind"] == "mlp":
        return state | {"x": made["x"], "h": made["h"],
                        "gate": prepare_optimized(made["gate"], _spec("llama_up", 8)),
                        "up": prepare_optimized(made["up"], _spec("llama_up", 8)),
                        "down": prepare_optimized(made["down"], _spec("llama_down", 16))}
    return state | {"x": made["x"], "aux": made.get("aux"),
                    "fn": prepare_optimized(made["cores"], _spec(case["shape"], case["rank"]))}


def run(state):
    kind, call = state["kind"], state["call"]
    if kind == "silu_mul":
        return consume_silu_mul(state["g"], state["u"], state["dtype"])
    if kind == "mlp":
        act = forward_swiglu(state["gate"], state["up"], state["x"])
        return state["down"].forward_add(act, state["h"])
    fn, x = state["fn"], state["x"]
    if call == "add":
        return fn.forward_add(x, state["aux"])
    if call == "silu_mul":
        return fn.forward_silu_mul(x, state["aux"])
    if call == "f32":
        return fn.accumulate(x)
    return fn(x)


# ---- what a pass cannot do without ------------------------------------------------------------
def _least_macs(shape, rank, tokens):
    """Multiply-adds of the cheapest contraction of x with the three cores: x through the
    cores one after another, in the best order, or two cores joined, then the third, then x."""
    ins, outs = SHAPES[shape]
    n_in, n_out, r = math.prod(ins), math.prod(outs), rank
    through = min(tokens * (n_in * outs[f] * r ** 2
                            + ins[s] * ins[l] * outs[f] * outs[s] * r ** 3
                            + ins[l] * n_out * r ** 2)
                  for f, s, l in ((0, 1, 2), (1, 2, 0), (2, 0, 1), (0, 2, 1), (1, 0, 2), (2, 1, 0)))
    joined = n_in * n_out * (tokens + r ** 2) + min(
        ins[a] * outs[a] * ins[b] * outs[b] * r ** 3 for a, b in ((0, 1), (1, 2), (2, 0)))
    return min(through, joined)


def _core_values(shape, rank):
    return sum(rank * rank * i * o for i, o in zip(*SHAPES[shape]))


def work(case):
    t, e = case["tokens"], DTYPES[case["dtype"]].itemsize
    if case["kind"] == "silu_mul":
        n = t * _features("llama_up")[1]
        return {"bytes": n * (4 + 4 + e), "flops": 5 * n}
    if case["kind"] == "mlp":
        n = _features("llama_up")[0]
        return {"bytes": e * (2 * _core_values("llama_up", 8) + _core_values("llama_down", 16)
                              + 3 * t * n),
                "flops": 2 * (2 * _least_macs("llama_up", 8, t) + _least_macs("llama_down", 16, t))}
    n_in, n_out = _features(case["shape"])
    aux = {"add": e, "silu_mul": 4}.get(case["call"], 0)
    out = 4 if case["call"] == "f32" else e
    return {"bytes": e * (_core_values(case["shape"], case["rank"]) + t * n_in)
            + t * n_out * (out + aux),
            "flops": 2 * _least_macs(case["shape"], case["rank"], t)}


def tolerance(case):
    """Four times the difference of two correct results: each is 3.6e-4 (fp16), 2.9e-3 (bf16)
    or 4.8e-7 (fp32) from the 64-bit one, measured (the intermediates between contractions are
    kept in the operator's type), so two of them differ by 1.4 times that. The consumer rounds
    once: about twice its measured distance (1.7e-3 in bf16)."""
    if case["kind"] == "silu_mul":
        return {"rel": {"f16": 4.5e-4, "bf16": 3.5e-3, "f32": 5e-7}[case["dtype"]]}
    if case["kind"] == "mlp":
        return {"rel": 2e-2}
    return {"rel": {"f16": 2e-3, "bf16": 1.6e-2, "f32": 3e-6}[case["dtype"]]}


# ---- the same results in 64 bits, by plain torch -----------------------------------------------
def _dense64(cores, shape):
    """The [in, out] weight the cores stand for, in 64 bits."""
    (ni, nj, nk), (p, q, r) = SHAPES[shape]
    g1, g2, g3 = (c.double() for c in cores)
    R = g1.shape[0]
    ab = (g1.reshape(-1, R) @ g2.reshape(R, -1)).reshape(R, p, ni, q, nj, R)
    ab = ab.permute(2, 4, 1, 3, 5, 0).reshape(ni * nj * p * q, R * R)      # (i j p q)(c a)
    w = ab @ g3.permute(0, 3, 2, 1).reshape(R * R, nk * r)                 # (i j p q)(k r)
    w = w.reshape(ni, nj, p, q, nk, r).permute(0, 1, 4, 2, 3, 5)
    return w.reshape(ni * nj * nk, p * q * r)


def _apply64(x, cores, shape):
    return x.double() @ _dense64(cores, shape)


def exact(case, seed):
    made = _inputs(case, seed)
    if case["kind"] == "silu_mul":
        return F.silu(made["g"].double()) * made["u"].double()
    if case["kind"] == "mlp":
        act = F.silu(_apply64(made["x"], made["gate"], "llama_up"))
        act = act * _apply64(made["x"], made["up"], "llama_up")
        return made["h"].double() + _apply64(act, made["down"], "llama_down")
    y = _apply64(made["x"], made["cores"], case["shape"])
    if case["call"] == "add":
        return made["aux"].double() + y
    if case["call"] == "silu_mul":
        return F.silu(made["aux"].double()) * y
    return y
