"""The work a serving engine hands to this package, as timed cases: quantized linear layers from one decoded token to a
prefill chunk of thousands, the activation quantizers on their own, and the grouped expert GEMM of a mixture-of-experts layer.

Every case goes through the entry points the layers of a model call (`fp8_utils`, `w8a8_int8`, `fp8_kernel`, `sgl_kernel`).
Shapes are the configurations of `sglang_amd.workloads` (DeepSeek-V3 MLP and MLA projections, Llama-3-8B), their slices under
tensor parallelism, and generic sizes of the same ranges.  Weights and their scales are prepared once, as at load time.
"""
from __future__ import annotations

import math
import random
from typing import Any, Dict, List

import torch

from sglang_amd import fp8_kernel, fp8_utils, sgl_kernel, w8a8_int8
from sglang_amd.workloads import DSV3_MLA, DSV3_MLP, LLAMA3_8B

BLOCK = [128, 128]
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
FP8 = torch.float8_e4m3fn

# The most multiply-adds, quantized values and expert weights of a drawn case, about those of the largest listed ones.
MOST_MACS = 4096 * 7168 * 36864
MOST_VALUES = 16384 * 7168
MOST_EXPERT_WEIGHTS = 256 * 512 * 7168

GATE_UP, DOWN = DSV3_MLP["gate_up"], DSV3_MLP["down"]
KV_A, Q_B, KV_B = DSV3_MLA["kv_a"], DSV3_MLA["q_b"], DSV3_MLA["kv_b"]


def _linear(kind: str, M: int, layer, dtype: str = "bf16", bias: bool = False, static: bool = False) -> Dict[str, Any]:
    K, N = layer
    return {"kind": kind, "M": M, "K": K, "N": N, "dtype": dtype, "bias": bias, "static": static}


def listed() -> List[Dict[str, Any]]:
    cases = {
        # one sequence being decoded through the smallest projection of a layer (64 x 9 channels: not whole 128-blocks)
        "block_decode_1_kv_a": _linear("block", 1, KV_A),
        # a small decode batch through the widest layer: the weight is streamed once per step
        "block_decode_8_gate_up": _linear("block", 8, GATE_UP),
        # a decode batch of a busy server, checkpoint re-quantized to power-of-two scales at load time
        "ue8m0_decode_48_down": _linear("ue8m0", 48, DOWN),
        # a chunk of a prompt that shares the step with decoding requests: a few hundred tokens, no round number
        "block_chunk_387_q_b": _linear("block", 387, Q_B),
        # prefill through a layer of short K and many channels, where writing the result is most of the traffic
        "block_prefill_3001_kv_b": _linear("block", 3001, KV_B),
        # a full prefill chunk through the widest layer: the most arithmetic of a step
        "block_prefill_4096_gate_up": _linear("block", 4096, GATE_UP),
        # INT8 checkpoints: one decoded token, and a prefill chunk with a bias
        "int8_decode_1_qkv": _linear("int8", 1, LLAMA3_8B["qkv"]),
        "int8_prefill_2048_down": _linear("int8", 2048, LLAMA3_8B["down"], bias=True),
        # per-channel FP8 checkpoints with dynamic per-token activation scales, fp16 model with biases, a medium batch
        "token_fp8_batch_160_gate_up": _linear("token_fp8", 160, LLAMA3_8B["gate_up"], dtype="fp16", bias=True),
        # the activation quantizer by itself on a prefill batch (what feeds grouped GEMMs and communication)
        "group_quant_16384": {"kind": "group_quant", "M": 16384, "K": 7168, "dtype": "bf16", "layout": "col_aligned"},
        # between the two GEMMs of an expert MLP in the masked layout: SwiGLU and the quantizer, rows up to each expert's count
        "silu_quant_masked_32x256": {"kind": "silu_quant", "E": 32, "T": 256, "H": 2048, "dtype": "bf16", "masked": True},
        # the expert GEMM of a mixture-of-experts layer, 128 tokens routed to 8 of 256 experts each (slice of 512 channels)
        "grouped_256_experts_1024_rows": {"kind": "grouped", "E": 256, "rows": 1024, "K": 7168, "N": 512, "dtype": "bf16"},
    }
    return [dict(case, name=name) for name, case in cases.items()]


# ---------------------------------------------------------------- drawn cases

def _spread(rng: random.Random, low: int, high: int) -> int:
    """An integer of [low, high], even over its logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _layer(rng: random.Random, block: bool):
    """(K, N): a layer of the configurations or a slice of it under tensor parallelism, or a generic one."""
    if rng.random() < 0.6:
        K, N = rng.choice([*DSV3_MLP.values(), *DSV3_MLA.values(), *LLAMA3_8B.values()])
        tp = rng.choice([1, 1, 2, 4, 8])
        if rng.random() < 0.5 and N % (64 * tp) == 0:
            N //= tp      # column-parallel
        elif K % (128 * tp) == 0:
            K //= tp      # row-parallel
        return max(K, 256), max(N, 128)
    K, N = 128 * _spread(rng, 4, 144), 128 * _spread(rng, 2, 288)
    if rng.random() < 0.25:
        N += 64           # channels not in whole 128-blocks
    if not block and rng.random() < 0.25:
        K += rng.choice([16, 32, 64, 96])  # a row-parallel slice of an intermediate size that is no multiple of 128
    return K, N


def draw(rng: random.Random) -> Dict[str, Any]:
    kind = rng.choice(["block", "block", "block", "block", "ue8m0", "ue8m0", "int8", "int8", "token_fp8", "token_fp8",
                       "group_quant", "silu_quant", "grouped"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if kind in ("block", "ue8m0", "int8", "token_fp8"):
        K, N = _layer(rng, block=kind in ("block", "ue8m0"))
        M = _spread(rng, 1, 4096 if K % 128 == 0 else 512)
        M = max(1, min(M, MOST_MACS // (2 * K * N)))
        return _linear(kind, M, (K, N), "bf16" if kind == "ue8m0" else dtype, bias=rng.random() < 0.25,
                       static=kind == "token_fp8" and rng.random() < 0.25)
    if kind == "group_quant":
        K = 128 * _spread(rng, 4, 144)
        M = min(_spread(rng, 1, 16384), MOST_VALUES // K)
        return {"kind": kind, "M": M, "K": K, "dtype": dtype, "layout": rng.choice(["row", "col", "col_aligned", "ue8m0"])}
    if kind == "silu_quant":
        masked = rng.random() < 0.5
        E = rng.choice([8, 16, 32]) if masked else 1
        H = 128 * _spread(rng, 4, 32)
        T = _spread(rng, 1, min(32768, MOST_VALUES // (2 * H)) // E)
        return {"kind": kind, "E": E, "T": T, "H": H, "dtype": dtype, "masked": masked}
    E = rng.choice([8, 16, 32, 64, 128, 256])
    K = 128 * _spread(rng, 4, 56)
    N = 128 * _spread(rng, 2, max(2, min(32, MOST_EXPERT_WEIGHTS // (E * K * 128))))
    rows = max(1, min(_spread(rng, 8, 8192), MOST_MACS // (4 * K * N)))
    return {"kind": kind, "E": E, "rows": rows, "K": K, "N": N, "dtype": dtype}


# ---------------------------------------------------------------- inputs

def _generator(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _activation(g: torch.Generator, *shape: int, dtype: torch.dtype) -> torch.Tensor:
    """N(0, 1) with one value in a thousand fifty times as large, as activations of large models have."""
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    x *= torch.where(torch.rand(shape, generator=g, device="cuda") < 1e-3, 50.0, 1.0)
    return x.to(dtype)


def _normal_weight(g: torch.Generator, *shape: int, dtype: torch.dtype = torch.float32) -> torch.Tensor:
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype) * 0.02


def _block_fp8_weight(g: torch.Generator, N: int, K: int):
    """e4m3fn codes [N, K] and one fp32 scale per 128 x 128 block."""
    nb, kb = -(-N // 128), -(-K // 128)
    w = torch.zeros((nb * 128, kb * 128), device="cuda")
    w[:N, :K] = _normal_weight(g, N, K)
    v = w.view(nb, 128, kb, 128)
    amax = v.abs().amax(dim=(1, 3), keepdim=True).clamp(min=1e-4)
    q = (v * (448.0 / amax)).clamp(-448.0, 448.0).to(FP8).view(nb * 128, kb * 128)[:N, :K].contiguous()
    return q, (amax / 448.0).view(nb, kb).contiguous()


def _prepare_linear(case: Dict[str, Any], g: torch.Generator) -> Dict[str, Any]:
    kind, M, K, N = case["kind"], case["M"], case["K"], case["N"]
    dtype = DTYPES[case["dtype"]]
    state = {"x": _activation(g, M, K, dtype=dtype), "input_scale": None}
    if kind == "block":
        state["fn"] = fp8_utils.dispatch_w8a8_block_fp8_linear()
        state["w"], state["ws"] = _block_fp8_weight(g, N, K)
    elif kind == "ue8m0":
        w, s = fp8_utils.quant_weight_ue8m0(_normal_weight(g, N, K, dtype=torch.bfloat16), BLOCK)
        state["w"], state["ws"] = w, fp8_utils.transform_scale_ue8m0(s, mn=N)
    else:
        w = _normal_weight(g, N, K)
        amax = w.abs().amax(dim=1, keepdim=True).clamp(min=1e-10)
        if kind == "int8":
            state["ws"] = amax / 127.0
            state["w"] = torch.round(w / state["ws"]).clamp(-127, 127).to(torch.int8).t()
        else:
            state["ws"] = amax / 448.0
            state["w"] = (w / state["ws"]).clamp(-448.0, 448.0).to(FP8).t()
            if case["static"]:
                state["input_scale"] = (state["x"].abs().amax().float() / 448.0).reshape(1)
    state["bias"] = torch.randn(N, generator=g, device="cuda").to(dtype) if case["bias"] else None
    return state


def _prepare_grouped(case: Dict[str, Any], g: torch.Generator) -> Dict[str, Any]:
    """Token rows sorted by expert, quantized, and what the engine keeps beside them for every step."""
    E, rows, K, N = case["E"], case["rows"], case["K"], case["N"]
    i32 = {"dtype": torch.int32, "device": "cuda"}
    # experts are not equally popular
    popular = torch.rand(E, generator=g, device="cuda") + 0.25
    counts = torch.bincount(torch.multinomial(popular, rows, replacement=True, generator=g), minlength=E)
    sizes = torch.stack([counts, torch.full_like(counts, N), torch.full_like(counts, K)], dim=1).to(torch.int32).contiguous()
    offsets = (torch.cumsum(counts, 0) - counts).to(torch.int32)
    a, sa = fp8_kernel.per_token_group_quant_fp8(_activation(g, rows, K, dtype=torch.bfloat16), 128)
    b, sb = _block_fp8_weight(g, E * N, K)
    pointers = [torch.empty(E, dtype=torch.int64, device="cuda") for _ in range(5)]
    strides = [torch.full((E,), s, dtype=torch.int64, device="cuda") for s in (K, K, N)]
    layouts = [torch.empty((E, 5), **i32) for _ in range(2)]
    return {
        "out": torch.empty((rows, N), dtype=DTYPES[case["dtype"]], device="cuda"), "pointers": pointers, "a": a,
        "b": b.view(E, N, K).transpose(1, 2), "sa": sa, "sb": sb.view(E, N // 128, K // 128).transpose(1, 2),
        "strides": strides, "layouts": layouts, "sizes": sizes, "offsets": offsets,
        "workspace": torch.empty(64 << 20, dtype=torch.uint8, device="cuda"),
    }


def prepare(case: Dict[str, Any], seed: int) -> Dict[str, Any]:
    g = _generator(seed)
    kind = case["kind"]
    if kind == "group_quant":
        state = {"x": _activation(g, case["M"], case["K"], dtype=DTYPES[case["dtype"]]), "layout": case["layout"]}
    elif kind == "silu_quant":
        E, T, H = case["E"], case["T"], case["H"]
        shape = (E, T, 2 * H) if case["masked"] else (T, 2 * H)
        state = {"x": _activation(g, *shape, dtype=DTYPES[case["dtype"]]), "masked_m": None}
        if case["masked"]:  # an expert's rows are allotted for the worst case and partly used
            state["masked_m"] = torch.randint(0, T + 1, (E,), generator=g, device="cuda", dtype=torch.int32)
    elif kind == "grouped":
        state = _prepare_grouped(case, g)
    else:
        state = _prepare_linear(case, g)
    state["kind"] = kind
    return state


# ---------------------------------------------------------------- one pass

def run(state: Dict[str, Any]):
    kind = state["kind"]
    if kind == "block":
        return state["fn"](state["x"], state["w"], BLOCK, state["ws"], None, state["bias"])
    if kind == "ue8m0":
        return fp8_utils.deepgemm_w8a8_block_fp8_linear_with_fallback(state["x"], state["w"], BLOCK, state["ws"], None, state["bias"])
    if kind == "int8":
        return w8a8_int8.apply_w8a8_int8_linear(state["x"], state["w"], state["ws"], state["bias"])
    if kind == "token_fp8":
        return fp8_utils.apply_fp8_linear(state["x"], state["w"], state["ws"], state["input_scale"], bias=state["bias"],
                                          use_per_token_if_dynamic=True)
    if kind == "group_quant":
        layout = state["layout"]
        return fp8_kernel.sglang_per_token_group_quant_fp8(
            state["x"], 128, column_major_scales=layout != "row", scale_tma_aligned=layout in ("col_aligned", "ue8m0"),
            scale_ue8m0=layout == "ue8m0")
    if kind == "silu_quant":
        return fp8_kernel.per_token_group_quant_8bit(
            state["x"], 128, FP8, column_major_scales=True, scale_tma_aligned=True, scale_ue8m0=True, fuse_silu_and_mul=True,
            masked_m=state["masked_m"])
    s = state
    sgl_kernel.fp8_blockwise_scaled_grouped_mm(
        s["out"], *s["pointers"], s["a"], s["b"], s["sa"], s["sb"], *s["strides"], *s["layouts"], s["sizes"], s["offsets"],
        s["workspace"])
    return s["out"]


# ---------------------------------------------------------------- what a pass cannot do without

def work(case: Dict[str, Any]) -> Dict[str, float]:
    kind = case["kind"]
    if kind == "group_quant":
        values = case["M"] * case["K"]
        return {"bytes": 3 * values + values // 128 * (1 if case["layout"] == "ue8m0" else 4), "flops": 0}
    if kind == "silu_quant":
        # masked: half of the rows are in use on average; the result's unused rows are zeros that have to be written too
        values = case["E"] * case["T"] * case["H"]
        return {"bytes": values * (2 if case["masked"] else 4) + values + values // 128, "flops": 0}
    K, N = case["K"], case["N"]
    if kind == "grouped":
        rows = case["rows"]
        experts = case["E"] * (1.0 - (1.0 - 1.0 / case["E"]) ** rows)  # experts that get any row, if all are equally popular
        blocks = N // 128 * (K // 128)
        return {"bytes": experts * (N * K + 4 * blocks) + rows * (K + 4 * (K // 128) + 2 * N), "flops": 2.0 * rows * N * K}
    M = case["M"]
    scales = {"block": 4 * -(-N // 128) * -(-K // 128), "ue8m0": -(-N // 128) * -(-K // 128)}.get(kind, 4 * N)
    return {"bytes": N * K + scales + 2 * M * K + 2 * M * N + (2 * N if case["bias"] else 0), "flops": 2.0 * M * N * K}


def tolerance(case: Dict[str, Any]):
    if case["kind"] in ("group_quant", "silu_quant"):
        return "exact"  # codes and scales are defined bit for bit
    # sums in another order, rounded to the 16-bit type once, or twice where a bias is added afterwards
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3}
