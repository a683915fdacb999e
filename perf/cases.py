"""The work a user has this package do, as cases that can be timed: paged-attention decode, the FFN
block and the decoder-layer decode step, each called through a registered program of a ``ChipWorker``
on device-resident tensors, the way a serving loop calls them.

``listed()`` holds named cases over the range in use - one interactive sequence, a serving batch, long
contexts, short and long prompts; 16-bit, int8 and e4m3 operands; ragged lengths and token counts that
are no multiple of any tile.  ``draw(rng)`` gives further cases of the same ranges.  A case is a plain
dict; ``prepare`` builds its inputs from a seed, ``run`` is one call of the program.
"""

from __future__ import annotations

import random

import torch

from pypto_amd import runtime, workloads
from pypto_amd.runtime import ChipWorker, RunConfig

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}

# What a serving process keeps: one worker, and each program registered once.
_worker: ChipWorker | None = None
_handles: dict = {}


def _handle(program):
    global _worker
    if _worker is None:
        _worker = ChipWorker(RunConfig(platform="mi355x", device_id=0))
    if id(program) not in _handles:
        _handles[id(program)] = _worker.register(program)
    return _handles[id(program)]


def listed() -> list[dict]:
    return [
        # one user waiting for the next token: launches and latency are all of it
        {"name": "attention_one_sequence", "kind": "attention", "batch": 1, "heads": 32, "kv_heads": 8, "head_dim": 128,
         "block": 128, "ctx_lo": 1531, "ctx_hi": 1531, "dtype": "bf16", "kv": "same"},
        # a small serving batch of ragged chats (bench.py's attention configuration)
        {"name": "attention_batch16", "kind": "attention", "batch": 16, "heads": 32, "kv_heads": 8, "head_dim": 128,
         "block": 128, "ctx_lo": 512, "ctx_hi": 4096, "dtype": "bf16", "kv": "same"},
        # long documents over a quantised cache (bench.py's long configuration)
        {"name": "attention_long_e4m3", "kind": "attention", "batch": 64, "heads": 64, "kv_heads": 8, "head_dim": 128,
         "block": 128, "ctx_lo": 8192, "ctx_hi": 32768, "dtype": "bf16", "kv": "e4m3"},
        # all query heads on one KV head, wide heads, small blocks (the attention system tests' widest shape)
        {"name": "attention_one_kv_head_d256", "kind": "attention", "batch": 64, "heads": 64, "kv_heads": 1,
         "head_dim": 256, "block": 64, "ctx_lo": 8192, "ctx_hi": 8192, "dtype": "bf16", "kv": "same"},
        # the FFN example's fp16 tile program: a small model, a small call
        {"name": "ffn_small_model", "kind": "ffn", "tokens": 128, "hidden": 512, "inter": 1024, "dtype": "fp16",
         "norm": False, "out": "fp32", "weights": "w16"},
        # the rest of a chunked prompt riding with a decode batch: some hundred tokens, no multiple of a tile
        {"name": "ffn_mixed_batch_333", "kind": "ffn", "tokens": 333, "hidden": 4096, "inter": 14336, "dtype": "fp16",
         "norm": True, "out": "same", "weights": "w16"},
        # prefill of a prompt (bench.py's FFN configuration)
        {"name": "ffn_prefill_2048", "kind": "ffn", "tokens": 2048, "hidden": 4096, "inter": 11008, "dtype": "bf16",
         "norm": True, "out": "fp32", "weights": "w16"},
        # the same prefill on e4m3 operands
        {"name": "ffn_prefill_2048_e4m3", "kind": "ffn", "tokens": 2048, "hidden": 4096, "inter": 11008, "dtype": "bf16",
         "norm": True, "out": "fp32", "weights": "e4m3"},
        # one layer of a decode step for one user, int8 weights
        {"name": "layer_one_sequence", "kind": "layer", "batch": 1, "hidden": 4096, "heads": 32, "kv_heads": 8,
         "inter": 14336, "block": 128, "ctx_lo": 2049, "ctx_hi": 2049, "dtype": "bf16", "weights": "int8", "kv": "same"},
        # one layer of a full decode batch, int8 weights (bench.py's layer configuration)
        {"name": "layer_batch32_int8", "kind": "layer", "batch": 32, "hidden": 4096, "heads": 32, "kv_heads": 8,
         "inter": 14336, "block": 128, "ctx_lo": 4096, "ctx_hi": 4096, "dtype": "bf16", "weights": "int8", "kv": "same"},
        # one layer of a larger model with the 16-bit weights the reference has, ragged lengths
        {"name": "layer_batch16_w16", "kind": "layer", "batch": 16, "hidden": 5120, "heads": 40, "kv_heads": 8,
         "inter": 17408, "block": 128, "ctx_lo": 700, "ctx_hi": 4096, "dtype": "bf16", "weights": "w16", "kv": "same"},
        # a throughput batch beyond the skinny projections' 32 rows, every operand quantised
        {"name": "layer_batch96_int8_e4m3", "kind": "layer", "batch": 96, "hidden": 4096, "heads": 32, "kv_heads": 8,
         "inter": 14336, "block": 64, "ctx_lo": 200, "ctx_hi": 3000, "dtype": "fp16", "weights": "int8", "kv": "e4m3"},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    """Spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def _lengths(rng: random.Random, longest: int) -> tuple[int, int]:
    """Context range of a batch: all alike, or ragged down to a tenth of the longest."""
    hi = _log_int(rng, 64, longest)
    return (hi, hi) if rng.random() < 0.25 else (max(1, int(hi * rng.uniform(0.1, 1.0))), hi)


def draw(rng: random.Random) -> dict:
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(("attention", "ffn", "layer"))
        dtype = rng.choice(("bf16", "bf16", "fp16"))
        if kind == "attention":
            kv_heads = rng.choice((1, 2, 4, 8))
            lo, hi = _lengths(rng, 32768)
            case = {"kind": kind, "batch": _log_int(rng, 1, 256), "heads": kv_heads * rng.choice((1, 2, 4, 5, 7, 8, 16)),
                    "kv_heads": kv_heads, "head_dim": rng.choice((128, 128, 128, 256)), "block": rng.choice((32, 64, 128, 256)),
                    "ctx_lo": lo, "ctx_hi": hi, "dtype": dtype, "kv": rng.choice(("same", "same", "e4m3"))}
        elif kind == "ffn":
            e4m3 = rng.random() < 0.25
            step = 128 if e4m3 else rng.choice((8, 64, 128, 256))
            hidden = max(step, _log_int(rng, 512, 8192) // step * step)
            inter = max(step, int(hidden * rng.uniform(2.0, 4.0)) // step * step)
            if e4m3 and inter > 16384:  # the row quantisers' limit
                continue
            case = {"kind": kind, "tokens": _log_int(rng, 1, 4096), "hidden": hidden, "inter": inter, "dtype": dtype,
                    "norm": e4m3 or rng.random() < 0.75, "out": rng.choice(("fp32", "same")),
                    "weights": "e4m3" if e4m3 else "w16"}
        else:
            kv_heads = rng.choice((1, 2, 4, 8))
            hidden = _log_int(rng, 1024, 8192) // 64 * 64
            lo, hi = _lengths(rng, 16384)
            case = {"kind": kind, "batch": _log_int(rng, 1, 160), "hidden": hidden,
                    "heads": kv_heads * rng.choice((1, 2, 4, 5, 7, 8)), "kv_heads": kv_heads,
                    "inter": int(hidden * rng.uniform(2.0, 4.0)) // 64 * 64, "block": rng.choice((64, 128, 256)),
                    "ctx_lo": lo, "ctx_hi": hi, "dtype": dtype, "weights": rng.choice(("int8", "w16")),
                    "kv": rng.choice(("same", "same", "e4m3"))}
        if _cost(case) <= most and work(case)["bytes"] <= 2.8e9:
            return case


def _cost(case: dict) -> float:
    w = work(case)
    return w["bytes"] / 8e12 + w["flops"] / 2.5e15


def _spread(case: dict, seed: int) -> list[int]:
    """One length per sequence: spread evenly over [ctx_lo, ctx_hi], dealt out in an order of the seed's -
    the sum, and with it the work and the size of the pool, is the same for every seed."""
    lo, hi, n = case["ctx_lo"], case["ctx_hi"], case["batch"]
    lens = [lo + round((hi - lo) * (i + 0.5) / n) for i in range(n)]
    random.Random(seed).shuffle(lens)
    return lens


def _quantised(cache: torch.Tensor, kv_heads: int, block: int) -> tuple[torch.Tensor, torch.Tensor]:
    """e4m3 codes and one fp32 scale per (block, KV head) of a 16-bit cache [pool * kv_heads * block, D]."""
    x = cache.float().reshape(-1, block * cache.shape[1])
    scale = x.abs().amax(dim=1).clamp_min(1e-12) / workloads.FP8_E4M3_MAX
    codes = (x / scale[:, None]).to(torch.float8_e4m3fn).reshape(cache.shape)
    return codes, scale.reshape(-1, kv_heads).contiguous()


def prepare(case: dict, seed: int) -> dict:
    dtype = _DTYPES[case["dtype"]]
    if case["kind"] == "attention":
        a = workloads.paged_attention_inputs(
            batch=case["batch"], num_heads=case["heads"], kv_head_num=case["kv_heads"], head_dim=case["head_dim"],
            block_size=case["block"], ctx_range=(case["ctx_lo"], case["ctx_hi"]), context_lens=_spread(case, seed),
            dtype=dtype, fp8_kv=case["kv"] == "e4m3", seed=seed, device="cuda")
        return {"handle": _handle(runtime.paged_attention), "args": a.args(), "outputs": (a.out,)}
    if case["kind"] == "ffn":
        out_dtype = torch.float32 if case["out"] == "fp32" else dtype
        shape = dict(tokens=case["tokens"], hidden=case["hidden"], intermediate=case["inter"], dtype=dtype,
                     out_dtype=out_dtype, seed=seed, device="cuda")
        if case["weights"] == "e4m3":
            q, _ = workloads.ffn_fp8_inputs(**shape)
            return {"handle": _handle(runtime.ffn_block_fp8), "args": q.args(), "outputs": (q.out,)}
        f = workloads.ffn_inputs(with_norm=case["norm"], **shape)
        if case["norm"]:
            return {"handle": _handle(runtime.ffn_block),
                    "args": (f.x, f.gamma, f.w_gate, f.w_up, f.w_down, f.out, f.eps), "outputs": (f.out,)}
        return {"handle": _handle(runtime.ffn_swiglu), "args": (f.x, f.w_gate, f.w_up, f.w_down, f.out),
                "outputs": (f.out,)}
    d = workloads.decoder_layer_inputs(
        batch=case["batch"], hidden=case["hidden"], num_heads=case["heads"], kv_head_num=case["kv_heads"],
        intermediate=case["inter"], block_size=case["block"], context_lens=_spread(case, seed), dtype=dtype, seed=seed,
        device="cuda", int8_weights=case["weights"] == "int8", weight_std=None)
    args = d.args()
    if case["kv"] == "e4m3":
        kc, ks = _quantised(d.key_cache, case["kv_heads"], case["block"])
        vc, vs = _quantised(d.value_cache, case["kv_heads"], case["block"])
        program = runtime.decoder_layer_decode_fp8kv if case["weights"] == "int8" else runtime.decoder_layer_decode_w16_fp8kv
        return {"handle": _handle(program), "args": args[:3] + (kc, vc, ks, vs) + args[5:],
                "outputs": (d.out, kc, vc, ks, vs)}
    program = runtime.decoder_layer_decode if case["weights"] == "int8" else runtime.decoder_layer_decode_w16
    return {"handle": _handle(program), "args": args, "outputs": (d.out, d.key_cache, d.value_cache)}


def run(state: dict) -> tuple:
    state["handle"](*state["args"])
    return state["outputs"]


def work(case: dict) -> dict:
    if case["kind"] == "ffn":
        t, h, i = case["tokens"], case["hidden"], case["inter"]
        wbytes = 3 * h * i * (1 if case["weights"] == "e4m3" else 2)
        return {"bytes": wbytes + t * h * (2 + (4 if case["out"] == "fp32" else 2)), "flops": 6 * t * h * i}
    b, hq, hkv = case["batch"], case["heads"], case["kv_heads"]
    tokens = b * (case["ctx_lo"] + case["ctx_hi"]) / 2  # cache rows attended to, summed over the batch
    d = case.get("head_dim", 128)
    kv = tokens * hkv * d * 2 * (1 if case["kv"] == "e4m3" else 2)
    attention = 4 * tokens * hq * d
    if case["kind"] == "attention":
        return {"bytes": kv + b * hq * d * (2 + 4), "flops": attention}
    h, i = case["hidden"], case["inter"]
    n_weights = h * (hq + 2 * hkv) * d + hq * d * h + 3 * h * i
    return {"bytes": kv + n_weights * (1 if case["weights"] == "int8" else 2) + 4 * b * h,
            "flops": attention + 2 * b * n_weights}


def tolerance(case: dict) -> dict:
    """About four times the distance measured between the path and the same mathematics in 64 bits.
    bf16: attention 1.3e-3 to 1.6e-3 (probabilities rounded before PV), layer 1.8e-3 to 2.2e-3, FFN 2.9e-3
    to 3.4e-3 (2.8e-4 at the same rounding points); fp16: attention 1.8e-4, layer 2.5e-4, FFN 4.2e-4.  The
    e4m3 FFN at the same rounding points: 1.4e-3 in norm and 0.10 in a single value, since a value of h that
    moves by an ulp takes another code; an appended e4m3 cache row: 0.06 in a single value, one code."""
    bf16 = case["dtype"] == "bf16"
    if case["kind"] == "ffn":
        return {"rel": 6e-3, "max": 0.4} if case["weights"] == "e4m3" else {"rel": 1.2e-2 if bf16 else 1.7e-3}
    if case["kind"] == "attention":
        return {"rel": 6e-3 if bf16 else 1e-3}
    return {"rel": 8e-3 if bf16 else 1e-3, "max": 0.25 if case["kv"] == "e4m3" else 0.3 if bf16 else 0.04}
