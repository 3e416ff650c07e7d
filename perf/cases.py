"""Workloads of the activation path, for timing it and comparing its outputs.

``listed()`` names the calls a transformer makes of this package: the norms,
the gated FFN activations, RoPE, the FP8 quantisers and the MoE dispatch, for
one decode step, for prefill and for weights, at widths that fill 16-byte
vectors and at widths that do not. ``draw(rng)`` gives another case of the
same ranges. ``prepare`` makes a case's inputs on the GPU from a seed,
``run`` is one pass through ``custom_cuda_kernals_amd.kernels``, ``exact``
is its result in float64 by plain torch.
"""

from __future__ import annotations

import math

import torch

from custom_cuda_kernals_amd import kernels as K
from custom_cuda_kernals_amd.llama_block import CONFIGS, rope_tables

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
FP8 = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
FP8_MAX = {"e4m3": 448.0, "e5m2": 57344.0}
EPS = 1e-5
THETA = 500000.0


def listed() -> list[dict]:
    return [
        # One decode step of a Llama-3-8B layer on the FP8 path, 16 sequences:
        # every activation call between its GEMMs. Latency and launches.
        {"name": "decode_layer", "op": "layer", "model": "llama3-8b", "tokens": 16},
        # The residual stream of a Llama-3-8B prefill: the benchmark's headline.
        {"name": "norm_prefill", "op": "norm", "rows": 8192, "width": 4096, "dtype": "bf16"},
        # A hidden size that is no multiple of a 16-byte vector, as an unpadded
        # or sliced width gives; the norm feeds an FP8 GEMM, one scale a row.
        {"name": "norm_fp8_ragged", "op": "norm", "rows": 3001, "width": 4100, "dtype": "bf16", "fp8": "e4m3"},
        # The reference benchmark's named FFN shape (Llama-2-7B), fp16, unfused.
        {"name": "ffn_prefill", "op": "glu", "rows": 4096, "width": 11008, "dtype": "fp16"},
        # A Llama-3-8B FFN over a 16 K-token batch, feeding the FP8 down projection.
        {"name": "ffn_fp8_batch", "op": "glu", "rows": 16384, "width": 14336, "dtype": "bf16", "fp8": "e4m3"},
        # The 8/3 rule's FFN of hidden 2048, not rounded up: odd rows.
        {"name": "ffn_fp8_odd", "op": "glu", "rows": 2048, "width": 5461, "dtype": "bf16", "fp8": "e4m3"},
        # RoPE of a Llama-3-8B prefill.
        {"name": "rope_prefill", "op": "rope", "batch": 1, "seq": 4096, "q_heads": 32, "kv_heads": 8,
         "head_dim": 128, "dtype": "bf16"},
        # Heads of 96, whose half is six 16-byte chunks: not a power of two.
        {"name": "rope_heads96", "op": "rope", "batch": 2, "seq": 2048, "q_heads": 32, "kv_heads": 32,
         "head_dim": 96, "dtype": "fp16"},
        # A Llama-3-8B FFN weight to 128 x 128-block FP8.
        {"name": "weight_block_fp8", "op": "quant", "rows": 14336, "width": 4096, "dtype": "bf16", "fp8": "e4m3",
         "granularity": "block"},
        # An activation of 2048 tokens under one dynamic scale.
        {"name": "act_tensor_fp8", "op": "quant", "rows": 2048, "width": 4096, "dtype": "bf16", "fp8": "e4m3",
         "granularity": "tensor"},
        # The reference benchmark's DeepSeek-shaped routing: router, then the
        # expert permutation of what it picked.
        {"name": "moe_route", "op": "route", "tokens": 4096, "experts": 160, "top_k": 6, "dtype": "fp32"},
        # The rows of that dispatch: gathered by expert, combined by weight.
        {"name": "moe_move", "op": "move", "tokens": 2048, "experts": 160, "top_k": 6, "width": 4096, "dtype": "bf16"},
    ]


# Hidden and FFN widths of this repository's benchmarks and tests.
WIDTHS = [768, 1024, 2048, 2560, 3072, 4096, 5120, 7168, 8192, 11008, 14336, 18944, 28672]
MAX_ELEMENTS = 1 << 26


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng) -> int:
    """A model width, or (one in three) any length."""
    return rng.choice(WIDTHS) if rng.random() < 2 / 3 else _log_int(rng, 100, 20000)


def _rows(rng, width: int) -> int:
    return _log_int(rng, 1, max(1, min(16384, MAX_ELEMENTS // width)))


def draw(rng) -> dict:
    op = rng.choice(["layer", "norm", "norm", "glu", "glu", "rope", "quant", "quant", "route", "move"])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    if op == "layer":
        return {"op": op, "model": rng.choice(["llama3-8b", "llama3-70b"]), "tokens": _log_int(rng, 1, 256)}
    if op in ("norm", "glu"):
        width = _width(rng)
        case = {"op": op, "rows": _rows(rng, width), "width": width, "dtype": dtype}
        kind = rng.choice(["plain", "token", "token", "static"])
        if kind != "plain":
            case["fp8"] = rng.choice(["e4m3", "e4m3", "e5m2"])
        if kind == "static":
            case["static"] = 0.05
        return case
    if op == "rope":
        head_dim = rng.choice([64, 80, 96, 128, 128, 256])
        q_heads = rng.randint(4, 64)
        kv_heads = rng.randint(1, q_heads)
        tokens = _log_int(rng, 1, min(16384, MAX_ELEMENTS // ((q_heads + kv_heads) * head_dim)))
        batch = _log_int(rng, 1, min(16, tokens))
        return {"op": op, "batch": batch, "seq": max(1, tokens // batch), "q_heads": q_heads, "kv_heads": kv_heads,
                "head_dim": head_dim, "dtype": dtype}
    if op == "quant":
        width = _width(rng)
        return {"op": op, "rows": _rows(rng, width), "width": width, "dtype": dtype,
                "fp8": rng.choice(["e4m3", "e4m3", "e5m2"]), "granularity": rng.choice(["token", "block", "tensor"])}
    experts = rng.choice([8, 16, 32, 64, 128, 160, 256, rng.randint(9, 255)])
    top_k = rng.randint(1, min(8, experts))
    if op == "route":
        return {"op": op, "tokens": _log_int(rng, 1, 32768), "experts": experts, "top_k": top_k, "dtype": dtype}
    width = min(_width(rng), 8192)
    tokens = _log_int(rng, 1, max(1, min(16384, MAX_ELEMENTS // (width * top_k))))
    return {"op": op, "tokens": tokens, "experts": experts, "top_k": top_k, "width": width, "dtype": dtype}


# ---- inputs -----------------------------------------------------------------

def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _activation(g, shape, dtype) -> torch.Tensor:
    """N(0, 1) with a level of its own per row, and one channel in a thousand
    twenty times as large: a residual stream or a GEMM's output."""
    x = torch.randn(shape, generator=g, device="cuda")
    x *= torch.exp(0.3 * torch.randn((*shape[:-1], 1), generator=g, device="cuda"))
    x *= torch.where(torch.rand(shape[-1], generator=g, device="cuda") < 1e-3, 20.0, 1.0)
    return x.to(dtype)


def _randn(g, shape, dtype) -> torch.Tensor:
    return torch.randn(shape, generator=g, device="cuda").to(dtype)


def _weight(g, n, dtype) -> torch.Tensor:
    return (1.0 + 0.1 * torch.randn(n, generator=g, device="cuda")).to(dtype)


def _expert_logits(g, tokens, experts, dtype) -> torch.Tensor:
    """Router logits with some experts preferred, as trained routers have."""
    bias = 0.5 * torch.randn(experts, generator=g, device="cuda")
    return (torch.randn((tokens, experts), generator=g, device="cuda") + bias).to(dtype)


def prepare(case: dict, seed: int) -> dict:
    g, op = _gen(seed), case["op"]
    s = {"case": case}
    if op == "layer":
        cfg, t, dt = CONFIGS[case["model"]], case["tokens"], torch.bfloat16
        s["cfg"] = cfg
        s["x"], s["residual"] = _activation(g, (t, cfg.hidden_size), dt), _activation(g, (t, cfg.hidden_size), dt)
        s["w1"], s["w2"] = _weight(g, cfg.hidden_size, dt), _weight(g, cfg.hidden_size, dt)
        s["q"] = _randn(g, (t, 1, cfg.num_heads, cfg.head_dim), dt)
        s["k"] = _randn(g, (t, 1, cfg.num_kv_heads, cfg.head_dim), dt)
        # The step's position: one row of the model's tables.
        position = 1 + seed % 4095
        cos, sin = rope_tables(4096, cfg.head_dim, cfg.rope_theta, "cuda")
        s["cos"], s["sin"] = cos[position:position + 1].contiguous(), sin[position:position + 1].contiguous()
        s["attn"] = _randn(g, (t, cfg.hidden_size), dt)
        s["proj"] = _activation(g, (t, cfg.hidden_size), dt)
        s["gate"] = _randn(g, (t, cfg.intermediate_size), dt)
        s["up"] = _randn(g, (t, cfg.intermediate_size), dt)
        return s
    dt = DTYPES[case["dtype"]]
    if op == "norm":
        shape = (case["rows"], case["width"])
        s["x"], s["residual"], s["w"] = _activation(g, shape, dt), _activation(g, shape, dt), _weight(g, shape[1], dt)
    elif op == "glu":
        shape = (case["rows"], case["width"])
        s["gate"], s["up"] = _randn(g, shape, dt), _randn(g, shape, dt)
    elif op == "rope":
        b, n, d = case["batch"], case["seq"], case["head_dim"]
        s["q"], s["k"] = _randn(g, (b, n, case["q_heads"], d), dt), _randn(g, (b, n, case["kv_heads"], d), dt)
        s["cos"], s["sin"] = rope_tables(n, d, THETA, "cuda")
    elif op == "quant":
        s["x"] = _activation(g, (case["rows"], case["width"]), dt)
    elif op == "route":
        s["logits"] = _expert_logits(g, case["tokens"], case["experts"], dt)
    else:
        t, k = case["tokens"], case["top_k"]
        w, ids = torch.topk(torch.softmax(_expert_logits(g, t, case["experts"], torch.float32), -1), k)
        order = torch.argsort(ids.reshape(-1), stable=True)
        s["permute"] = order // k
        s["unpermute"] = torch.empty_like(order).scatter_(0, order, torch.arange(t * k, device="cuda")).view(t, k)
        s["w"] = (w / w.sum(-1, keepdim=True)).contiguous()
        s["tokens"] = _activation(g, (t, case["width"]), dt)
        s["expert_out"] = _randn(g, (t * k, case["width"]), dt)
    return s


# ---- one pass ---------------------------------------------------------------

def run(s: dict):
    case = s["case"]
    op, fp8, static = case["op"], case.get("fp8"), case.get("static")
    if op == "layer":
        h, hs, residual = K.rmsnorm_residual_fp8(s["x"], s["residual"], s["w1"], EPS)
        q, k = K.rope(s["q"], s["k"], s["cos"], s["sin"])
        a, a_s = K.fp8_quant(s["attn"], "e4m3", "token")
        h2, h2s, residual2 = K.rmsnorm_residual_fp8(s["proj"], residual, s["w2"], EPS)
        m, ms = K.swiglu_fp8(s["gate"], s["up"])
        return h, hs, residual, q, k, a, a_s, h2, h2s, residual2, m, ms
    if op == "norm":
        if fp8:
            return K.rmsnorm_residual_fp8(s["x"], s["residual"], s["w"], EPS, fp8, static)
        return K.rmsnorm_residual(s["x"], s["residual"], s["w"], EPS)
    if op == "glu":
        return K.swiglu_fp8(s["gate"], s["up"], fp8, static) if fp8 else K.swiglu(s["gate"], s["up"])
    if op == "rope":
        return K.rope(s["q"], s["k"], s["cos"], s["sin"])
    if op == "quant":
        return K.fp8_quant(s["x"], fp8, case["granularity"])
    if op == "route":
        weights, ids = K.moe_router(s["logits"], case["top_k"])
        permute, unpermute = K.compute_permutation(ids, case["experts"])
        return weights, ids, permute, unpermute
    return K.token_gather(s["tokens"], s["permute"]), K.token_combine(s["expert_out"], s["unpermute"], s["w"])


# ---- what a pass cannot do without -------------------------------------------

def work(case: dict) -> dict:
    op, fp8 = case["op"], case.get("fp8")
    es = DTYPES[case.get("dtype", "bf16")].itemsize
    if op == "layer":
        cfg, t = CONFIGS[case["model"]], case["tokens"]
        h, i, d = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim
        # Two norms (two rows read, one row and its codes written), RoPE,
        # the attention output's codes, the FFN's codes.
        b = 2 * (t * h * 7 + 2 * h + 4 * t) + t * (cfg.num_heads + cfg.num_kv_heads) * d * 4 + 4 * d
        b += t * h * 3 + 4 * t + t * i * 5 + 4 * t
        return {"bytes": b, "flops": t * (16 * h + 3 * (cfg.num_heads + cfg.num_kv_heads) * d + 2 * h + 8 * i)}
    if op in ("norm", "glu"):
        r, w = case["rows"], case["width"]
        out = r * w + (4 if case.get("static") else 4 * r) if fp8 else r * w * es
        if op == "norm":
            return {"bytes": 3 * r * w * es + w * es + out, "flops": 6 * r * w + (2 * r * w if fp8 else 0)}
        return {"bytes": 2 * r * w * es + out, "flops": 6 * r * w + (2 * r * w if fp8 else 0)}
    if op == "rope":
        n = case["batch"] * case["seq"] * (case["q_heads"] + case["kv_heads"]) * case["head_dim"]
        return {"bytes": 2 * n * es + case["seq"] * case["head_dim"] * 4, "flops": 3 * n}
    if op == "quant":
        r, w = case["rows"], case["width"]
        scales = {"token": r, "block": -(-r // 128) * -(-w // 128), "tensor": 1}[case["granularity"]]
        return {"bytes": r * w * (es + 1) + 4 * scales, "flops": 2 * r * w}
    t, k = case["tokens"], case["top_k"]
    if op == "route":
        # Logits in; weights, ids, and both permutation indices out.
        return {"bytes": t * case["experts"] * es + t * k * (4 + 8 + 8 + 8), "flops": 8 * t * case["experts"]}
    h = case["width"]
    gather = t * h * es + t * k * h * es + 8 * t * k
    combine = t * k * h * es + t * h * es + 12 * t * k
    return {"bytes": gather + combine, "flops": 2 * t * k * h}


def tolerance(case: dict):
    """Outputs are rounded once or twice to their type, and a code that lands
    on the other side of a tie is one step of its format away (1/8 of the
    value in e4m3, 1/4 in e5m2)."""
    op, dtype = case["op"], case.get("dtype", "bf16")
    fp8 = "e4m3" if op == "layer" else case.get("fp8")
    if fp8:
        step = 0.13 if fp8 == "e4m3" else 0.26
        # Codes of inputs taken as they are flip only where two quotients
        # round apart; codes of a fused result also where the result does.
        fused = {"bf16": 3e-2, "fp16": 2.5e-2, "fp32": 2e-3}[dtype]
        return {"rel": 2.5e-3 if op == "quant" else fused, "max": step}
    if op == "route":
        return {"rel": 2e-6, "max": 2e-5, "differ": 1e-3}
    rel = {"bf16": 1.2e-2, "fp16": 1.2e-3, "fp32": 2e-6}[dtype]
    return {"rel": rel, "max": 10 * rel}


# ---- the same in float64 -----------------------------------------------------

def _codes(y: torch.Tensor, scale, fp8: str) -> torch.Tensor:
    return (y / scale).to(FP8[fp8]).double()


def _scale(amax: torch.Tensor, fp8: str) -> torch.Tensor:
    return (amax / FP8_MAX[fp8]).clamp(min=1e-12)


def _token_fp8(y: torch.Tensor, fp8: str):
    s = _scale(y.abs().amax(-1, keepdim=True), fp8)
    return _codes(y, s, fp8), s.squeeze(-1)


def _norm64(x, residual, w):
    ro = x.double() + residual.double()
    return ro * torch.rsqrt(ro.square().mean(-1, keepdim=True) + EPS) * w.double(), ro


def _glu64(gate, up):
    g = gate.double()
    return g * torch.sigmoid(g) * up.double()


def _rope64(x, cos, sin):
    c, n = cos.double()[None, :, None, :], sin.double()[None, :, None, :]
    a, b = x.double().chunk(2, -1)
    return torch.cat([a * c - b * n, b * c + a * n], -1)


def exact(case: dict, seed: int):
    s = prepare(case, seed)
    op, fp8, static = case["op"], case.get("fp8"), case.get("static")
    if op == "layer":
        y, ro = _norm64(s["x"], s["residual"], s["w1"])
        # The second norm's residual is the first one's output, stored in bf16.
        y2, ro2 = _norm64(s["proj"], ro.to(torch.bfloat16), s["w2"])
        q, k = _rope64(s["q"], s["cos"], s["sin"]), _rope64(s["k"], s["cos"], s["sin"])
        return (*_token_fp8(y, "e4m3"), ro, q, k, *_token_fp8(s["attn"].double(), "e4m3"),
                *_token_fp8(y2, "e4m3"), ro2, *_token_fp8(_glu64(s["gate"], s["up"]), "e4m3"))
    if op in ("norm", "glu"):
        if op == "norm":
            y, ro = _norm64(s["x"], s["residual"], s["w"])
        else:
            y, ro = _glu64(s["gate"], s["up"]), None
        if fp8:
            sc = torch.full((1,), float(static), dtype=torch.float64, device="cuda") if static else None
            y, sc = (_codes(y, sc, fp8), sc) if static else _token_fp8(y, fp8)
            return (y, sc, ro) if op == "norm" else (y, sc)
        return (y, ro) if op == "norm" else y
    if op == "rope":
        return _rope64(s["q"], s["cos"], s["sin"]), _rope64(s["k"], s["cos"], s["sin"])
    if op == "quant":
        x = s["x"].double()
        if case["granularity"] == "token":
            return _token_fp8(x, fp8)
        if case["granularity"] == "tensor":
            sc = _scale(x.abs().amax().reshape(1), fp8)
            return _codes(x, sc, fp8), sc
        m, n = x.shape
        mb, nb = -(-m // 128), -(-n // 128)
        padded = torch.zeros(mb * 128, nb * 128, dtype=torch.float64, device="cuda")
        padded[:m, :n] = x
        tiles = padded.view(mb, 128, nb, 128)
        sc = _scale(tiles.abs().amax((1, 3)), fp8)
        return _codes((tiles / sc[:, None, :, None]).view(mb * 128, nb * 128)[:m, :n], 1.0, fp8), sc
    if op == "route":
        p = torch.softmax(s["logits"].double(), -1)
        # Equal probabilities: the lower expert first.
        w, ids = (v[:, :case["top_k"]] for v in torch.sort(p, dim=-1, descending=True, stable=True))
        order = torch.argsort(ids.reshape(-1), stable=True)
        unpermute = torch.empty_like(order).scatter_(0, order, torch.arange(order.numel(), device="cuda"))
        return w / w.sum(-1, keepdim=True), ids, order // case["top_k"], unpermute.view(ids.shape)
    combined = (s["expert_out"].double()[s["unpermute"]] * s["w"].double()[..., None]).sum(1)
    return s["tokens"][s["permute"]].double(), combined
