"""The workloads this framework's speed is measured on.

Every case is one call (or one short greedy decode) through ``HipDecodeBackend``, the
decoders or the load-time quantizers, on inputs made from a seed alone.  The listed
cases span the framework's use: one projection of a single token, the batched
projections and the lm_head of several sequences decoded together, decode attention at
ordinary and long contexts, the MoE experts, weight packing at load time, and whole
decode steps of the two benchmark models.  ``draw`` gives more cases of the same kinds
over the ranges those stand for.

``exact`` restates each operator in float64 with plain torch.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from thintensor_amd.backend import HipDecodeBackend
from thintensor_amd.decode import DenseDecoder, MoEBatchDecoder
from thintensor_amd.quantize import quantize_to_int4_cpu
from thintensor_amd.synth import DenseShape, MoEShape, make_dense, make_moe

_DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def listed() -> list[dict]:
    return [
        # the MLP up-projection of one token of a 1B model: the smallest call of a decode step
        {"name": "int4-gemv", "kind": "int4-gemv", "rows": 8192, "cols": 2048, "dtype": "f16"},
        # a 14B model's fp8 gate and up projections of one token with the SiLU product
        {"name": "fp8-gate-up", "kind": "fp8-gate-up", "rows": 17920, "cols": 5120, "dtype": "bf16"},
        # a 14B model's int4 MLP projection for 64 sequences decoded together
        {"name": "int4-gemm-m64", "kind": "int4-gemm", "m": 64, "rows": 17920, "cols": 5120},
        # the fp8 form of that projection for a small batch
        {"name": "fp8-gemm-m8", "kind": "fp8-gemm", "m": 8, "rows": 17920, "cols": 5120},
        # a square fp8 attention projection for an odd number of sequences
        {"name": "fp8-gemm-m33", "kind": "fp8-gemm", "m": 33, "rows": 5120, "cols": 5120},
        # the greedy lm_head of 16 sequences over a large vocabulary
        {"name": "lm-head-m16", "kind": "lm-head", "m": 16, "rows": 152064, "cols": 5120},
        # decode attention of a 14B model (40 query heads on 10 KV heads of dim 128), part-filled cache
        {"name": "attention-d128", "kind": "attention", "heads": 40, "kv_heads": 10, "head_dim": 128, "tokens": 4001,
         "capacity": 4096, "dtype": "bf16", "sinks": False},
        # decode attention with sinks at a long context, gpt-oss heads
        {"name": "attention-16k", "kind": "attention", "heads": 64, "kv_heads": 8, "head_dim": 64, "tokens": 16385,
         "capacity": 20480, "dtype": "f16", "sinks": True},
        # one gpt-oss MoE layer's experts for eight sequences decoded together
        {"name": "experts-8", "kind": "experts", "tokens": 8, "hidden": 2880, "inter": 2880, "experts": 32, "top_k": 4},
        # packing one 14B MLP projection to int4 at load time
        {"name": "quantize-int4", "kind": "quantize-int4", "rows": 17920, "cols": 5120, "group": 128, "dtype": "bf16"},
        # greedy decode of the 1B benchmark model, one sequence, graph replay
        {"name": "dense-decode", "kind": "dense-decode", "layers": 16, "prior": 512, "steps": 8},
        # greedy decode of the 20B MoE benchmark model, eight sequences in lockstep, graph replay
        {"name": "moe-decode-8", "kind": "moe-decode", "layers": 24, "batch": 8, "prior": 1024, "steps": 4},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _steps_of(rng, lo: int, hi: int, step: int) -> int:
    return step * rng.randint(-(-lo // step), hi // step)


def draw(rng) -> dict:
    kind = rng.choice(["int4-gemv", "fp8-gate-up", "int4-gemm", "int4-gemm", "fp8-gemm", "fp8-gemm", "lm-head",
                       "lm-head", "attention", "attention", "attention", "experts", "experts", "quantize-int4",
                       "dense-decode", "moe-decode"])
    if kind == "int4-gemv":
        return {"kind": kind, "rows": _log_int(rng, 512, 17920), "cols": _steps_of(rng, 1024, 8192, 128),
                "dtype": rng.choice(["f16", "bf16"])}
    if kind == "fp8-gate-up":
        return {"kind": kind, "rows": _log_int(rng, 2048, 17920), "cols": _steps_of(rng, 1024, 8192, 32),
                "dtype": rng.choice(["f16", "bf16"])}
    if kind in ("int4-gemm", "fp8-gemm"):
        return {"kind": kind, "m": _log_int(rng, 2, 64), "rows": _log_int(rng, 1000, 20000),
                "cols": _steps_of(rng, 1024, 8192, 256)}
    if kind == "lm-head":
        return {"kind": kind, "m": _log_int(rng, 2, 64), "rows": _log_int(rng, 20000, 152064),
                "cols": _steps_of(rng, 2048, 5120, 32)}
    if kind == "attention":
        tokens = _log_int(rng, 16, 32768)
        capacity = tokens + rng.randint(0, tokens // 2)
        if rng.random() < 0.75:      # most caches are allocated in whole pages
            capacity = -(-capacity // 64) * 64
        kv_heads = rng.choice([2, 4, 8, 10])
        return {"kind": kind, "heads": kv_heads * rng.choice([1, 4, 8]), "kv_heads": kv_heads,
                "head_dim": rng.choice([64, 128]), "tokens": tokens, "capacity": capacity,
                "dtype": rng.choice(["f16", "bf16"]), "sinks": rng.random() < 0.4}
    if kind == "experts":
        return {"kind": kind, "tokens": _log_int(rng, 1, 32), "hidden": _steps_of(rng, 1024, 2880, 32),
                "inter": _steps_of(rng, 1024, 2880, 32), "experts": rng.choice([8, 16, 32]), "top_k": 4}
    if kind == "quantize-int4":
        group = rng.choice([32, 64, 128])
        return {"kind": kind, "rows": _log_int(rng, 512, 17920), "cols": _steps_of(rng, 1024, 8192, 128),
                "group": group, "dtype": rng.choice(["f16", "bf16", "f32"])}
    if kind == "dense-decode":
        return {"kind": kind, "layers": rng.randint(2, 16), "prior": _log_int(rng, 1, 4096), "steps": rng.randint(2, 8)}
    return {"kind": kind, "layers": rng.randint(2, 16), "batch": rng.randint(1, 8), "prior": _log_int(rng, 1, 2048),
            "steps": rng.randint(1, 4)}


# ------------------------------------------------------------------------------- inputs
def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, shape, std, dtype):
    return torch.randn(shape, generator=g, device="cuda").mul_(std).to(dtype)


def _backend(dtype) -> HipDecodeBackend:
    return HipDecodeBackend(torch.device("cuda:0"), dtype, 2048, 2048, 512, 8192)


def _int4(g, rows, cols):
    """int4 codes uniform over 0 .. 15 (value c - 8) and fp16 scales |N(0, 1)| * 0.02, group 128"""
    packed = torch.randint(0, 256, (rows, cols // 2), generator=g, device="cuda", dtype=torch.uint8)
    return packed, _normal(g, (rows, cols // 128), 0.02, torch.float32).abs_().to(torch.float16)


def _fp8(g, rows, cols):
    """fp8 rows as a quantizer leaves them (normal weights, row maximum at 448) and fp32 row scales"""
    weight = torch.empty((rows, cols), device="cuda", dtype=torch.float8_e4m3fn)
    for r in range(0, rows, 4096):
        weight[r:r + 4096] = _normal(g, (min(4096, rows - r), cols), 110.0, torch.float32).clamp_(-448, 448) \
            .to(torch.float8_e4m3fn)
    return weight, _normal(g, (rows,), 2e-5, torch.float32).abs_().add_(1e-4)


def _inputs(case: dict, seed: int) -> dict:
    g, kind = _gen(seed), case["kind"]
    if kind == "int4-gemv":
        w, s = _int4(g, case["rows"], case["cols"])
        return {"w": w, "s": s, "x": _normal(g, case["cols"], 1.0, _DTYPES[case["dtype"]])}
    if kind == "fp8-gate-up":
        gate, up = (_fp8(g, case["rows"], case["cols"]) for _ in range(2))
        return {"gate": gate, "up": up, "x": _normal(g, case["cols"], 1.0, _DTYPES[case["dtype"]])}
    if kind in ("int4-gemm", "fp8-gemm"):
        w, s = (_int4 if kind == "int4-gemm" else _fp8)(g, case["rows"], case["cols"])
        return {"w": w, "s": s, "x": _normal(g, (case["m"], case["cols"]), 1.0, torch.float16)}
    if kind == "lm-head":
        return {"w": _normal(g, (case["rows"], case["cols"]), 0.02, torch.float16),
                "x": _normal(g, (case["m"], case["cols"]), 1.0, torch.float16)}
    if kind == "attention":
        dt, shape = _DTYPES[case["dtype"]], (case["kv_heads"], case["capacity"], case["head_dim"])
        return {"q": _normal(g, case["heads"] * case["head_dim"], 1.0, dt), "k": _normal(g, shape, 1.0, dt),
                "v": _normal(g, shape, 1.0, dt),
                "sinks": _normal(g, case["heads"], 1.0, dt) if case["sinks"] else None,
                "count": torch.tensor([case["tokens"]], device="cuda", dtype=torch.int32)}
    if kind == "experts":
        E, H, I, T, k = (case[n] for n in ("experts", "hidden", "inter", "tokens", "top_k"))

        def mxfp4(rows, cols):
            return (torch.randint(0, 256, (E, rows, cols // 32, 16), generator=g, device="cuda", dtype=torch.uint8),
                    torch.randint(119, 124, (E, rows, cols // 32), generator=g, device="cuda", dtype=torch.uint8))

        # router logits of independent tokens: slots of different tokens share experts
        top = _normal(g, (T, E), 1.0, torch.float32).topk(k, dim=1)
        return {"gate_up": mxfp4(2 * I, H), "down": mxfp4(H, I), "x": _normal(g, (T, H), 1.0, torch.float16),
                "gate_up_bias": _normal(g, (E, 2 * I), 0.02, torch.float16),
                "down_bias": _normal(g, (E, H), 0.02, torch.float16),
                "idx": top.indices.to(torch.int32).contiguous(),
                "scores": top.values.softmax(dim=1).to(torch.float16).contiguous()}
    if kind == "quantize-int4":
        return {"w": _normal(g, (case["rows"], case["cols"]), 0.02, _DTYPES[case["dtype"]])}
    raise ValueError(kind)


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "dense-decode":
        shape = DenseShape(name="dense", layers=case["layers"], prior_tokens=case["prior"], max_new_tokens=case["steps"])
        w = make_dense(shape, device="cuda", seed=seed, centered_codes=True)
        be = HipDecodeBackend(torch.device("cuda:0"), torch.float16, shape.hidden, shape.q_dim, shape.kv_dim,
                              shape.intermediate)
        dec = DenseDecoder(be, w, fused=True)
        dec.capture()
        return {"case": case, "dec": dec, "logits": be.logits_buffer(shape.vocab, torch.float16),
                "start": 1 + seed % 1000}
    if kind == "moe-decode":
        shape = MoEShape(name="moe", layers=case["layers"], prior_tokens=case["prior"], max_new_tokens=case["steps"])
        w = make_moe(shape, device="cuda", seed=seed)
        be = HipDecodeBackend(torch.device("cuda:0"), torch.float16, shape.hidden, shape.q_dim, shape.kv_dim,
                              shape.intermediate)
        B = case["batch"]
        # every sequence its own cache: the model's prior tokens, rotated by the sequence
        k, v = (torch.cat([c.roll(b, dims=1) for b in range(B)], dim=1).contiguous() for c in (w.k_cache, w.v_cache))
        dec = MoEBatchDecoder(be, w, B, k, v)
        dec.capture()
        return {"case": case, "dec": dec, "be": be, "start": [1 + (seed + 37 * b) % 1000 for b in range(B)],
                "logits": torch.empty((B, shape.vocab), device="cuda", dtype=torch.float16),
                "best": torch.empty(B, device="cuda", dtype=torch.int64)}
    s = _inputs(case, seed)
    s["case"] = case
    if kind == "int4-gemv":
        s["be"] = _backend(_DTYPES[case["dtype"]])
        s["out"] = torch.empty(case["rows"], device="cuda", dtype=_DTYPES[case["dtype"]])
    elif kind == "fp8-gate-up":
        s["be"] = _backend(_DTYPES[case["dtype"]])
        s["out"] = torch.empty(case["rows"], device="cuda", dtype=_DTYPES[case["dtype"]])
    elif kind in ("int4-gemm", "fp8-gemm"):
        s["be"] = _backend(torch.float16)
        s["out"] = torch.empty((case["m"], case["rows"]), device="cuda", dtype=torch.float16)
    elif kind == "lm-head":
        s["be"] = _backend(torch.float16)
        s["logits"] = torch.empty((case["m"], case["rows"]), device="cuda", dtype=torch.float16)
        s["tokens"] = torch.empty(case["m"], device="cuda", dtype=torch.int64)
    elif kind == "attention":
        s["be"] = _backend(_DTYPES[case["dtype"]])
        s["out"] = torch.empty(case["heads"] * case["head_dim"], device="cuda", dtype=_DTYPES[case["dtype"]])
    elif kind == "experts":
        s["be"] = _backend(torch.float16)
        s["act"] = torch.empty((case["tokens"] * case["top_k"], case["inter"]), device="cuda", dtype=torch.float16)
        s["out"] = torch.empty((case["tokens"], case["hidden"]), device="cuda", dtype=torch.float16)
    return s


# ------------------------------------------------------------------------------- one pass
_ALPHA, _LIMIT = 1.702, 7.0   # gpt-oss SwiGLU


def run(s: dict):
    case = s["case"]
    kind = case["kind"]
    if kind == "int4-gemv":
        return s["be"].int4_scaled_matvec(s["w"], s["s"], s["x"], s["out"], rows=case["rows"], cols=case["cols"],
                                          group_size=128)
    if kind == "fp8-gate-up":
        return s["be"].fused_scaled_gate_up_silu(s["gate"][0], s["gate"][1], s["up"][0], s["up"][1], s["x"], s["out"])
    if kind == "int4-gemm":
        return s["be"].int4_batched_matvec(s["w"], s["s"], s["x"], s["out"])
    if kind == "fp8-gemm":
        return s["be"].scaled_batched_matvec(s["w"], s["s"], s["x"], s["out"])
    if kind == "lm-head":
        tokens = s["be"].matvec_argmax_batched(s["w"], s["x"], s["logits"], out=s["tokens"])
        return {"logits": s["logits"], "tokens": tokens}
    if kind == "attention":
        return s["be"].single_token_gqa_attention(s["q"], s["k"], s["v"], s["out"], case["heads"], case["kv_heads"],
                                                  case["head_dim"], sinks=s["sinks"], active_tokens=s["count"])
    if kind == "experts":
        s["be"].mxfp_lowbit_selected_swiglu_tokens(s["gate_up"][0], s["gate_up"][1], s["x"], s["idx"], s["act"], bits=4,
                                                   alpha=_ALPHA, limit=_LIMIT, bias=s["gate_up_bias"])
        s["be"].mxfp_lowbit_weighted_down_tokens(s["down"][0], s["down"][1], s["act"], s["idx"], s["scores"], s["out"],
                                                 bits=4, bias=s["down_bias"])
        return {"act": s["act"], "out": s["out"]}
    if kind == "quantize-int4":
        packed, scales = quantize_to_int4_cpu(s["w"], group_size=case["group"])
        return {"packed": packed, "scales": scales}
    dec = s["dec"]
    tokens = dec.generate(s["start"], case["prior"], case["steps"])
    if kind == "moe-decode":   # the last step's logits as well as its tokens
        s["be"].matvec_argmax_batched(dec.w.lm_head, dec.final_all, s["logits"], out=s["best"])
    return {"logits": s["logits"], "tokens": np.array(tokens, dtype=np.int64)}


# ------------------------------------------------------------------------------- cost
def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "int4-gemv":
        n, k = case["rows"], case["cols"]
        return {"bytes": n * k // 2 + n * k // 128 * 2 + 2 * (n + k), "flops": 2 * n * k}
    if kind == "fp8-gate-up":
        n, k = case["rows"], case["cols"]
        return {"bytes": 2 * (n * k + 4 * n) + 2 * (n + k), "flops": 4 * n * k}
    if kind in ("int4-gemm", "fp8-gemm"):
        n, k, m = case["rows"], case["cols"], case["m"]
        w = n * k // 2 + n * k // 128 * 2 if kind == "int4-gemm" else n * k + 4 * n
        return {"bytes": w + 2 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "lm-head":
        n, k, m = case["rows"], case["cols"], case["m"]
        return {"bytes": 2 * n * k + 2 * m * (n + k) + 8 * m, "flops": 2 * m * n * k}
    if kind == "attention":
        kv = case["kv_heads"] * case["tokens"] * case["head_dim"]
        return {"bytes": 4 * kv + 4 * case["heads"] * case["head_dim"],
                "flops": 4 * case["heads"] * case["tokens"] * case["head_dim"]}
    if kind == "experts":
        E, H, I, T, k = (case[n] for n in ("experts", "hidden", "inter", "tokens", "top_k"))
        slots, seen = T * k, E * (1 - (1 - min(1, k / E)) ** T)   # experts that some token is expected to choose
        return {"bytes": seen * (3 * H * I * 17 / 32 + 2 * (2 * I + H)) + 2 * T * H * 2 + 2 * slots * I * 2,
                "flops": 6 * slots * H * I}
    if kind == "quantize-int4":
        n, k = case["rows"], case["cols"]
        size = 4 if case["dtype"] == "f32" else 2
        return {"bytes": n * k * size + n * k // 2 + n * (k // case["group"]) * 2, "flops": 8 * n * k}
    if kind == "dense-decode":
        s = DenseShape(layers=case["layers"])
        params = s.layers * (s.hidden * (2 * s.q_dim + 2 * s.kv_dim) + 3 * s.hidden * s.intermediate)
        head = s.vocab * s.hidden
        kv = s.layers * 2 * s.kv_dim * (case["prior"] + case["steps"] / 2)
        return {"bytes": case["steps"] * (params * 0.5 * (1 + 4 / 128) + 2 * head + 2 * kv),
                "flops": case["steps"] * 2 * (params + head + s.heads // s.kv_heads * kv)}
    s, B = MoEShape(layers=case["layers"]), case["batch"]
    dense = s.layers * (s.hidden * (2 * s.q_dim + 2 * s.kv_dim) + s.experts * s.hidden)
    expert, head = 3 * s.hidden * s.intermediate, s.vocab * s.hidden
    seen = s.experts * (1 - (1 - s.top_k / s.experts) ** B)
    kv = s.layers * 2 * s.kv_dim * (case["prior"] + case["steps"] / 2)
    n = case["steps"]
    return {"bytes": n * (2 * dense + s.layers * seen * expert * 17 / 32 + 2 * B * kv) + (n + 1) * 2 * head,
            "flops": 2 * B * (n * (dense + s.layers * s.top_k * expert + s.heads // s.kv_heads * kv) + (n + 1) * head)}


def tolerance(case: dict):
    kind = case["kind"]
    if kind == "quantize-int4":
        return "exact"                       # codes and scales are defined to the bit
    if kind in ("dense-decode", "moe-decode"):
        # every operator of the decoders has a fixed reduction order, and the parity tests
        # compare their logits and streams with the oracle's bit for bit
        return "exact"
    # four times the distance to ``exact`` that the operators showed: 2.1e-4 for one fp16
    # rounding of the result (2.8e-4 where the weights are rounded too, 3.5e-4 / 4.9e-4 after
    # the experts' intermediate roundings), 1.7e-3 for one bf16 rounding (3.2e-3 for the
    # gate / up product, whose two factors are rounded to bf16 for every output type)
    if kind == "lm-head":
        return {"rel": 9e-4, "max": 4e-3, "differ": 0.0}
    if kind == "experts":
        return {"rel": 2e-3, "max": 1e-2}
    if kind == "fp8-gate-up":
        return {"rel": 1.2e-2, "max": 5e-2}
    if case.get("dtype") == "bf16":
        return {"rel": 7e-3, "max": 3e-2}
    return {"rel": 1.2e-3, "max": 6e-3}


# ------------------------------------------------------------------------------- float64
def _int4_values(packed, scales):
    codes = torch.stack([packed & 15, packed >> 4], dim=2).reshape(packed.shape[0], -1)
    return (codes.double() - 8) * scales.double().repeat_interleave(128, dim=1)


_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _mxfp4_values(blocks, scales):
    """one expert's [rows, K / 32, 16] bytes and [rows, K / 32] exponents as float64 [rows, K]"""
    table = torch.tensor(_E2M1 + [-v for v in _E2M1], device=blocks.device, dtype=torch.float64)
    v = table[torch.stack([blocks & 15, blocks >> 4], dim=3).long()].reshape(*scales.shape, 32)
    return (v * torch.exp2(scales.double() - 127)[..., None]).reshape(blocks.shape[0], -1)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("quantize-int4", "dense-decode", "moe-decode"):
        return None
    s = _inputs(case, seed)
    if kind == "int4-gemv":
        return _int4_values(s["w"], s["s"]) @ s["x"].double()
    if kind == "fp8-gate-up":
        gate, up = ((w.float().double() @ s["x"].double()) * c.double() for w, c in (s["gate"], s["up"]))
        return gate * torch.sigmoid(gate) * up
    if kind == "int4-gemm":
        return s["x"].double() @ _int4_values(s["w"], s["s"]).T.contiguous()
    if kind == "fp8-gemm":
        return (s["x"].double() @ s["w"].float().double().T.contiguous()) * s["s"].double()
    if kind == "lm-head":
        x = s["x"].double()
        parts = [x @ s["w"][r:r + 8192].double().T.contiguous() for r in range(0, case["rows"], 8192)]
        return {"logits": torch.cat(parts, dim=1), "tokens": None}
    if kind == "attention":
        G, D, n = case["heads"] // case["kv_heads"], case["head_dim"], case["tokens"]
        out = []
        for h in range(case["kv_heads"]):
            q = s["q"].view(-1, D)[h * G:(h + 1) * G].double()
            logits = q @ s["k"][h, :n].double().T.contiguous() / math.sqrt(D)
            if s["sinks"] is not None:
                logits = torch.cat([logits, s["sinks"][h * G:(h + 1) * G, None].double()], dim=1)
            out.append(logits.softmax(dim=1)[:, :n] @ s["v"][h, :n].double())
        return torch.cat(out).reshape(-1)
    # experts
    T, k = case["tokens"], case["top_k"]
    act = torch.empty((T * k, case["inter"]), device="cuda", dtype=torch.float64)
    out = torch.zeros((T, case["hidden"]), device="cuda", dtype=torch.float64)
    for e in s["idx"].unique().tolist():
        t, slot = (s["idx"] == e).nonzero(as_tuple=True)
        y = s["x"][t].double() @ _mxfp4_values(s["gate_up"][0][e], s["gate_up"][1][e]).T.contiguous() \
            + s["gate_up_bias"][e].double()
        gate, up = y[:, 0::2].clamp(max=_LIMIT), y[:, 1::2].clamp(-_LIMIT, _LIMIT)
        a = (up + 1) * gate * torch.sigmoid(_ALPHA * gate)
        act[t * k + slot] = a
        y = a @ _mxfp4_values(s["down"][0][e], s["down"][1][e]).T.contiguous() + s["down_bias"][e].double()
        out.index_add_(0, t, y * s["scores"][t, slot].double()[:, None])
    return {"act": act, "out": out}
