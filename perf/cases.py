"""The calls whose speed matters, as data, with inputs, bounds and references.

A case is one call sequence that a program makes for one MoE layer.  ``layer`` selects the
entry point:

* ``int4``   ``fused_experts`` on a packed INT4 bank with group size 128, the layer call of the
  SGLang hook, from one decoded token up to a prefill batch;
* ``group``  the same call with the other group sizes that the packing accepts (32, 64, 96, 192)
  and the hidden / intermediate sizes that go with them, as tensor-parallel shards have them;
* ``mixed``  ``fused_experts_mixed``: BF16, INT8 and INT4 experts of one layer as a quant plan
  assigns them, with or without always-on shared experts;
* ``steps_int4`` / ``steps_full``  the layer put together from its primitives, router logits to
  output: ``fused_topk``, ``dispatch``, one grouped GEMM per projection (INT4, or the weights as
  the model stores them), ``silu_and_mul`` and ``unsort_output``;
* ``pack``   quantising a layer's banks when a model is loaded.

Model sizes are those of ``exq_amd.synth.CONFIGS``; ``draw`` adds generic ones between them.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from exq_amd import synth

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_MAX_FLOPS = 2.0 * 4096 * 2 * 3 * 4096 * 14336   # the largest listed case (Mixtral, 4096 tokens)
_MAX_WEIGHTS = 8 * 3 * 4096 * 14336              # weight elements of its layer


def _model(name: str, layer: str, tokens: int, act: str, **extra) -> dict:
    c = synth.CONFIGS[name]
    case = dict(layer=layer, tokens=tokens, hidden=c.hidden, inter=c.inter, experts=c.n_experts,
                top_k=c.top_k, shared=0, group=128, renorm=c.renormalize, zipf=c.zipf, act=act)
    case.update(extra)
    return case


def listed() -> list[dict]:
    return [
        # One user generating: a single token through one layer, bound by latency.
        dict(_model("qwen3", "int4", 1, "bf16"), name="decode_qwen3_t1"),
        # An ordinary decode batch of a server; the repository's headline size.
        dict(_model("qwen3", "int4", 16, "bf16"), name="decode_qwen3_t16"),
        # A full decode batch: most experts active, several tokens each.
        dict(_model("olmoe", "int4", 64, "bf16"), name="decode_olmoe_t64"),
        # A decode batch of a layer whose quant plan keeps the hot experts BF16 / INT8.
        dict(_model("mixed_olmoe", "mixed", 32, "bf16"), name="decode_mixed_olmoe_t32"),
        # A short prompt, or a decode batch too large for the decode kernels: few rows for each
        # of many experts.
        dict(_model("qwen3", "int4", 187, "bf16"), name="chunk_qwen3_t187"),
        # A prefill chunk of the mixed-precision layer, with a ragged last chunk's size.
        dict(_model("mixed_olmoe", "mixed", 1000, "bf16"), name="prefill_mixed_olmoe_t1000"),
        # A prefill chunk with BF16 shared experts beside the INT4 routed ones.
        dict(_model("deepseek_v2_lite", "mixed", 2048, "bf16", shared=2, plan="int4"),
             name="prefill_deepseek_t2048"),
        # The largest: a long prompt through a layer of a few large experts.
        dict(_model("mixtral", "int4", 4096, "bf16"), name="prefill_mixtral_t4096"),
        # A bank packed with a finer group, in fp16.
        dict(_model("qwen3", "group", 48, "f16", group=64), name="group64_qwen3_t48"),
        # The layer from its primitives, INT4 in fp16 (the reference's activation type).
        dict(_model("olmoe", "steps_int4", 331, "f16"), name="steps_int4_olmoe_t331"),
        # The same on the model's own BF16 weights (layers that a plan does not cover).
        dict(_model("olmoe", "steps_full", 96, "bf16"), name="steps_full_olmoe_t96"),
        # Loading: both banks of a layer quantised once.
        dict(layer="pack", experts=64, hidden=2048, inter=1024, group=128, bits=4, act="f16",
             name="pack_int4_olmoe"),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    while True:
        case = _draw(rng)
        w = case["experts"] * 3 * case["hidden"] * case["inter"]
        big = _MAX_WEIGHTS // 4 if case["layer"] in ("steps_full", "pack") else _MAX_WEIGHTS
        if w <= big and work(case)["flops"] <= 0.8 * _MAX_FLOPS:
            return case


def _draw(rng) -> dict:
    layer = rng.choice(["int4", "int4", "int4", "mixed", "mixed", "group", "steps_int4",
                        "steps_full", "pack"])
    if layer == "pack":
        bits = rng.choice([4, 4, 8])
        return dict(layer=layer, experts=_log_int(rng, 4, 64), hidden=128 * rng.randint(6, 24),
                    inter=128 * rng.randint(2, 16), group=rng.choice([128, 128, 64, 32]),
                    bits=bits, act=rng.choice(["f16", "bf16", "f32"]))
    act = rng.choice(["bf16", "bf16", "f16"])
    top_tokens = {"int4": 4096, "mixed": 2500, "group": 1024, "steps_int4": 1500,
                  "steps_full": 1500}[layer]
    tokens = _log_int(rng, 1, top_tokens)
    if layer in ("int4", "mixed") and rng.random() < 0.5:
        name = rng.choice(["olmoe", "qwen3", "mixtral"] if layer == "int4"
                          else ["mixed_olmoe", "deepseek_v2_lite"])
        if name == "deepseek_v2_lite":
            return _model(name, layer, tokens, act, shared=2, plan="int4")
        return _model(name, layer, tokens, act)
    experts = _log_int(rng, 8, 128)
    case = dict(layer=layer, tokens=tokens, hidden=128 * rng.randint(6, 32),
                inter=128 * rng.randint(2, 18), experts=experts,
                top_k=rng.choice([2, 4, 6, 8]), shared=0, group=128,
                renorm=rng.random() < 0.5, zipf=rng.random() < 0.75, act=act)
    if layer == "mixed":
        case["shared"] = rng.choice([0, 0, 1, 2])
    if layer == "group":
        g = case["group"] = rng.choice([32, 64, 96, 192])
        case["hidden"] = g * rng.randint(-(-768 // g), 4096 // g)
        case["inter"] = g * rng.randint(-(-96 // g), 2048 // g)
    return case


# ---- inputs -----------------------------------------------------------------------------------

def _config(case: dict) -> synth.MoeConfig:
    return synth.MoeConfig("case", 0, case["hidden"], case["inter"], case["experts"],
                           case["top_k"], case["renorm"], zipf=case["zipf"],
                           n_shared=case["shared"])


def _generator(seed: int, part: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(1000003 * (seed % (1 << 40)) + part)


def _logits(case: dict, seed: int) -> np.ndarray:
    # Zipf-skewed router logits, as a trained router's expert popularity is
    return synth.router_logits(_config(case), case["tokens"], (seed * 7919 + 17) % (1 << 32))


def _routing(case: dict, seed: int):
    ids, w = synth.softmax_topk(_logits(case, seed), case["top_k"], case["renorm"])
    return (torch.from_numpy(ids.astype(np.int32)).cuda(), torch.from_numpy(w).cuda())


def _hidden(case: dict, seed: int) -> torch.Tensor:
    return torch.randn(case["tokens"], case["hidden"], generator=_generator(seed, 1),
                       device="cuda").to(DTYPES[case["act"]])


def _weights(n: int, rows: int, k: int, seed: int, part: int,
             dtype: torch.dtype = torch.float16) -> torch.Tensor:
    w = torch.empty(n, rows, k, dtype=dtype, device="cuda")
    g = _generator(seed, part)
    for e in range(n):
        w[e] = torch.randn(rows, k, generator=g, device="cuda") * 0.02
    return w


def _banks(case: dict, seed: int, dtype: torch.dtype = torch.float16):
    n, h, i = case["experts"], case["hidden"], case["inter"]
    return _weights(n, 2 * i, h, seed, 2, dtype), _weights(n, h, i, seed, 3, dtype)


def _shared_banks(case: dict, seed: int):
    s, h, i = case["shared"], case["hidden"], case["inter"]
    if s == 0:
        return None, None
    return _weights(s, 2 * i, h, seed, 4), _weights(s, h, i, seed, 5)


def _tiers(case: dict, seed: int) -> list[int]:
    """Quant plan: the experts that the router favours stay BF16 (10 %) or INT8 (20 %)."""
    n = case["experts"]
    if case.get("plan") == "int4":
        return [2] * n
    ids = _routing(dict(case, tokens=512), seed)[0].long().flatten()
    order = torch.argsort(torch.bincount(ids, minlength=n), descending=True, stable=True).tolist()
    n_bf, n_i8 = round(0.1 * n), round(0.2 * n)
    tiers = [2] * n
    for rank, e in enumerate(order):
        tiers[e] = 0 if rank < n_bf else (1 if rank < n_bf + n_i8 else 2)
    return tiers


def _rtn_int4(w: torch.Tensor, group: int):
    """Round-to-nearest INT4: integers [.., K] and fp16 scales [.., K / group] of [.., K]."""
    g = w.float().unflatten(-1, (-1, group))
    s = (g.abs().amax(-1) / 7.0).clamp_min(torch.finfo(torch.float32).eps)
    q = torch.round(g / s.unsqueeze(-1)).clamp_(-8, 7).to(torch.int8).flatten(-2)
    return q, s.to(torch.float16)


def _pack(w: torch.Tensor, group: int):
    """An [E, N, K] bank in the packed layout: low nibble even k, nibble = q + 8."""
    packed, scales = [], []
    for e in range(w.shape[0]):
        q, s = _rtn_int4(w[e], group)
        u = (q + 8).to(torch.uint8)
        packed.append(u[:, 0::2] | (u[:, 1::2] << 4))
        scales.append(s)
    return torch.stack(packed), torch.stack(scales)


def prepare(case: dict, seed: int) -> dict:
    from exq_amd.kernels import MixedExpertBank

    layer = case["layer"]
    state = {"case": case}
    if layer == "pack":
        state["w13"], state["w2"] = _banks(case, seed, DTYPES[case["act"]])
        return state
    state["x"] = _hidden(case, seed)
    if layer in ("int4", "group", "mixed"):
        state["ids"], state["weights"] = _routing(case, seed)
    else:
        state["logits"] = torch.from_numpy(_logits(case, seed)).cuda()
    if layer == "mixed":
        w13, w2 = _banks(case, seed)
        s13, s2 = _shared_banks(case, seed)
        state["bank"] = MixedExpertBank.from_weights(
            w13, w2, _tiers(case, seed), act_dtype=DTYPES[case["act"]], shared_w13=s13,
            shared_w2=s2, shared_tier=0)
    elif layer == "steps_full":
        state["w13"], state["w2"] = _banks(case, seed, DTYPES[case["act"]])
    else:
        w13, w2 = _banks(case, seed)
        state["w13"] = _pack(w13, case["group"])
        del w13
        state["w2"] = _pack(w2, case["group"])
    return state


# ---- one pass ---------------------------------------------------------------------------------

def _steps(state: dict, gemm) -> dict:
    from exq_amd.kernels import fused_topk, unsort_output
    from exq_amd.kernels.exq_dispatch import dispatch, silu_and_mul

    case, x = state["case"], state["x"]
    n_exp, slots = case["experts"], case["tokens"] * case["top_k"]
    weights, ids = fused_topk(state["logits"], case["top_k"], case["renorm"])
    order = torch.empty(slots, dtype=torch.int64, device=x.device)
    sorted_ids = torch.empty(slots, dtype=torch.int64, device=x.device)
    ends = torch.empty(n_exp + 1, dtype=torch.int32, device=x.device)
    dispatch(ids, order, sorted_ids, ends, n_exp)
    gate_up = gemm(x, "w13", ids)
    mid = torch.empty(slots, case["inter"], dtype=x.dtype, device=x.device)
    silu_and_mul(gate_up, mid)
    down = gemm(mid, "w2", sorted_ids.view(slots, 1))  # rows are already in expert order
    out = unsort_output(down, ids, weights, n_exp)
    return {"weights": weights, "ids": ids, "order": order, "ends": ends, "out": out}


def run(state: dict):
    from exq_amd.kernels import (fused_experts, fused_experts_mixed, moe_grouped_gemm,
                                 moe_int4_forward, pack_experts_int4, quantize_int8_rows)

    case = state["case"]
    layer = case["layer"]
    if layer in ("int4", "group"):
        return fused_experts(state["x"], *state["w13"], *state["w2"], state["weights"],
                             state["ids"])
    if layer == "mixed":
        return fused_experts_mixed(state["x"], state["bank"], state["weights"], state["ids"])
    if layer == "steps_int4":
        return _steps(state, lambda x, w, ids: moe_int4_forward(x, *state[w], ids,
                                                                case["experts"]))
    if layer == "steps_full":
        return _steps(state, lambda x, w, ids: moe_grouped_gemm(x, state[w], ids,
                                                                case["experts"]))
    if case["bits"] == 8:
        return [*quantize_int8_rows(state["w13"]), *quantize_int8_rows(state["w2"])]
    return [*pack_experts_int4(state["w13"], case["group"]),
            *pack_experts_int4(state["w2"], case["group"])]


# ---- bounds -----------------------------------------------------------------------------------

def _expert_bytes(case: dict, tier: int) -> float:
    h, i = case["hidden"], case["inter"]
    if tier == 0:
        return 6.0 * h * i
    if tier == 1:
        return 3.0 * h * i + 2 * (2 * i + h)
    return 1.5 * h * i + 6.0 * h * i / case["group"]


def work(case: dict) -> dict:
    """Active weights, rows in and out once; 2 flops per multiply-add of a routed row."""
    n, h, i = case["experts"], case["hidden"], case["inter"]
    if case["layer"] == "pack":
        el = 3.0 * n * h * i
        src = el * DTYPES[case["act"]].itemsize
        out = (el + 2.0 * n * (2 * i + h)) if case["bits"] == 8 else el / 2 + 2 * el / case["group"]
        return {"bytes": src + out, "flops": 0}
    t, k, s = case["tokens"], case["top_k"], case["shared"]
    # the active experts of one seeded batch; a mixed layer's plan ranks them by popularity
    ids, _ = synth.softmax_topk(_logits(case, 1), k, case["renorm"])
    active = np.unique(ids)
    if case["layer"] == "mixed" and case.get("plan") != "int4":
        rows = np.bincount(synth.softmax_topk(_logits(dict(case, tokens=512), 1), k,
                                              case["renorm"])[0].ravel(), minlength=n)
        rank = np.empty(n, dtype=np.int64)
        rank[np.argsort(-rows, kind="stable")] = np.arange(n)
        n_bf, n_i8 = round(0.1 * n), round(0.2 * n)
        weights = sum(_expert_bytes(case, 0 if rank[e] < n_bf else
                                    (1 if rank[e] < n_bf + n_i8 else 2)) for e in active)
    else:
        weights = len(active) * _expert_bytes(case, 0 if case["layer"] == "steps_full" else 2)
    weights += s * _expert_bytes(case, 0)
    rows_io = 2.0 * t * h * 2
    routing = 8.0 * t * k
    if case["layer"].startswith("steps"):
        routing = 4.0 * t * n + 8.0 * t * k + 8.0 * t * k + 4.0 * (n + 1)
    return {"bytes": weights + rows_io + routing, "flops": 2.0 * t * (k + s) * 3 * h * i}


def tolerance(case: dict):
    if case["layer"] == "pack":
        return "exact"
    # One rounding to the activation type at `mid` and one at the output (and, in large
    # prefill batches, one of each scaled weight): bf16 2.3e-3 to 3.7e-3 from the 64-bit
    # result, fp16 2.6e-4 to 4.2e-4; the primitives round the gate / up rows too.  A single
    # element is off by up to 2.1e-2 of the rms in bf16 over 10^7 elements.
    if case["act"] == "f16":
        tol = {"rel": 1.6e-3, "max": 1.5e-2}
    else:
        tol = {"rel": 1.2e-2, "max": 1.0e-1}
    if case["layer"].startswith("steps"):
        tol["differ"] = 1e-3  # ids of experts whose probabilities differ by an ulp
    return tol


# ---- 64-bit references ------------------------------------------------------------------------

def _deq_int4(w: torch.Tensor, group: int) -> torch.Tensor:
    q, s = _rtn_int4(w.to(torch.float16), group)
    return (q.double().unflatten(-1, (-1, group)) * s.double().unsqueeze(-1)).flatten(-2)


def _deq_int8(w: torch.Tensor) -> torch.Tensor:
    w = w.float()
    s = (w.abs().amax(-1, keepdim=True) / 127.0).clamp_min(torch.finfo(torch.float32).eps)
    q = torch.round(w / s).clamp_(-128, 127)
    return q.double() * s.to(torch.float16).double()


def exact(case: dict, seed: int):
    layer = case["layer"]
    if layer == "pack":
        return None  # whole numbers: compared as they are
    x = _hidden(case, seed).double()
    if layer == "steps_full":
        w13, w2 = _banks(case, seed, DTYPES[case["act"]])
    else:
        w13, w2 = _banks(case, seed)
    n, t, k, i = case["experts"], case["tokens"], case["top_k"], case["inter"]
    tiers = [2] * n
    steps = layer.startswith("steps")
    if layer == "mixed":
        tiers = _tiers(case, seed)
    if layer == "steps_full":
        tiers = [0] * n
    if steps:
        p = torch.softmax(torch.from_numpy(_logits(case, seed)).cuda().double(), -1)
        top, ids = torch.sort(p, dim=-1, descending=True, stable=True)
        weights, ids = top[:, :k], ids[:, :k]
        if case["renorm"]:
            weights = weights / weights.sum(-1, keepdim=True)
    else:
        ids, weights = _routing(case, seed)
        ids, weights = ids.long(), weights.double()
    act = DTYPES[case["act"]]

    def expert(rows, a, b, tier):
        if tier == 2:
            a, b = _deq_int4(a, case["group"]), _deq_int4(b, case["group"])
        elif tier == 1:
            a, b = _deq_int8(a), _deq_int8(b)
        else:
            a, b = a.to(act).double(), b.to(act).double()
        gu = torch.mm(rows, a.t().contiguous())
        return torch.mm(torch.nn.functional.silu(gu[:, :i]) * gu[:, i:], b.t().contiguous())

    out = torch.zeros(t, case["hidden"], dtype=torch.float64, device="cuda")
    for e in range(n):
        tok, slot = torch.where(ids == e)
        if tok.numel():
            y = expert(x[tok], w13[e], w2[e], tiers[e])
            out.index_add_(0, tok, y * weights[tok, slot].unsqueeze(-1))
    s13, s2 = _shared_banks(case, seed)
    for s in range(case["shared"]):
        out += expert(x, s13[s], s2[s], 0)
    if not steps:
        return out
    return {"weights": weights, "ids": None, "order": None, "ends": None, "out": out}
