"""Performance cases of the framework: what a program that serves NF4 mixture-of-experts
models has it do, through its public entry points, each with its inputs, its algorithmic
work, its tolerance and a 64-bit reference in plain torch.

Kinds of case:
  layer    MoELayer.forward on resident NF4 experts (routing, grouping, expert FFN, combine):
           T = 1 is one decode token, 2-64 decode batches and short prompts, hundreds to
           thousands prompt prefill.
  expert   QuantizedMixtralExpert.forward: one expert on all rows (a program with its own
           routing).
  decode   NativeDecoder.decode_step: one generated token behind `past` cached ones.
  prefill  NativeDecoder.forward: T prompt tokens behind `past` cached ones.
  nf4      QuantizedMixtralExpert(w1, w2, w3) and NF4Linear.dequantize: an expert's bf16
           weights packed at load time, and read back.
"""
from __future__ import annotations

import math

import torch

from moeinfra_amd import ops
from moeinfra_amd._lib import MoeNf4Expert
from moeinfra_amd.cache.manager import CacheManager
from moeinfra_amd.cache.types import EvictionPolicy
from moeinfra_amd.engine.decoder import DecoderWeights, LayerWeights, MixtralShape, NativeDecoder
from moeinfra_amd.engine.router import ExpertRouter
from moeinfra_amd.model.expert import QuantizedMixtralExpert
from moeinfra_amd.model.moe_layer import MoELayer

DEV = "cuda:0"
BLOCK = 64
# The published NormalFloat4 levels (QLoRA).
NF4 = (-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453,
       -0.28444138169288635, -0.18477343022823334, -0.09105003625154495, 0.0,
       0.07958029955625534, 0.16093020141124725, 0.24611230194568634, 0.33791524242401123,
       0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0)

# The Mixtral-8x7B shape of the benchmark.
MIX = {"hidden": 4096, "ffn": 14336, "experts": 8, "top_k": 2}
# Other shapes: the reduced one of the smoke run, and generic ones (hidden not a power of
# two, more experts, other top-k).
OTHER = ({"hidden": 1024, "ffn": 3584, "experts": 8, "top_k": 2},
         {"hidden": 2048, "ffn": 7168, "experts": 16, "top_k": 4},
         {"hidden": 3072, "ffn": 8192, "experts": 8, "top_k": 2},
         {"hidden": 6144, "ffn": 16384, "experts": 8, "top_k": 1})
# Attention of the same model: grouped-query, 32 / 8 heads of 128, vocabulary 32000.
HEADS, KV_HEADS, HEAD_DIM, VOCAB, THETA, EPS = 32, 8, 128, 32000, 1e6, 1e-5


def _layer(name, tokens, skew=False, shape=MIX):
    c = {"kind": "layer", "tokens": tokens, "skew": skew, **shape}
    return {"name": name, **c} if name else c


def listed():
    return [
        # One decode token: the latency of every generated token of a model.
        _layer("layer_t1", 1),
        # Decode batches: a few requests at once, skewed (hot experts) and uniform.
        _layer("layer_t4_skew", 4, True),
        _layer("layer_t16", 16),
        # The 40-token prompt of the end-to-end benchmark.
        _layer("layer_t40_skew", 40, True),
        # A paragraph-sized prompt, ragged.
        _layer("layer_t101", 101),
        # Prompt prefill: a page, and the largest batch the benchmark prices.
        _layer("layer_t512", 512),
        _layer("layer_t4096", 4096),
        # A small model's layer, where launches count.
        _layer("layer_small_t13", 13, False, OTHER[0]),
        # A program that routes by itself and calls experts one by one.
        {"name": "expert_t7", "kind": "expert", "tokens": 7, "hidden": 4096, "ffn": 14336},
        # One generated token far into a conversation.
        {"name": "decode_p3000", "kind": "decode", "past": 3000, "max_seq": 4096},
        # A long prompt.
        {"name": "prefill_t1500", "kind": "prefill", "tokens": 1500, "past": 0, "max_seq": 2048},
        # Loading an expert: quantised from bf16, and reconstructed.
        {"name": "nf4_expert", "kind": "nf4", "hidden": 4096, "ffn": 14336},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    u = rng.random()
    if u < 0.55:
        if rng.random() < 0.7:
            return _layer("", _log(rng, 1, 4096), rng.random() < 0.4)
        shape = rng.choice(OTHER)
        return _layer("", _log(rng, 1, 1024), rng.random() < 0.4, shape)
    if u < 0.65:
        hidden, ffn = rng.choice(((4096, 14336), (1024, 3584), (3072, 8192)))
        return {"kind": "expert", "tokens": _log(rng, 1, 2048), "hidden": hidden, "ffn": ffn}
    if u < 0.80:
        return {"kind": "decode", "past": _log(rng, 16, 3000), "max_seq": rng.choice((4096, 8192))}
    if u < 0.93:
        tokens = _log(rng, 5, 1500)
        room = min(2500, int(1500 * 750 / tokens - tokens / 2))   # no more work than the listed one
        past = 0 if rng.random() < 0.5 else rng.randint(0, max(0, room))
        return {"kind": "prefill", "tokens": tokens, "past": past, "max_seq": 4096}
    # Odd row counts: a projection's rows need not divide anything.
    return {"kind": "nf4", "hidden": 256 * rng.randint(2, 16), "ffn": 64 * rng.randint(9, 223)}


# --------------------------------------------------------------------------- inputs
def _gen(seed, part):
    return torch.Generator(device=DEV).manual_seed((int(seed) * 1000003 + part) % (1 << 62))


def _normal(gen, shape, std=1.0):
    return torch.randn(shape, generator=gen, device=DEV).mul_(std).to(torch.bfloat16)


def _expert_bf16(case, seed, e):
    """(w1 [F, H], w3 [F, H], w2 [H, F]) of expert e: N(0, 0.02), as a fresh linear layer."""
    H, F = case["hidden"], case["ffn"]
    g = _gen(seed, 100 + e)
    return _normal(g, (F, H), 0.02), _normal(g, (F, H), 0.02), _normal(g, (H, F), 0.02)


def _skew_bias(experts):
    """Zipf-shaped logit offsets (exponent 1.2, weight 4), hottest expert not the first."""
    p = torch.tensor([1.0 / (1 + (5 * e + 3) % experts) ** 1.2 for e in range(experts)],
                     dtype=torch.float64)
    return (4.0 * torch.log(p / p.sum())).to(torch.float32).to(DEV)


def _layer_inputs(case, seed):
    g = _gen(seed, 1)
    gate = _normal(g, (case["experts"], case["hidden"]), 0.02)
    x = _normal(g, (1, case["tokens"], case["hidden"]))
    return gate, x, _skew_bias(case["experts"]) if case["skew"] else None


def _model_case(case):
    return {**case, **MIX}


def _decoder_inputs(case, seed):
    """Dense tensors of a one-layer model of the Mixtral shape, the cached keys and values and
    the token ids.  Each token's embedding leans towards two experts' gate rows, as in a
    trained model, so that its routing does not hang on a rounding."""
    H, E = MIX["hidden"], MIX["experts"]
    g = _gen(seed, 2)
    t = {"embed": torch.randn((VOCAB, H), generator=g, device=DEV).mul_(0.02),
         "gate": _normal(g, (E, H), 0.02),
         "qkv": _normal(g, ((HEADS + 2 * KV_HEADS) * HEAD_DIM, H), 0.02),
         "o": _normal(g, (H, HEADS * HEAD_DIM), 0.02),
         "lm_head": _normal(g, (VOCAB, H), 0.02)}
    for n in ("n1", "n2", "n3"):
        t[n] = (1.0 + 0.1 * torch.randn((H,), generator=g, device=DEV)).to(torch.bfloat16)
    tok = torch.arange(VOCAB, device=DEV)
    e1 = (tok * 7) % E
    e2 = (e1 + 1 + (tok // E) % (E - 1)) % E
    t["embed"] = (t["embed"] + 0.1 * t["gate"].float()[e1] + 0.08 * t["gate"].float()[e2]).to(torch.bfloat16)
    n = case.get("tokens", 1)
    t["ids"] = torch.randint(0, VOCAB, (n,), generator=g, device=DEV)
    t["k"] = _normal(g, (KV_HEADS, case["past"], HEAD_DIM), 1.28)
    t["v"] = _normal(g, (KV_HEADS, case["past"], HEAD_DIM), 1.28)
    return t


def prepare(case, seed):
    kind = case["kind"]
    if kind == "layer":
        gate, x, bias = _layer_inputs(case, seed)
        E = case["experts"]
        cache = CacheManager(gpu_slots=E, cpu_slots=E, policy=EvictionPolicy.LRU)
        for e in range(E):
            w1, w3, w2 = _expert_bf16(case, seed, e)
            cache.put(0, e, QuantizedMixtralExpert(w1, w2, w3), device=DEV)
        router = ExpertRouter(gate, case["top_k"], bias=bias)
        layer = MoELayer(0, router, cache, model_loader=None, transfer_scheduler=None)
        return {"kind": kind, "layer": layer, "x": x}
    if kind == "expert":
        w1, w3, w2 = _expert_bf16(case, seed, 0)
        x = _normal(_gen(seed, 1), (case["tokens"], case["hidden"]))
        return {"kind": kind, "expert": QuantizedMixtralExpert(w1, w2, w3), "x": x}
    if kind == "nf4":
        w1, w3, w2 = _expert_bf16(case, seed, 0)
        return {"kind": kind, "w": (w1, w2, w3)}
    t = _decoder_inputs(case, seed)
    m = _model_case(case)
    experts = []
    for e in range(MIX["experts"]):
        w1, w3, w2 = _expert_bf16(m, seed, e)
        experts.append({"w1": ops.nf4_quantize(w1), "w3": ops.nf4_quantize(w3),
                        "w2": ops.nf4_quantize(w2)})
    table = ops.expert_table([MoeNf4Expert(*(p.data_ptr() for n in ("w1", "w3", "w2") for p in st[n]))
                              for st in experts])
    shape = MixtralShape(layers=1)
    weights = DecoderWeights(shape, t["embed"],
                             [LayerWeights(t["n1"], t["qkv"], t["o"], t["n2"], t["gate"], experts, table)],
                             t["n3"], t["lm_head"])
    dec = NativeDecoder(weights, case["max_seq"], DEV)
    dec.k_cache[0, :, :case["past"]] = t["k"]
    dec.v_cache[0, :, :case["past"]] = t["v"]
    past = torch.full((1,), case["past"], dtype=torch.int32, device=DEV)
    return {"kind": kind, "dec": dec, "ids": t["ids"], "past": past, "tok": t["ids"][:1].clone()}


def run(state):
    kind = state["kind"]
    if kind == "layer":
        out = state["layer"].forward(state["x"])
        return {"out": out, "experts": state["layer"].last_expert_indices}
    if kind == "expert":
        return {"out": state["expert"].forward(state["x"])}
    if kind == "nf4":
        expert = QuantizedMixtralExpert(*state["w"])
        lins = {"w1": expert.w1, "w2": expert.w2, "w3": expert.w3}
        return {n: {"packed": l.weight, "absmax": l.quant_state.absmax, "bf16": l.dequantize()}
                for n, l in lins.items()}
    dec = state["dec"]
    dec.pos.copy_(state["past"])
    if kind == "decode":
        state["tok"].copy_(state["ids"][:1])     # the program's own choice of token
        logits = dec.decode_step(state["tok"])
    else:
        logits = dec.forward(state["ids"])
    return {"logits": logits, "k": dec.k_cache, "v": dec.v_cache}


# --------------------------------------------------------------------------- work
def _nf4_bytes(n):
    return n // 2 + 4 * (n // BLOCK)


def _routed(case):
    """Expected number of distinct experts that the tokens are routed to."""
    E, k, T = case["experts"], case["top_k"], case["tokens"]
    if not case["skew"]:
        return E * (1.0 - (1.0 - k / E) ** T)
    w = sorted((1.0 / (1 + e) ** 4.8 for e in range(E)), reverse=True)
    share = [min(1.0, k * v / sum(w)) for v in w]
    return max(float(k), sum(1.0 - (1.0 - s) ** T for s in share))


def work(case):
    kind = case["kind"]
    if kind == "layer":
        H, F, T, k = case["hidden"], case["ffn"], case["tokens"], case["top_k"]
        return {"bytes": _routed(case) * 3 * _nf4_bytes(H * F) + 4 * T * H + 2 * case["experts"] * H + 8 * T * k,
                "flops": 6.0 * T * k * H * F}
    H, F = case.get("hidden", MIX["hidden"]), case.get("ffn", MIX["ffn"])
    if kind == "expert":
        return {"bytes": 3 * _nf4_bytes(H * F) + 4 * case["tokens"] * H, "flops": 6.0 * case["tokens"] * H * F}
    if kind == "nf4":     # bf16 read, NF4 written; NF4 read, bf16 written
        return {"bytes": 3 * (4 * H * F + 2 * _nf4_bytes(H * F)), "flops": 0}
    T, P = case.get("tokens", 1), case["past"]
    E, k = MIX["experts"], MIX["top_k"]
    rows = (HEADS + 2 * KV_HEADS) * HEAD_DIM
    dense = rows * H + H * HEADS * HEAD_DIM
    keys = T * P + T * (T + 1) // 2
    U = E * (1.0 - (1.0 - k / E) ** T)
    return {"bytes": 2 * dense + 2 * VOCAB * H + U * 3 * _nf4_bytes(H * F) + 2 * 2 * KV_HEADS * HEAD_DIM * (P + T)
            + 2 * T * H + 2 * VOCAB,
            "flops": 2.0 * T * dense + 6.0 * T * k * H * F + 4.0 * HEADS * HEAD_DIM * keys + 2.0 * VOCAB * H}


def tolerance(case):
    # bf16 results of bf16 activations and NF4 weights with fp32 sums.  About four times the
    # error measured against the 64-bit reference below: layer 5.1e-3 to 5.4e-3, expert
    # 4.7e-3 to 5.4e-3; whole calls (rounded cos/sin, scores, hidden states) 2.0e-2 to 2.4e-2,
    # held at 3e-2.  NF4 bytes and the reconstructed values are the same in any
    # implementation.  Routing ties are decided by bf16 logits: one choice in a thousand may
    # differ with the order of the fp32 sums behind them.
    kind = case["kind"]
    if kind == "layer":
        return {"rel": 0.02, "max": 0.15, "differ": 0.001}
    if kind == "expert":
        return {"rel": 0.02, "max": 0.15}
    if kind == "nf4":
        return "exact"
    return {"rel": 0.03, "max": 0.25}


# --------------------------------------------------------------------------- 64-bit reference
def _nf4_f64(w):
    """The values that NF4 keeps of w (fp64): per 64-value block the nearest level times the
    block's largest magnitude, ties to the lower level."""
    f = w.float().reshape(-1, BLOCK)
    absmax = f.abs().amax(dim=1, keepdim=True)
    inv = torch.where(absmax > 0, 1.0 / absmax, torch.zeros_like(absmax))
    code = torch.tensor(NF4, dtype=torch.float32, device=w.device)
    mid = (code[1:] + code[:-1]) / 2
    q = torch.bucketize(f * inv, mid)
    return (code.double()[q] * absmax.double()).reshape(w.shape), absmax.reshape(-1)


def _expert_f64(case, seed, e, x):
    w1, w3, w2 = (_nf4_f64(w)[0] for w in _expert_bf16(case, seed, e))
    return (torch.nn.functional.silu(x @ w1.t()) * (x @ w3.t())) @ w2.t()


def _moe_f64(case, seed, x, gate, bias):
    """The MoE layer of rows x (fp64); the gate logits are bf16 values by definition."""
    logits = (x @ gate.double().t()).to(torch.bfloat16).double()
    if bias is not None:
        logits = logits + bias.double()
    p = torch.softmax(logits, dim=-1)
    order = torch.sort(p, dim=-1, descending=True, stable=True)
    w, idx = order.values[:, :case["top_k"]], order.indices[:, :case["top_k"]]
    w = w / w.sum(dim=-1, keepdim=True)
    out = torch.zeros_like(x)
    for e in range(case["experts"]):
        hit = idx == e
        rows = hit.any(dim=-1).nonzero().reshape(-1)
        if rows.numel():
            out[rows] += _expert_f64(case, seed, e, x[rows]) * (w * hit).sum(dim=-1)[rows, None]
    return out, idx


def _rms_f64(h, w):
    return h * torch.rsqrt(h.pow(2).mean(dim=-1, keepdim=True) + EPS) * w.double()


def _rope_f64(x, pos):
    half = HEAD_DIM // 2
    inv = THETA ** (-torch.arange(half, device=DEV, dtype=torch.float64) / half)
    a = pos.double()[:, None] * inv[None, :]
    c, s = a.cos()[:, None, :], a.sin()[:, None, :]
    x1, x2 = x[..., :half], x[..., half:]
    return torch.cat((x1 * c - x2 * s, x2 * c + x1 * s), dim=-1)


def _decoder_f64(case, seed):
    t, m = _decoder_inputs(case, seed), _model_case(case)
    T, P = t["ids"].numel(), case["past"]
    pos = torch.arange(P, P + T, device=DEV)
    h = t["embed"][t["ids"]].double()
    qkv = _rms_f64(h, t["n1"]) @ t["qkv"].double().t()
    q, k, v = qkv.split((HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM), dim=-1)
    q = _rope_f64(q.reshape(T, HEADS, HEAD_DIM), pos)
    k = _rope_f64(k.reshape(T, KV_HEADS, HEAD_DIM), pos)
    kc = torch.zeros((1, KV_HEADS, case["max_seq"], HEAD_DIM), dtype=torch.float64, device=DEV)
    vc = torch.zeros_like(kc)
    kc[0, :, :P], vc[0, :, :P] = t["k"], t["v"]
    kc[0, :, P:P + T] = k.transpose(0, 1)
    vc[0, :, P:P + T] = v.reshape(T, KV_HEADS, HEAD_DIM).transpose(0, 1)
    mask = torch.arange(P + T, device=DEV)[None, :] > pos[:, None]
    a = torch.empty((T, HEADS, HEAD_DIM), dtype=torch.float64, device=DEV)
    for i in range(HEADS):
        kv = i // (HEADS // KV_HEADS)
        s = (q[:, i] @ kc[0, kv, :P + T].t()) * HEAD_DIM ** -0.5
        a[:, i] = torch.softmax(s.masked_fill(mask, float("-inf")), dim=-1) @ vc[0, kv, :P + T]
    h = h + a.reshape(T, -1) @ t["o"].double().t()
    y, _ = _moe_f64(m, seed, _rms_f64(h, t["n2"])[-1:], t["gate"], None)
    logits = _rms_f64(h[-1:] + y, t["n3"]) @ t["lm_head"].double().t()
    return {"logits": logits, "k": kc, "v": vc}


def exact(case, seed):
    kind = case["kind"]
    if kind == "layer":
        gate, x, bias = _layer_inputs(case, seed)
        out, idx = _moe_f64(case, seed, x[0].double(), gate, bias)
        return {"out": out.reshape(x.shape), "experts": idx}
    if kind == "expert":
        x = _normal(_gen(seed, 1), (case["tokens"], case["hidden"]))
        return {"out": _expert_f64(case, seed, 0, x.double())}
    if kind == "nf4":
        out = {}
        for n, w in zip(("w1", "w3", "w2"), _expert_bf16(case, seed, 0)):
            v, absmax = _nf4_f64(w)
            out[n] = {"packed": None, "absmax": absmax.double(), "bf16": v}
        return out
    return _decoder_f64(case, seed)
