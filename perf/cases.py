"""The work that users of this framework give it, as cases that can be timed and checked.

A case is one step of an engine that serves a model of the registry:

``decode``  one decode step of ``streams`` live sequences of about ``context`` tokens each (ragged), as the serving loop
            replays it: the captured graph of the batch over the weights, the paged cache and the recurrent states.
``prompt``  one pass over ``prompts`` new prompts of ``tokens`` tokens together (ragged) through ``LLMEngine.force_step``,
            which returns the logits of the asked positions: prompt processing and the scoring of given texts.
``mixed``   one step that decodes ``streams - 1`` sequences and takes in ``tokens`` prompt rows for the slot that is free,
            as a loaded server does it all the time.

Models, widths and types are the registry's own: the 7B Mistral of the headline benchmark and the two sizes of the
configuration-driven families that ``bench.py --families`` compares.  Weights are random, tokens uniform.  Dironex and
Murulorn stand aside: with random weights the close calls of their routers flip under any change of rounding and a flipped
row differs by tens of percent, so two correct implementations cannot be told from a wrong one by their logits; the
kernels that they run on are those of the other families.  A decode step returns logits and not the sampled ids for the
same reason: two nearly equal candidates may change places.
"""
from __future__ import annotations

import math
import random

import torch

from distributed_sse_for_llm_response_amd.engine.engine import LLMEngine
from distributed_sse_for_llm_response_amd.engine.kv_cache import PAGE, blocks_needed
from distributed_sse_for_llm_response_amd.engine.model_runner import PrefillSeq
from distributed_sse_for_llm_response_amd.engine.weights import convert_standard
from distributed_sse_for_llm_response_amd.models import kagorax, lobidra, muderax, registry, surodra

DECIDED = 40.0       # what a chosen expert's router logit is ahead of the others, which spread over about four
ROWS = 64            # positions whose logits a prompt case asks for, spread evenly over its prompts
EXACT_FLOPS = 7e14   # the float64 pass of a larger case takes too long
MODELS = ("mistral-7b-v0.3", "mistral-7b-v0.3", "surodra-mid", "surodra-wide", "lobidra-mid", "lobidra-wide", "kagorax-mid",
          "kagorax-wide", "muderax-mid", "muderax-wide")
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
INIT = {"surodra": surodra.init_weights, "lobidra": lobidra.init_weights, "kagorax": kagorax.init_weights,
        "muderax": muderax.init_weights}
SHAPES = {"surodra": surodra.tensor_shapes, "lobidra": lobidra.tensor_shapes, "kagorax": kagorax.tensor_shapes,
          "muderax": muderax.tensor_shapes}


def _decode(model, streams, context):
    return {"kind": "decode", "model": model, "dtype": "bf16", "streams": streams, "context": context}


def _prompt(model, prompts, tokens, dtype="bf16"):
    return {"kind": "prompt", "model": model, "dtype": dtype, "prompts": prompts, "tokens": tokens}


def _mixed(model, streams, context, tokens):
    return {"kind": "mixed", "model": model, "dtype": "bf16", "streams": streams, "context": context, "tokens": tokens}


def listed():
    return [
        # a single user waits for each token: the smallest step, bound by one reading of the weights
        dict(_decode("mistral-7b-v0.3", 1, 700), name="mistral-7b decode 1"),
        # the headline workload: 64 concurrent streams behind 512-token prompts
        dict(_decode("mistral-7b-v0.3", 64, 512), name="mistral-7b decode 64"),
        # time to first token of an 8k prompt
        dict(_prompt("mistral-7b-v0.3", 1, 8192), name="mistral-7b prompt 8192"),
        # a new prompt arrives while the other streams go on
        dict(_mixed("mistral-7b-v0.3", 64, 512, 300), name="mistral-7b mixed 64+300"),
        # matrix-state mixers (delta rule, gated linear attention, retention) beside full attention: a few prompts at once
        dict(_prompt("surodra-mid", 3, 1500), name="surodra-mid prompt 1500"),
        dict(_decode("surodra-wide", 16, 1000), name="surodra-wide decode 16"),
        # convolved attention, matrix memory, experts by token id: one long prompt, and many short conversations
        dict(_prompt("lobidra-wide", 1, 2048), name="lobidra-wide prompt 2048"),
        dict(_decode("lobidra-mid", 64, 512), name="lobidra-mid decode 64"),
        # distance-biased window attention with input-weighted experts: two prompts, and a handful of long conversations
        dict(_prompt("kagorax-mid", 2, 1024), name="kagorax-mid prompt 1024"),
        dict(_decode("kagorax-wide", 5, 2000), name="kagorax-wide decode 5"),
        # latent attention, gated linear recurrence, routed experts
        dict(_prompt("muderax-wide", 2, 3000), name="muderax-wide prompt 3000"),
        # the exact mode: a text scored in 32 bits
        dict(_prompt("surodra-mid", 1, 400, "fp32"), name="surodra-mid fp32 prompt 400"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("prompt", "decode", "mixed"), (5, 5, 1))[0]
    if kind == "mixed":
        return _mixed("mistral-7b-v0.3", _log(rng, 2, 128), _log(rng, 64, 512), _log(rng, 32, 384))
    if kind == "decode":
        model = rng.choice(MODELS)
        streams = _log(rng, 1, 192)
        return _decode(model, streams, _log(rng, 32, min(4096, 36000 // streams)))
    model = rng.choice(MODELS)
    if "-mid" in model and rng.random() < 0.2:
        return _prompt(model, 1, _log(rng, 64, 600), "fp32")
    tokens = _log(rng, 64, 6000 if model.startswith("mistral") else 4096)
    return _prompt(model, rng.randint(1, min(4, tokens // 64 + 1)), tokens)


# ---------------------------------------------------------------------------------------------------- the inputs
def _lengths(case) -> list:
    """Tokens of each prompt (prompt) or cached tokens of each live sequence (decode, mixed): ragged, from the sizes alone."""
    rng = random.Random(str([case[k] for k in sorted(case) if k != "name"]))
    if case["kind"] == "prompt":
        n, total = case["prompts"], case["tokens"]
        share = [rng.uniform(0.5, 1.5) for _ in range(n)]
        lens = [max(1, int(total * s / sum(share))) for s in share]
        lens[0] += total - sum(lens)
        return lens
    n = case["streams"] - (case["kind"] == "mixed")
    return [max(2, int(case["context"] * rng.uniform(0.7, 1.3))) if n > 1 else case["context"] for _ in range(n)]


def _want(lens: list) -> list:
    """The asked positions of each prompt: every prompt's last one and evenly spread ones before it."""
    step = max(1, sum(lens) // ROWS)
    return [sorted(range(n - 1, -1, -step)) for n in lens]


def _tokens(case, cfg, seed: int) -> list:
    g = torch.Generator().manual_seed(seed)
    extra = [case["tokens"]] if case["kind"] == "mixed" else []
    one = case["kind"] != "prompt"   # the token that a decode step reads
    return [torch.randint(3, cfg.vocab_size, (n + one,), generator=g).tolist() for n in _lengths(case) + extra]


def _standard_mistral(cfg, seed: int) -> dict:
    g = torch.Generator(device="cuda").manual_seed(seed)
    H, F, D = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim

    def lin(n, k):
        return torch.empty(n, k, device="cuda", dtype=torch.bfloat16).normal_(0.0, 1.0 / math.sqrt(k), generator=g)

    def norm():
        return torch.empty(H, device="cuda").normal_(1.0, 0.1, generator=g).bfloat16()

    layers = [{"attn_norm": norm(), "q": lin(cfg.num_heads * D, H), "k": lin(cfg.num_kv_heads * D, H),
               "v": lin(cfg.num_kv_heads * D, H), "o": lin(H, cfg.num_heads * D), "ffn_norm": norm(), "gate": lin(F, H),
               "up": lin(F, H), "down": lin(H, F)} for _ in range(cfg.num_layers)]
    embed = torch.empty(cfg.vocab_size, H, device="cuda", dtype=torch.bfloat16).normal_(0.0, 1.0, generator=g)
    return {"embed": embed, "layers": layers, "final_norm": norm(), "lm_head": lin(cfg.vocab_size, H)}


def _checkpoint(fam, cfg, dtype, seed: int) -> dict:
    """The tensors that a checkpoint of the model would hold."""
    if fam.name == "mistral":
        return _standard_mistral(cfg, seed)
    w = INIT[fam.name](cfg, seed=seed, device="cuda", dtype=dtype)
    if fam.name == "muderax":
        # a trained router is decided, a random one leaves many choices to rounding: every token gets its experts, and its
        # embedding a share of their router rows
        g = torch.Generator(device="cuda").manual_seed(seed + 1)
        for i, L in enumerate(cfg.layers):
            if L.mlp is not None and L.weights_of == i:
                router = w[f"l{i}.mlp.router"]
                chosen = torch.rand(cfg.vocab_size, L.mlp.experts, generator=g, device="cuda").argsort(-1)[:, :L.mlp.top]
                w["embed"] += DECIDED * router[chosen].sum(1)
    return w


def _engine_weights(fam, cfg, dtype, seed: int):
    w = _checkpoint(fam, cfg, dtype, seed)
    if fam.name == "mistral":
        return convert_standard(cfg, w, device="cuda")
    from distributed_sse_for_llm_response_amd.engine import weights as W

    convert = {"surodra": W.convert_surodra, "lobidra": W.convert_lobidra, "kagorax": W.convert_kagorax,
               "muderax": W.convert_layered}[fam.name]
    return convert(cfg, w, device="cuda", dtype=dtype)


def prepare(case, seed):
    fam, cfg, _ = registry.resolve(case["model"])
    weights = _engine_weights(fam, cfg, DTYPES[case["dtype"]], seed)
    toks, lens = _tokens(case, cfg, seed), _lengths(case)
    if case["kind"] == "prompt":
        r = registry.make_runner(fam, weights, num_blocks=sum(map(blocks_needed, lens)) + 4, max_batch=len(lens),
                                 max_model_len=max(lens) + PAGE, max_prefill_tokens=sum(lens), device="cuda")
        entries = [(f"chat.{i}", t, w) for i, (t, w) in enumerate(zip(toks, _want(lens)))]
        return {"kind": "prompt", "engine": LLMEngine(r, eos_id=-1), "entries": entries, "end": [e[0] for e in entries]}
    B, mixed = case["streams"], case["kind"] == "mixed"
    need = [n + 1 for n in lens] + ([case["tokens"] + 1] if mixed else [])
    longest = max(need)
    # a decode-only runner keeps no captured prompt passes; a mixed step's chunk sizes are captured with its prompt passes
    r = registry.make_runner(fam, weights, num_blocks=sum(map(blocks_needed, need)) + 4, max_batch=B,
                             max_model_len=longest + PAGE, max_prefill_tokens=512 if mixed else 64, device="cuda")
    free, tables = 0, []
    for s, n in enumerate(need):
        k = blocks_needed(n)
        tables.append(list(range(free, free + k)))
        r.block_tables[s, :k] = torch.arange(free, free + k, dtype=torch.int32)
        free += k
    batch, rows = [], 0
    for s, n in enumerate(lens):
        batch.append(PrefillSeq(slot=s, tokens=toks[s][:n], start_pos=0, block_table=tables[s], last_chunk=False))
        rows += n
        if rows >= 8192 or s == len(lens) - 1:
            r.prefill(batch, ring_row=0)
            batch, rows = [], 0
    r.capture([B])
    r.active[:len(lens)] = 1
    r.temperature[:len(lens)] = 1.0
    r.seeds[:, 0] = torch.arange(1, B + 1, dtype=torch.int32)
    pad = [0] * (B - len(lens))
    state = {"kind": case["kind"], "runner": r, "B": B, "live": len(lens),
             "ids": torch.tensor([t[n] for t, n in zip(toks, lens)] + pad, dtype=torch.int32, device="cuda"),
             "pos": torch.tensor(lens + pad, dtype=torch.int32, device="cuda")}
    if mixed:
        state["chunk"] = [PrefillSeq(slot=B - 1, tokens=toks[-1][:case["tokens"]], start_pos=0, block_table=tables[-1],
                                     last_chunk=True)]
    return state


def run(state):
    if state["kind"] == "prompt":
        return state["engine"].force_step(state["entries"], state["end"])
    r = state["runner"]
    r.ids.copy_(state["ids"])         # the step reads the same tokens at the same positions each time
    r.positions.copy_(state["pos"])
    if state["kind"] == "mixed":
        r.mixed(state["B"], state["chunk"], ring_row=0)
    else:
        r.decode(state["B"])
    return r.logits[:state["live"]]


# ------------------------------------------------------------------------------- what a case cannot do without
def _matrices(fam, cfg):
    """(elements of the weights that every row meets, elements of one expert of each routed layer, experts, top)."""
    if fam.name == "mistral":
        return cfg.num_params() - 2 * cfg.vocab_size * cfg.hidden_size, [], 0, 0
    shared, expert = 0, {}
    layers = [L.get("weights_of", i) for i, L in enumerate(cfg.to_dict()["layers"])]
    for name, shape in SHAPES[fam.name](cfg).items():
        if name in ("embed", "head") or name.endswith("table"):
            continue
        n = math.prod(max(x, 1) for x in shape)
        part = name.split(".")
        if len(part) > 2 and part[1] == "mlp" and part[2][0] == "e" and part[2][1:].isdigit():
            if part[2] == "e0":
                expert[part[0]] = expert.get(part[0], 0) + n
        else:
            shared += n * (layers.count(int(part[0][1:])) if part[0][1:].isdigit() else 1)
    mlps = [L["mlp"] for L in cfg.to_dict()["layers"] if L.get("mlp") and "router" in L["mlp"]]
    router = mlps[0]["router"] if mlps else {"experts": 0, "top": 0}
    return shared, [expert[f"l{j}"] for j in layers if f"l{j}" in expert], router["experts"], router["top"]


def _attention(fam, cfg):
    """(heads, kv heads, score width, value width, window) of each attention, and (heads, dim, vdim) of each matrix state."""
    if fam.name == "mistral":
        return [(cfg.num_heads, cfg.num_kv_heads, cfg.head_dim, cfg.head_dim, 1 << 30)] * cfg.num_layers, []
    att, mat = [], []
    for L in cfg.to_dict()["layers"]:
        m = L["mixer"]
        if "kv_rank" in m:  # one latent row per token, shared by the heads
            att.append((m["heads"], 1, m["dim"] + m["rot_dim"], m["vdim"], (m.get("mask") or {}).get("size", 1 << 30)))
            continue
        left, right = (m["left"], m["right"]) if "left" in m else (m, None)
        if "scale" in left:
            att.append((left["heads"], left["kv_heads"], left["dim"], left["vdim"],
                        (left.get("mask") or {}).get("size", 1 << 30)))
            left = right
        if left is not None and "vdim" in left:
            mat.append((left["heads"], left["dim"], left["vdim"]))
    return att, mat


def work(case):
    fam, cfg, _ = registry.resolve(case["model"])
    size = 4 if case["dtype"] == "fp32" else 2
    width = cfg.hidden_size if fam.name == "mistral" else cfg.width
    lens = _lengths(case)
    spans = [(n, n + 1) for n in lens] if case["kind"] != "prompt" else [(0, n) for n in lens]
    logits = len(lens) if case["kind"] != "prompt" else sum(map(len, _want(lens)))
    if case["kind"] == "mixed":
        spans.append((0, case["tokens"]))
        logits += 1  # the first token of the finished prompt
    rows = sum(b - a for a, b in spans)
    shared, experts, count, top = _matrices(fam, cfg)
    head = cfg.vocab_size * width
    met = count * (1.0 - (1.0 - top / count) ** rows) if count else 0.0
    nbytes = size * (shared + head + sum(experts) * met + rows * width) + 4.0 * logits * cfg.vocab_size
    flops = 2.0 * (rows * (shared + top * sum(experts)) + logits * head)
    att, mat = _attention(fam, cfg)
    for a, b in spans:
        for H, G, D, V, window in att:
            keys = sum(min(p + 1, window) for p in range(a, b))
            nbytes += size * G * (D + V) * ((min(a, window) if a else 0) + b - a)
            flops += 2.0 * H * (D + V) * keys
        for H, D, V in mat:
            nbytes += 4.0 * H * D * V * (2 if a else 1)
            flops += 4.0 * H * D * V * (b - a)
    return {"bytes": nbytes, "flops": flops}


# Up to four times the relative error of the logits against the float64 pass (mistral-7b 0.0072-0.0086, muderax 0.007-0.015,
# surodra 0.0025-0.0027, lobidra 0.0017, kagorax 0.0016; in 32 bits 0.8-4.4e-6): bf16 projections, caches and attention weights
# accumulate over the layers.
REL = {"mistral-7b-v0.3": 0.03, "surodra-mid": 0.012, "surodra-wide": 0.012, "lobidra-mid": 0.006, "lobidra-wide": 0.006,
       "kagorax-mid": 0.006, "kagorax-wide": 0.006, "muderax-mid": 0.03, "muderax-wide": 0.03}


def tolerance(case):
    if case["dtype"] == "fp32":
        return {"rel": 2e-5, "max": 2e-4}
    return {"rel": REL[case["model"]], "max": 12 * REL[case["model"]]}


# ----------------------------------------------------------------------------------- the same in 64 bits, plain torch
F64 = torch.float64


def _rms(v, eps):
    return v / torch.sqrt((v * v).mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def _turn(v, freq, pairs: bool):
    """Rotates the first 2 * len(freq) coordinates of v [B, T, heads, D]: neighbours (pairs) or halves."""
    n, half = 2 * len(freq), len(freq)
    ang = torch.arange(v.shape[1], dtype=F64, device=v.device)[:, None] * freq
    cos, sin = ang.cos()[None, :, None], ang.sin()[None, :, None]
    ia, ib = (slice(0, n, 2), slice(1, n, 2)) if pairs else (slice(0, half), slice(half, n))
    out, a, b = v.clone(), v[..., ia], v[..., ib]
    out[..., ia], out[..., ib] = a * cos - b * sin, b * cos + a * sin
    return out


def _powers(base, dims, device):
    return float(base) ** (-2.0 * torch.arange(dims // 2, dtype=F64, device=device) / dims)


def _band(rot, device):
    f, s = _powers(rot["base"], rot["dims"], device), rot.get("scaling")
    if not s:
        return f
    wave = 2.0 * math.pi / f
    mix = (s["original"] / wave - s["low"]) / (s["high"] - s["low"])
    slow = f / s["factor"]
    return torch.where(wave > s["original"] / s["low"], slow,
                       torch.where(wave < s["original"] / s["high"], f, (1.0 - mix) * slow + mix * f))


def _attend(q, k, v, scale, sink=None, bias=None, seen=None):
    """Causal attention of q [B, T, H, D] over k [B, T, G, D], v [B, T, G, V]; `sink` [H] joins the denominator, `bias`
    [H, T] by distance, `seen` [T, T] instead of the causal mask."""
    B, T, H, _ = q.shape
    G = k.shape[2]
    i = torch.arange(T, device=q.device)
    seen = i[:, None] >= i[None, :] if seen is None else seen
    out = torch.empty(B, T, H, v.shape[3], dtype=F64, device=q.device)
    for b in range(B):
        for h in range(H):
            g = h // (H // G)
            s = (q[b, :, h] @ k[b, :, g].t().contiguous()) * scale
            if bias is not None:
                s = s + bias[h][(i[:, None] - i[None, :]).clamp(min=0)]
            s = s.masked_fill(~seen, float("-inf"))
            top = s.max(-1, keepdim=True).values
            if sink is not None:
                top = torch.maximum(top, sink[h])
            e = torch.exp(s - top)
            den = e.sum(-1, keepdim=True) + (torch.exp(sink[h] - top) if sink is not None else 0.0)
            out[b, :, h] = (e / den) @ v[b, :, g].contiguous()
    return out


def _conv(x, taps):
    K = taps.shape[1]
    out = torch.zeros_like(x)
    for j in range(K):
        back = K - 1 - j
        if back < x.shape[1]:
            out[:, back:] += taps[:, j] * x[:, :x.shape[1] - back]
    return out


def _walk(q, k, v, decay, beta=None):
    """Matrix states walked token by token: q, k [B, T, H, D], v [B, T, H, V], decay [B, T, H, D or 1]; `beta`: delta rule."""
    B, T, H, D = k.shape
    S = torch.zeros(B, H, D, v.shape[3], dtype=F64, device=k.device)
    out = torch.empty_like(v)
    for t in range(T):
        S = S * decay[:, t, :, :, None]
        u = v[:, t]
        if beta is not None:
            u = beta[:, t, :, None] * (u - (S * k[:, t, :, :, None]).sum(2))
        S = S + k[:, t, :, :, None] * u[:, :, None, :]
        out[:, t] = (S * q[:, t, :, :, None]).sum(2)
    return out


def _memory(q, k, v, ig, fg):
    B, T, H, D = k.shape
    S = torch.zeros(B, H, D, v.shape[3], dtype=F64, device=k.device)
    n, m = torch.zeros(B, H, D, dtype=F64, device=k.device), torch.zeros(B, H, dtype=F64, device=k.device)
    out = torch.empty_like(v)
    for t in range(T):
        new = torch.maximum(fg[:, t] + m, ig[:, t])
        keep, put, m = torch.exp(fg[:, t] + m - new), torch.exp(ig[:, t] - new), new
        S = keep[..., None, None] * S + (put[..., None] * k[:, t])[..., None] * v[:, t][:, :, None, :]
        n = keep[..., None] * n + put[..., None] * k[:, t]
        den = torch.maximum((n * q[:, t]).sum(-1).abs(), torch.exp(-m)) + 1e-6
        out[:, t] = (S * q[:, t][..., None]).sum(2) / den[..., None]
    return out


class _Part:
    """Tensors of one layer by their short names, in 64 bits, loaded when they are used."""

    def __init__(self, w, prefix):
        self.w, self.prefix = w, prefix

    def __call__(self, name):
        return self.w[self.prefix + name].to(F64)

    def __contains__(self, name):
        return self.prefix + name in self.w

    def lin(self, x, name):
        return x @ self(name).t()

    def heads(self, x, name, n):
        return self.lin(x, name).unflatten(-1, (n, -1))


def _mistral64(cfg, w, x):
    f = _powers(cfg.rope_theta, cfg.head_dim, x.device)
    for L in w["layers"]:
        p = _Part(L, "")
        h = _rms(x, cfg.rms_eps) * p("attn_norm")
        q, k, v = p.heads(h, "q", cfg.num_heads), p.heads(h, "k", cfg.num_kv_heads), p.heads(h, "v", cfg.num_kv_heads)
        o = _attend(_turn(q, f, False), _turn(k, f, False), v, cfg.head_dim ** -0.5)
        x = x + p.lin(o.flatten(2), "o")
        h = _rms(x, cfg.rms_eps) * p("ffn_norm")
        x = x + p.lin(_silu(p.lin(h, "gate")) * p.lin(h, "up"), "down")
    return _rms(x, cfg.rms_eps) * w["final_norm"].to(F64)


def _surodra64(d, w, x, _tokens):
    eps, mult = d["norm"]["eps"], d["residual_mult"]

    def norm(v, name):
        return torch.tanh(w[name + ".alpha"].to(F64) * v) * w[name].to(F64) + w[name + ".b"].to(F64)

    def freq(rot):
        return _powers(rot["base"], rot["dims"], x.device) / (rot.get("scaling") or {}).get("factor", 1.0)

    def gated(o, p, h, gain=None):
        o = _rms(o, eps) if gain is None else _rms(o, eps) * p(gain)
        return p.lin(o.flatten(2) * _silu(p.lin(h, "g")), "o")

    for i, L in enumerate(d["layers"]):
        m, h = L["mixer"], norm(x, f"l{i}.norm1")
        p = _Part(w, f"l{i}.mix.")
        if L["type"] == "delta":
            q, k, v = (_silu(_conv(p.lin(h, c), p(c + ".conv"))) for c in "qkv")
            rep = m["heads"] // m["kv_heads"]
            q, k = (t.unflatten(-1, (m["kv_heads"], -1)).repeat_interleave(rep, 2) for t in (q, k))
            q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
            g = torch.exp(-torch.exp(p("A_log")) * torch.nn.functional.softplus(p.lin(h, "a") + p("dt_bias")))
            o = _walk(q * m["dim"] ** -0.5, k, v.unflatten(-1, (m["heads"], -1)), g[..., None], torch.sigmoid(p.lin(h, "b")))
            y = gated(o, p, h, "norm")
        elif L["type"] == "retention":
            H = m["heads"]
            q, k = (_turn(p.heads(h, c, H), freq(m["rot"]), False) for c in "qk")
            decay = torch.tensor(m["decay"], dtype=F64, device=x.device).view(1, 1, H, 1).expand(*q.shape[:3], 1)
            y = gated(_walk(q, k * m["dim"] ** -0.5, p.heads(h, "v", H), decay), p, h)
        else:
            a, r, pl, pr = m["left"], m["right"], _Part(w, f"l{i}.mix.left."), _Part(w, f"l{i}.mix.right.")
            q, k = (_rms(pl.lin(h, c), eps) * pl(c + ".norm") for c in "qk")
            q, k = q.unflatten(-1, (a["heads"], -1)), k.unflatten(-1, (a["kv_heads"], -1))
            o = _attend(_turn(q, freq(a["rot"]), False), _turn(k, freq(a["rot"]), False), pl.heads(h, "v", a["kv_heads"]),
                        a["scale"], pl("sink")) * torch.sigmoid(pl.lin(h, "g"))[..., None]
            left = _rms(pl.lin(o.flatten(2), "o"), eps) * pl("out")
            H = r["heads"]
            z = pr.lin(pr.lin(h, "a1"), "a2") + pr("a2.b")
            decay = torch.exp(torch.nn.functional.logsigmoid(z) / r["tau"]).unflatten(-1, (H, -1))
            o = _walk(pr.heads(h, "q", H) * r["dim"] ** -0.5, pr.heads(h, "k", H), pr.heads(h, "v", H), decay)
            y = 0.5 * (left + _rms(gated(o, pr, h, "norm"), eps) * pr("out"))
        x = x + mult * y
        if L.get("mlp"):
            h, p = norm(x, f"l{i}.norm2"), _Part(w, f"l{i}.mlp.")
            x = x + mult * p.lin(_gelu(p.lin(h, "gate")) * p.lin(h, "up"), "down")
    return norm(x, "final.norm")


def _expert(p, name, h):
    return p.lin(_silu(p.lin(h, name + ".gate")) * p.lin(h, name + ".up"), name + ".down")


def _lobidra64(d, w, x, tokens):
    eps = d["norm"]["eps"]
    pos = torch.arange(x.shape[1], dtype=F64, device=x.device)
    for i, L in enumerate(d["layers"]):
        own, m, T = L.get("weights_of", i), L["mixer"], x.shape[1]
        n, p = _Part(w, f"l{own}."), _Part(w, f"l{own}.mix.")
        h = _rms(x, eps) * (1.0 + n("norm1"))
        if L["type"] == "attention":
            q, k = p.lin(h, "q"), p.lin(h, "k")
            if "q.conv" in p:
                q, k = _conv(q, p("q.conv")), _conv(k, p("k.conv"))
            q, k, f = q.unflatten(-1, (m["heads"], -1)), k.unflatten(-1, (m["kv_heads"], -1)), _band(m["rot"], x.device)
            o = _attend(_turn(q, f, True), _turn(k, f, True), k, m["scale"], torch.zeros(m["heads"], dtype=F64, device=x.device))
            y = p.lin((o * torch.sigmoid(p.lin(h, "g"))[..., None]).flatten(2), "o")
        else:
            a, r, pl, pr = m["left"], m["right"], _Part(w, f"l{own}.mix.left."), _Part(w, f"l{own}.mix.right.")
            t = a["q_temp"]
            temp = 1.0 + t["coef"] * torch.log(torch.floor((pos + 1.0) / t["every"]) + 1.0)
            o = _attend(pl.heads(h, "q", a["heads"]) * temp[None, :, None, None], pl.heads(h, "k", a["kv_heads"]),
                        pl.heads(h, "v", a["kv_heads"]), a["scale"], pl("sink")).flatten(2)
            y = m["left_scale"] * pl.lin(o * torch.sigmoid(pl.lin(h, "g")), "o")
            cap, H = r["gate_cap"], r["heads"]
            ig = cap * torch.tanh((pr.lin(h, "i") + pr("i.b")) / cap)
            fg = torch.nn.functional.logsigmoid(cap * torch.tanh((pr.lin(h, "f") + pr("f.b")) / cap))
            o = _memory(pr.heads(h, "q", H) * r["dim"] ** -0.5, pr.heads(h, "k", H), pr.heads(h, "v", H), ig, fg)
            o = _rms(o, eps).flatten(2) * pr("norm") * torch.sigmoid(pr.lin(h, "g"))
            y = y + m["right_scale"] * pr.lin(o, "o")
        x = x + _rms(y, eps) * (1.0 + n("norm1b"))
        f, p = L["mlp"], _Part(w, f"l{own}.mlp.")
        h = _rms(x, eps) * (1.0 + n("norm2"))
        if f["kind"] == "dense":
            y = p.lin(_gelu(p.lin(h, "up")), "down")
        else:
            chosen = w[f"l{own}.mlp.table"].long()[tokens].flatten(0, 1)
            flat = h.flatten(0, 1)
            y = _expert(p, "shared", flat) if f.get("shared") else torch.zeros_like(flat)
            for e in range(f["router"]["experts"]):
                sel = (chosen == e).any(-1).nonzero()[:, 0]
                if len(sel):
                    y[sel] += _expert(p, f"e{e}", flat[sel]) / f["router"]["top"]
            y = y.view_as(h)
        x = x + _rms(y, eps) * (1.0 + n("norm2b"))
    return _rms(x, eps) * (1.0 + w["final.norm"].to(F64))


def _kagorax64(d, w, x, _tokens):
    eps, T, W = d["norm"]["eps"], x.shape[1], x.shape[2]
    i = torch.arange(T, device=x.device)
    ang = i.to(F64)[:, None] * _powers(10000.0, W, x.device)
    x = x + torch.stack([ang.sin(), ang.cos()], -1).flatten(1)
    kvs = {}
    for n, L in enumerate(d["layers"]):
        m, p = L["mixer"], _Part(w, f"l{n}.mix.")
        h = _rms(x, eps) * w[f"l{n}.norm1"].to(F64)
        q = _rms((p.lin(h, "q") + p("q.b")).unflatten(-1, (m["heads"], -1)), eps)
        src = m.get("kv_from", n)
        if src == n:
            kvs[n] = (_rms((p.lin(h, "k") + p("k.b")).unflatten(-1, (m["kv_heads"], -1)), eps),
                      (p.lin(h, "v") + p("v.b")).unflatten(-1, (m["kv_heads"], -1)))
        rel, far = p("rel"), m["bias_max"]
        half, rows = rel.shape[0] // 2, rel.shape[0]
        row = [t if t < half else min(rows - 1, half + math.floor(math.log(t / half) / math.log(far / half) * (rows - half) + 1e-9))
               for t in range(T)]
        gap = i[:, None] - i[None, :]
        seen = gap >= 0
        if m.get("mask"):
            seen = seen & ((gap < m["mask"]["size"]) | (i[None, :] < m["mask"].get("keep_first", 0)))
        o = _attend(q, *kvs[src], m["scale"], bias=rel[torch.tensor(row, device=x.device)].t().contiguous(), seen=seen)
        y = p.lin(o.flatten(2) * torch.sigmoid(p.lin(h, "g")), "o")
        f, p, flat = L["mlp"], _Part(w, f"l{n}.mlp."), h.flatten(0, 1)
        val, idx = torch.sigmoid(p.lin(flat, "router")).topk(f["router"]["top"], dim=-1)
        z = torch.sigmoid(p.lin(flat, "shared.sg")) * _expert(p, "shared", flat)
        for e in range(f["router"]["experts"]):
            hit = idx == e
            sel = hit.any(-1).nonzero()[:, 0]
            if len(sel):
                z[sel] += _expert(p, f"e{e}", flat[sel] * (val * hit).sum(-1)[sel, None])
        x = x + y + z.view_as(h)
    return _rms(x, eps) * w["final.norm"].to(F64)


def _muderax64(d, w, x, _tokens):
    eps, T = d["norm"]["eps"], x.shape[1]
    i = torch.arange(T, device=x.device)
    gap = i[:, None] - i[None, :]
    for n, L in enumerate(d["layers"]):
        own, m = L.get("weights_of", n), L["mixer"]
        p = _Part(w, f"l{own}.mix.")
        if L["type"] == "latent_attention":
            H, dn, rk, rot = m["heads"], m["dim"], m["kv_rank"], m["rot"]
            freq, amp, s = _powers(rot["base"], rot["dims"], x.device), 1.0, rot.get("scaling")
            if s:  # frequencies blended between two turn counts, an amplitude on the rotated part
                at = [rot["dims"] * math.log(s["original"] / (2.0 * math.pi * s[k])) / (2.0 * math.log(rot["base"]))
                      for k in ("fast", "slow")]
                lo, hi = max(math.floor(at[0]), 0), min(math.ceil(at[1]), rot["dims"] - 1)
                ramp = ((torch.arange(len(freq), dtype=F64, device=x.device) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
                freq, amp = freq / s["factor"] * ramp + freq * (1.0 - ramp), 0.1 * math.log(s["factor"]) + 1.0

            def turned(v):
                out = _turn(v, freq, True)
                out[..., :rot["dims"]] *= amp
                return out

            q, c = p.heads(x, "q", H), p.lin(x, "dkv")
            lat = _rms(c[..., :rk], eps) * p("dkv.norm")
            key = torch.cat([p.heads(lat, "uk", H), turned(c[:, :, None, rk:]).expand(-1, -1, H, -1)], -1)
            q = torch.cat([q[..., :dn], turned(q[..., dn:])], -1)
            seen = (gap >= 0) & (gap < (m.get("mask") or {}).get("size", 1 << 30))
            y = p.lin(_attend(q, key, p.heads(lat, "uv", H), m["scale"], seen=seen).flatten(2), "o")
        else:
            branch = _gelu(p.lin(x, "y") + p("y.b"))
            u = _conv(p.lin(x, "x") + p("x.b"), p("conv")) + p("conv.b")
            ub = u.unflatten(-1, (m["blocks"], -1))
            r, g = (torch.sigmoid(torch.stack([ub[:, :, b] @ p(c)[b].t() for b in range(m["blocks"])], 2) + p(c + ".b")).flatten(2)
                    for c in ("ra", "ri"))
            a = torch.exp(-8.0 * r * torch.nn.functional.softplus(p("lam")))
            drive, state, out = torch.sqrt(1.0 - a * a) * g * u, torch.zeros_like(u[:, 0]), torch.empty_like(u)
            for t in range(T):
                state = a[:, t] * state + drive[:, t]
                out[:, t] = state
            y = p.lin(out * branch, "o")
        x = x + _rms(y, eps) * w[f"l{own}.norm1"].to(F64)
        f, p, flat = L["mlp"], _Part(w, f"l{own}.mlp."), x.flatten(0, 1)
        val, idx = (p.lin(flat, "router") + p("router.b")).topk(f["router"]["top"], dim=-1)
        z, val = _expert(p, "shared", flat), torch.softmax(val, -1)
        for e in range(f["router"]["experts"]):
            hit = idx == e
            sel = hit.any(-1).nonzero()[:, 0]
            if len(sel):
                z[sel] += _expert(p, f"e{e}", flat[sel]) * (val * hit).sum(-1)[sel, None]
        x = x + _rms(z.view_as(x), eps) * w[f"l{own}.norm2"].to(F64)
    return _rms(x, eps) * w["final.norm"].to(F64)


@torch.no_grad()
def exact(case, seed):
    """The logits by whole sequences in 64 bits."""
    fam, cfg, _ = registry.resolve(case["model"])
    lens = [n + (case["kind"] != "prompt") for n in _lengths(case)]
    shared, experts, _, top = _matrices(fam, cfg)
    if 2.0 * (shared + top * sum(experts)) * len(lens) * max(lens) > EXACT_FLOPS:
        return None
    w = _checkpoint(fam, cfg, DTYPES[case["dtype"]], seed)
    toks = _tokens(case, cfg, seed)
    want = _want(lens) if case["kind"] == "prompt" else [[n - 1] for n in lens]
    out = []
    for at in range(0, len(lens), 16):  # sequences side by side, shorter ones padded at the end
        part = list(range(at, min(len(lens), at + 16)))
        T = max(lens[i] for i in part)
        ids = torch.tensor([toks[i][:lens[i]] + [0] * (T - lens[i]) for i in part], device="cuda")
        if fam.name == "mistral":
            x = _mistral64(cfg, w, w["embed"][ids].to(F64))
        else:
            d = cfg.to_dict()
            walk = {"surodra": _surodra64, "lobidra": _lobidra64, "kagorax": _kagorax64, "muderax": _muderax64}[fam.name]
            x = walk(d, w, w["embed"][ids].to(F64) * (d.get("embedding") or {}).get("scale", 1.0), ids)
        rows = torch.cat([x[j, want[i]] for j, i in enumerate(part)])
        head = w["lm_head" if fam.name == "mistral" else "head" if "head" in w else "embed"].to(F64)
        z = rows @ head.t().contiguous()
        if fam.name == "surodra":
            z = d["logit_softcap"] * torch.tanh(z * d["logit_scale"] / d["logit_softcap"])
        out.append(z)
    return torch.cat(out)
