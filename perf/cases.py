"""The work that this framework is used for, as calls that can be timed and checked.

`listed()` names twelve calls: the quantized linears of a Qwen3-4B decoder layer from one
token to a long prefill chunk, paged decode attention over 8-bit caches, the OLMoE expert
layer at decode and prefill sizes, and one whole decode step of a small decoder. `draw(rng)`
gives further calls of the same ranges. A case goes through `prepare` (what a serving program
holds before the call: quantized modules, caches, tables, inputs), `run` (one call), `exact`
(the same result in 64 bits from plain torch formulas) and `work` / `tolerance`.
"""
import math
import os
import sys
import types

import torch
from torch import nn

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mini-inference_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from engine.core.kv_cache import KVCache  # noqa: E402
from engine.core.model_runner import ModelRunner, Request  # noqa: E402
from engine.quantization import get_method  # noqa: E402
from engine.quantization.modules import QuantExperts, QuantLinear  # noqa: E402
from kernels.paged_attention import paged_decode_attention  # noqa: E402

DEV = "cuda"
GROUP = 128        # INT4 quantization group
PAGE = 16          # tokens per KV page
HEAD_DIM = 128
BF16_BYTES = 2

# (N, K) of the linears: Qwen3-4B (hidden 2560, MLP 9728, 32 + 8 + 8 heads of 128) ...
SHAPES = {"qkv": (6144, 2560), "o": (2560, 4096), "gate_up": (19456, 2560), "down": (2560, 9728)}
# ... and the expert layer: OLMoE-1B-7B (hidden 2048, expert MLP 1024, 64 experts, top 8)
MOE = {"H": 2048, "I": 1024, "E": 64, "k": 8}


def _linear(name, method, shape, M):
    N, K = SHAPES[shape]
    return {"name": name, "kind": "linear", "method": method, "M": M, "N": N, "K": K}


def listed():
    return [
        # one user, one token at a time: the smallest call of a step
        _linear("int4_down_m1", "int4_wo", "down", 1),
        # a ragged decode batch of a busy server
        _linear("int4_down_m48", "int4_wo", "down", 48),
        # the widest linear of a full decode batch
        _linear("int8_gate_up_m64", "int8_wo", "gate_up", 64),
        # FP8 weights and activations in a small decode batch
        _linear("fp8_qkv_m16", "fp8", "qkv", 16),
        # a prompt of odd length (prefill)
        _linear("int4_down_m1000", "int4_wo", "down", 1000),
        # the largest call: a long prefill chunk through the widest linear
        _linear("int8_gate_up_m2048", "int8_wo", "gate_up", 2048),
        # FP8 prefill
        _linear("fp8_qkv_m2048", "fp8", "qkv", 2048),
        # a full decode batch with contexts of every length
        {"name": "paged_fp8_b64", "kind": "paged", "kv": "fp8", "B": 64, "lo": 512, "hi": 8192, "heads": 32, "kv_heads": 8},
        # a few users with long documents
        {"name": "paged_int8_b3_long", "kind": "paged", "kv": "int8", "B": 3, "lo": 12000, "hi": 32768, "heads": 32,
         "kv_heads": 8},
        # expert layer of a decode batch
        {"name": "moe_int4_t64", "kind": "moe", "method": "int4_wo", "T": 64},
        # expert layer of a prompt (prefill)
        {"name": "moe_int8_t1000", "kind": "moe", "method": "int8_wo", "T": 1000},
        # a whole decode step, metadata to logits: INT4 linears, FP8 cache
        {"name": "decode_step_b16", "kind": "step", "method": "int4_wo", "kv": "fp8", "B": 16, "lo": 512, "hi": 4096},
    ]


def _log_int(rng, lo, hi):
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "paged", "moe", "step"])
    if kind == "linear":
        M = _log_int(rng, 1, 2048)
        if rng.random() < 0.4:
            N, K = SHAPES[rng.choice(sorted(SHAPES))]
        else:  # other widths that the formats take
            N = 16 * _log_int(rng, 16, 768)
            K = 128 * _log_int(rng, 4, min(76, 19456 * 2560 // (128 * N)))
        return {"kind": kind, "method": rng.choice(["int4_wo", "int8_wo", "fp8"]), "M": M, "N": N, "K": K}
    if kind == "paged":
        B = _log_int(rng, 1, 64)
        hi = _log_int(rng, 64, min(32768, 400000 // B))
        kv_heads = rng.choice([4, 8, 16])
        return {"kind": kind, "kv": rng.choice(["fp8", "int8"]), "B": B, "lo": max(1, hi // rng.choice([1, 4, 16])), "hi": hi,
                "heads": kv_heads * rng.choice([1, 2, 4]), "kv_heads": kv_heads}
    if kind == "moe":
        return {"kind": kind, "method": rng.choice(["int4_wo", "int8_wo", "fp8"]), "T": _log_int(rng, 1, 1000)}
    hi = _log_int(rng, 64, 4096)
    return {"kind": kind, "method": rng.choice(["int4_wo", "int8_wo"]), "kv": rng.choice(["fp8", "int8"]),
            "B": _log_int(rng, 1, 32), "lo": max(2, hi // 8), "hi": hi}


# ------------------------------------------------------------------ inputs, from the seed alone
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, std=1.0):
    """bf16 normal values, drawn in bounded pieces so that large weights need no fp32 copy."""
    out = torch.empty(shape, dtype=torch.bfloat16, device=DEV)
    for piece in out.view(-1).split(1 << 26):
        piece.copy_(torch.randn(piece.numel(), generator=g, device=DEV) * std)
    return out


def _linear_inputs(case, seed):
    g = _gen(seed)
    return _randn(g, case["M"], case["K"]), _randn(g, case["N"], case["K"], std=0.02)


def _contexts(case, seed):
    g = torch.Generator().manual_seed(int(seed) + 1)
    lens = torch.randint(case["lo"], case["hi"] + 1, (case["B"],), generator=g)
    lens[0] = case["hi"]
    return lens


def _paged_inputs(case, seed):
    """q, K and V by slot, the shuffled block table and the context lengths."""
    g, lens = _gen(seed), _contexts(case, seed)
    pages = [-(-int(n) // PAGE) for n in lens]
    perm = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(int(seed) + 2)).to(torch.int32)
    table = torch.zeros(case["B"], max(pages), dtype=torch.int32)
    at = 0
    for b, n in enumerate(pages):
        table[b, :n] = perm[at:at + n]
        at += n
    q = _randn(g, case["B"], case["heads"], HEAD_DIM)
    k, v = (_randn(g, sum(pages) * PAGE, case["kv_heads"], HEAD_DIM) for _ in range(2))
    return q, k, v, table, lens


def _moe_inputs(case, seed):
    g, m = _gen(seed), MOE
    x = _randn(g, case["T"], m["H"])
    gate_up = _randn(g, m["E"], 2 * m["I"], m["H"], std=0.02)
    down = _randn(g, m["E"], m["H"], m["I"], std=0.02)
    router = _randn(g, m["E"], m["H"], std=0.02)
    probs = (x.float() @ router.float().t()).softmax(-1)
    weights, ids = probs.topk(m["k"], dim=-1)
    return x, gate_up, down, ids, weights.to(torch.bfloat16)


# the decoder of the whole step: two layers of Qwen3-4B's widths, a short vocabulary
STEP = {"layers": 2, "hidden": 2560, "mlp": 9728, "heads": 32, "kv_heads": 8, "vocab": 8192, "theta": 1e6, "eps": 1e-6}
_STEP_LINEARS = {"q_proj": ("heads", "hidden"), "k_proj": ("kv_heads", "hidden"), "v_proj": ("kv_heads", "hidden"),
                 "o_proj": ("hidden", "heads"), "gate_proj": ("mlp", "hidden"), "up_proj": ("mlp", "hidden"),
                 "down_proj": ("hidden", "mlp")}


def _width(key):
    return STEP[key] * (HEAD_DIM if key in ("heads", "kv_heads") else 1)


def _step_inputs(case, seed):
    g, lens = _gen(seed), _contexts(case, seed)
    weights = [{name: _randn(g, _width(n), _width(k), std=0.02) for name, (n, k) in _STEP_LINEARS.items()}
               for _ in range(STEP["layers"])]
    embed, head = (_randn(g, STEP["vocab"], STEP["hidden"], std=s) for s in (1.0, 0.02))
    past = sum(int(n) - 1 for n in lens)
    kv = [tuple(_randn(g, past, STEP["kv_heads"], HEAD_DIM) for _ in range(2)) for _ in range(STEP["layers"])]
    tokens = torch.randint(0, STEP["vocab"], (case["B"],), generator=torch.Generator().manual_seed(int(seed) + 2))
    return weights, embed, head, kv, tokens.tolist(), [int(n) for n in lens]


# ------------------------------------------------------------------ the decoder's modules
class _Rotary(nn.Module):
    def __init__(self):
        super().__init__()
        inv = STEP["theta"] ** (-torch.arange(0, HEAD_DIM, 2, device=DEV).float() / HEAD_DIM)
        self.register_buffer("inv", inv)

    def forward(self, x, positions):
        angle = positions[..., None].float() * self.inv
        angle = torch.cat((angle, angle), dim=-1)
        return angle.cos().to(x.dtype), angle.sin().to(x.dtype)


class _Mlp(nn.Module):
    def forward(self, x):
        return self.down_proj(nn.functional.silu(self.gate_proj(x)) * self.up_proj(x))


def _norm(width):
    return nn.RMSNorm(width, eps=STEP["eps"], device=DEV, dtype=torch.bfloat16)


def _linear_module(weight, method=None):
    lin = nn.Linear(weight.shape[1], weight.shape[0], bias=False, device="meta")
    lin.weight = nn.Parameter(weight, requires_grad=False)
    return lin if method is None else QuantLinear(lin, method)


def _decoder(weights, embed, head, method):
    model, inner = nn.Module(), nn.Module()
    inner.embed_tokens = nn.Embedding.from_pretrained(embed)
    inner.layers = nn.ModuleList()
    for w in weights:
        layer, attn, layer_mlp = nn.Module(), nn.Module(), _Mlp()
        for name, tensor in w.items():
            setattr(layer_mlp if name in ("gate_proj", "up_proj", "down_proj") else attn, name, _linear_module(tensor, method))
        attn.q_norm, attn.k_norm, attn.scaling = _norm(HEAD_DIM), _norm(HEAD_DIM), HEAD_DIM ** -0.5
        layer.self_attn, layer.mlp = attn, layer_mlp
        layer.input_layernorm, layer.post_attention_layernorm = _norm(STEP["hidden"]), _norm(STEP["hidden"])
        inner.layers.append(layer)
    inner.norm, inner.rotary_emb = _norm(STEP["hidden"]), _Rotary()
    model.model, model.lm_head, model.config = inner, _linear_module(head), types.SimpleNamespace()
    return model


# ------------------------------------------------------------------ prepare and run
def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, w = _linear_inputs(case, seed)
        return {"kind": kind, "layer": _linear_module(w, get_method(case["method"], device=DEV, group_size=GROUP)), "x": x}
    if kind == "paged":
        q, k, v, table, lens = _paged_inputs(case, seed)
        cache = KVCache("paged", 1, case["kv_heads"], HEAD_DIM, k.shape[0], torch.bfloat16, DEV, block_size=PAGE,
                        kv_dtype=case["kv"])
        cache.write(0, torch.arange(k.shape[0], device=DEV), k, v)
        return {"kind": kind, "q": q, "cache": cache, "table": table.to(DEV), "lens": lens.to(torch.int32).to(DEV),
                "max_len": int(lens.max())}
    if kind == "moe":
        x, gate_up, down, ids, weights = _moe_inputs(case, seed)
        experts = nn.Module()
        experts.act_fn = nn.SiLU()
        experts.gate_up_proj = nn.Parameter(gate_up, requires_grad=False)
        experts.down_proj = nn.Parameter(down, requires_grad=False)
        layer = QuantExperts(experts, get_method(case["method"], device=DEV, group_size=GROUP))
        return {"kind": kind, "layer": layer, "x": x, "ids": ids, "weights": weights}
    weights, embed, head, kv, tokens, lens = _step_inputs(case, seed)
    model = _decoder(weights, embed, head, get_method(case["method"], device=DEV, group_size=GROUP))
    capacity = sum(-(-n // PAGE) * PAGE for n in lens)
    cache = KVCache("paged", STEP["layers"], STEP["kv_heads"], HEAD_DIM, capacity, torch.bfloat16, DEV, block_size=PAGE,
                    kv_dtype=case["kv"])
    chunks, slots = [], []
    for i, (n, token) in enumerate(zip(lens, tokens)):
        req = Request([0] * (n - 1) + [token], 1, rid=i)
        cache.admit(req, n, n)
        cache.ensure(req, n)
        chunks.append((req, n - 1, n))
        slots.append(cache.slots(req, 0, n - 1))
    slots = torch.cat(slots).to(DEV)
    for layer, (k, v) in enumerate(kv):
        cache.write(layer, slots, k, v)
    arch = {"architecture": "Qwen3ForCausalLM", "qk_norm": "per_head", "moe": False, "heads": STEP["heads"],
            "kv_heads": STEP["kv_heads"], "head_dim": HEAD_DIM}
    return {"kind": kind, "runner": ModelRunner(model, cache, arch=arch), "chunks": chunks}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "paged":
        c = state["cache"]
        return paged_decode_attention(state["q"], c.k[0], c.v[0], state["table"], state["lens"], PAGE, HEAD_DIM ** -0.5,
                                      state["max_len"], k_scale=c.k_scale[0], v_scale=c.v_scale[0])
    if kind == "moe":
        return state["layer"](state["x"], state["ids"], state["weights"])
    return state["runner"].forward(state["chunks"])


# ------------------------------------------------------------------ what a call cannot do without
def _weight_bytes(method, N, K):
    if method == "int4_wo":  # codes, and a bf16 scale and zero per group
        return N * K // 2 + 2 * N * (K // GROUP) * BF16_BYTES
    return N * K + N * (4 if method == "fp8" else BF16_BYTES)


def _kv_bytes(tokens, kv_heads):
    return 2 * tokens * kv_heads * (HEAD_DIM + BF16_BYTES)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": _weight_bytes(case["method"], N, K) + (M * K + M * N) * BF16_BYTES, "flops": 2 * M * N * K}
    if kind == "paged":  # (the contexts' expected length: the drawn ones depend on the seed)
        tokens = case["hi"] + (case["B"] - 1) * (case["lo"] + case["hi"]) / 2
        return {"bytes": _kv_bytes(tokens, case["kv_heads"]) + 2 * case["B"] * case["heads"] * HEAD_DIM * BF16_BYTES,
                "flops": 4 * tokens * case["heads"] * HEAD_DIM}
    if kind == "moe":
        T, m = case["T"], MOE
        touched = m["E"] * (1 - (1 - m["k"] / m["E"]) ** T)
        expert = _weight_bytes(case["method"], 2 * m["I"], m["H"]) + _weight_bytes(case["method"], m["H"], m["I"])
        return {"bytes": touched * expert + 2 * T * m["H"] * BF16_BYTES + T * m["k"] * 10,
                "flops": 6 * T * m["k"] * m["H"] * m["I"]}
    B, L = case["B"], STEP["layers"]
    shapes = [(_width(n), _width(k)) for n, k in _STEP_LINEARS.values()]
    tokens = case["hi"] + (B - 1) * (case["lo"] + case["hi"]) / 2
    head = STEP["vocab"] * STEP["hidden"]
    return {"bytes": L * (sum(_weight_bytes(case["method"], n, k) for n, k in shapes) + _kv_bytes(tokens, STEP["kv_heads"]))
            + head * BF16_BYTES + B * STEP["vocab"] * 4,
            "flops": L * (sum(2 * B * n * k for n, k in shapes) + 4 * tokens * STEP["heads"] * HEAD_DIM) + 2 * B * head}


def tolerance(case):
    """About four times what two correct orders of the same sums, each rounded to bf16, and
    weights rounded once to bf16 show against 64 bits."""
    if case["kind"] == "linear":
        return {"rel": 1e-2, "max": 4e-2}
    if case["kind"] == "paged":
        return {"rel": 1e-2, "max": 4e-2}
    if case["kind"] == "moe":
        # bf16 gate, up, product, down and eight bf16 additions; FP8 re-quantizes the product
        return {"rel": 2e-2, "max": 1e-1}
    return {"rel": 2e-2, "max": 1.5e-1}


# ------------------------------------------------------------------ the same results in 64 bits
def _div(a, b):
    """fp32 quotient, correctly rounded (a device division by a constant may multiply by its
    reciprocal, and a quantizer's ties then fall the other way)."""
    return (a.double() / b).float()


def _dequantized(method, w):
    """The quantized weight's value in 64 bits, from the formats' formulas."""
    f = w.float()
    if method == "int4_wo":
        grp = f.unflatten(-1, (-1, GROUP))
        lo, hi = grp.amin(-1, keepdim=True), grp.amax(-1, keepdim=True)
        s = _div(hi - lo, 15.0).clamp(min=1e-8)
        q = _div(grp - lo, s).round().clamp(0, 15)
        return (q.double() * s.bfloat16().double() + lo.bfloat16().double()).flatten(-2)
    if method == "int8_wo":
        s = _div(f.abs().amax(-1, keepdim=True).clamp(min=1e-8), 127.0)
        return _div(f, s).round().clamp(-127, 127).double() * s.bfloat16().double()
    return _fp8_rows(f)


def _fp8_rows(f):
    s = _div(f.abs().amax(-1, keepdim=True).clamp(min=1e-12), 448.0)
    return _div(f, s).clamp(-448, 448).to(torch.float8_e4m3fn).double() * s.double()


def _times(method, x, w64):
    """x (64 bits, rounded to bf16 first where the format quantizes activations) @ w^T."""
    return (_fp8_rows(x.bfloat16().float()) if method == "fp8" else x) @ w64.t()


def _kv64(kv, x):
    """Cached value of bf16 rows x [.., D]: per-row scale rounded to bf16, then the code."""
    f, qmax = x.float(), 127.0 if kv == "int8" else 448.0
    s = _div(f.abs().amax(-1, keepdim=True), qmax).clamp(min=1e-8).bfloat16()
    q = _div(f, s.double()).clamp(-qmax, qmax)
    q = q.round() if kv == "int8" else q.to(torch.float8_e4m3fn)
    return q.double() * s.double()


def _attend(q, k, v, scale):
    """q [H, D] over k, v [n, KV, D], all in 64 bits."""
    rep = q.shape[0] // k.shape[1]
    k, v = (t.permute(1, 0, 2) for t in (k, v))                     # [KV, n, D]
    p = ((q.view(k.shape[0], rep, -1) @ k.transpose(1, 2).contiguous()) * scale).softmax(-1)
    return (p @ v.contiguous()).reshape(q.shape)


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, w = _linear_inputs(case, seed)
        return _times(case["method"], x.double(), _dequantized(case["method"], w))
    if kind == "paged":
        q, k, v, table, lens = _paged_inputs(case, seed)
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        for b, n in enumerate(lens.tolist()):
            slots = (table[b].long()[:, None] * PAGE + torch.arange(PAGE)).view(-1)[:n].to(DEV)
            out[b] = _attend(q[b].double(), _kv64(case["kv"], k[slots]), _kv64(case["kv"], v[slots]), HEAD_DIM ** -0.5)
        return out
    if kind == "moe":
        x, gate_up, down, ids, weights = _moe_inputs(case, seed)
        out = torch.zeros(x.shape, dtype=torch.float64, device=DEV)
        for e in range(MOE["E"]):
            tok, slot = (ids == e).nonzero(as_tuple=True)
            if not len(tok):
                continue
            gu = _times(case["method"], x[tok].double(), _dequantized(case["method"], gate_up[e]))
            gate, up = gu.chunk(2, dim=-1)
            y = _times(case["method"], nn.functional.silu(gate) * up, _dequantized(case["method"], down[e]))
            out.index_add_(0, tok, y * weights[tok, slot, None].double())
        return out
    return _exact_step(case, seed)


def _rms(x):
    return x * (x.square().mean(-1, keepdim=True) + STEP["eps"]).rsqrt()


def _exact_step(case, seed):
    weights, embed, head, kv, tokens, lens = _step_inputs(case, seed)
    method, B = case["method"], case["B"]
    x = embed[torch.tensor(tokens, device=DEV)].double()
    pos = torch.tensor(lens, device=DEV).double() - 1
    inv = STEP["theta"] ** (-torch.arange(0, HEAD_DIM, 2, device=DEV).double() / HEAD_DIM)
    angle = torch.cat((pos[:, None] * inv,) * 2, dim=-1)[:, None, :]
    cos, sin = angle.cos(), angle.sin()

    def rope(t):
        lo, hi = t.chunk(2, dim=-1)
        return t * cos + torch.cat((-hi, lo), dim=-1) * sin

    for w, (past_k, past_v) in zip(weights, kv):
        def lin(name, t):
            return _times(method, t, _dequantized(method, w[name]))
        h = _rms(x)
        q, k, v = (lin(n, h).view(B, -1, HEAD_DIM) for n in ("q_proj", "k_proj", "v_proj"))
        q, k = rope(_rms(q)), rope(_rms(k))
        k, v = (_kv64(case["kv"], t.bfloat16()) for t in (k, v))
        att, at = [], 0
        for b, n in enumerate(lens):
            pk, pv = (_kv64(case["kv"], p[at:at + n - 1]) for p in (past_k, past_v))
            at += n - 1
            att.append(_attend(q[b], torch.cat((pk, k[b:b + 1])), torch.cat((pv, v[b:b + 1])), HEAD_DIM ** -0.5))
        x = x + lin("o_proj", torch.stack(att).flatten(1))
        h = _rms(x)
        x = x + lin("down_proj", nn.functional.silu(lin("gate_proj", h)) * lin("up_proj", h))
    return _rms(x) @ head.double().t()
