"""The calls that a user of this package has it make, with the sizes they come in.

Each case is one pass through the public functions of nanovllm_hip.kernels (and, for the whole decode step, through the
model of nanovllm_hip.harness.qwen3), on inputs as a serving loop holds them: strided views of the qkv projection, a
paged KV cache with scattered 256-slot blocks, ragged lengths. The shapes are those of the package's model
configuration (hidden 1024, MLP 3072, 16 query and 8 kv heads of 128) and, among the drawn cases, the widths and head
counts that its tests use.
"""
import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-vllm-triton-kernels_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from nanovllm_hip import kernels as hip  # noqa: E402
from nanovllm_hip.harness.qwen3 import Context, Qwen3, Qwen3Config, rope_table  # noqa: E402
from nanovllm_hip.kernels.attention import (flash_attn_varlen_func, flash_attn_with_kvcache,  # noqa: E402
                                            qk_norm_rope_kv_decode_attention)

BF16 = torch.bfloat16
DEV = "cuda:0"
EPS = 1e-6
BLOCK = 256          # tokens per KV-cache block
VOCAB = 151936
MAX_POS = 40960
THETA = 1e6
D = 128

SMALL = {"hidden": 1024, "inter": 3072, "hq": 16, "hkv": 8}     # the package's model configuration
WIDE = {"hidden": 2048, "inter": 6144, "hq": 16, "hkv": 8}      # hidden 2048: the widest its fused norms take


def listed():
    return [
        # One request being decoded, run eagerly layer by layer: the smallest calls, where every launch is latency.
        {"name": "decode_layer_1", "kind": "decode_layer", "batch": 1, "lo": 700, "hi": 700, **SMALL},
        # The decode step of a server with 32 requests: 28 layers, LM head and greedy pick, replayed from a HIP graph.
        {"name": "decode_step_32", "kind": "decode_step", "batch": 32, "lo": 512, "hi": 2048, "layers": 28},
        # The attention of a large decode batch with ragged contexts: all KV-cache bandwidth.
        {"name": "decode_attention_250", "kind": "decode_attention", "batch": 250, "lo": 40, "hi": 4096, "hq": 16,
         "hkv": 8},
        # The LM head and greedy pick of such a batch.
        {"name": "lm_head_250", "kind": "lm_head", "rows": 250, "vocab": VOCAB, "hidden": 1024},
        # A prefill batch of ragged prompts without a cached prefix.
        {"name": "prefill_attention_24", "kind": "prefill_attention", "seqs": 24, "lo": 30, "hi": 2100, "hq": 16,
         "hkv": 8},
        # A chunk of a long prompt over the prefix that is cached already.
        {"name": "chunk_attention_2048", "kind": "mixed_attention", "decodes": 0, "lo": 0, "hi": 0, "chunk": 2048,
         "prefix": 14001, "hq": 16, "hkv": 8},
        # A mixed step: decode requests and one prompt chunk in a single call over the paged cache.
        {"name": "mixed_attention_512", "kind": "mixed_attention", "decodes": 48, "lo": 512, "hi": 2048,
         "chunk": 464, "prefix": 1000, "hq": 16, "hkv": 8},
        # Norm, qkv projection and the fused q/k norm + RoPE + KV write of a prefill batch with an odd token count.
        {"name": "pre_attn_4099", "kind": "pre_attn", "tokens": 4099, **SMALL},
        # o_proj, norm, MLP and the next norm of a small ragged prefill...
        {"name": "post_attn_777", "kind": "post_attn", "tokens": 777, **SMALL},
        # ... and of the largest batch of prompt tokens.
        {"name": "post_attn_16384", "kind": "post_attn", "tokens": 16384, **SMALL},
        # The memory-bound kernels on their own, as the layers call them around another library's projections.
        {"name": "elementwise_8192", "kind": "elementwise", "tokens": 8192, **SMALL},
        # The GEMM on fp32 inputs (row-major operands).
        {"name": "matmul_fp32_4096", "kind": "matmul", "m": 4096, "n": 4096, "k": 4096, "dtype": "fp32",
         "precision": "ieee", "b_rows": "k"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode_layer", "decode_attention", "lm_head", "prefill_attention", "mixed_attention",
                       "pre_attn", "post_attn", "elementwise", "matmul"])
    model = rng.choice([SMALL, SMALL, WIDE])
    heads = rng.choice([{"hq": 16, "hkv": 8}, {"hq": 16, "hkv": 8}, {"hq": 32, "hkv": 8}, {"hq": 16, "hkv": 4}])
    if kind == "decode_layer":
        lo = _log(rng, 20, 1000)
        return {"kind": kind, "batch": _log(rng, 1, 128), "lo": lo, "hi": lo + _log(rng, 1, 3000), **model}
    if kind == "decode_attention":
        lo = _log(rng, 1, 1000)
        return {"kind": kind, "batch": _log(rng, 1, 250), "lo": lo, "hi": lo + _log(rng, 1, 3000), **heads}
    if kind == "lm_head":
        return {"kind": kind, "rows": _log(rng, 1, 250), "vocab": VOCAB, "hidden": 1024}
    if kind == "prefill_attention":
        lo = _log(rng, 1, 500)
        return {"kind": kind, "seqs": _log(rng, 1, 24), "lo": lo, "hi": lo + _log(rng, 1, 1600), **heads}
    if kind == "mixed_attention":
        lo = _log(rng, 1, 1000)
        return {"kind": kind, "decodes": rng.choice([0, 1, 7, 16, 48]), "lo": lo, "hi": lo + _log(rng, 1, 2000),
                "chunk": _log(rng, 32, 2048), "prefix": _log(rng, 1, 13000), **heads}
    if kind == "pre_attn":
        return {"kind": kind, "tokens": _log(rng, 33, 8192), **model}
    if kind == "post_attn":
        return {"kind": kind, "tokens": _log(rng, 33, 16384 if model is SMALL else 4096), **model}
    if kind == "elementwise":
        return {"kind": kind, "tokens": _log(rng, 1, 8192), **SMALL}
    dtype = rng.choice(["fp32", "fp32", "bf16"])
    m, n, k = (8 * _log(rng, 8, 500) for _ in range(3))
    return {"kind": kind, "m": m + rng.choice([0, 0, 1, 5]), "n": n, "k": k, "dtype": dtype,
            "precision": rng.choice(["ieee", "tf32"]), "b_rows": rng.choice(["k", "n"])}


# ------------------------------------------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, scale=1.0, dtype=BF16):
    x = torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)
    return (x * scale).to(dtype)


def _norm_w(g, n):
    return (1 + 0.1 * torch.randn(n, generator=g, device=DEV)).to(BF16)


def _lengths(n, lo, hi):
    """n lengths from lo to hi, evenly spread, in an order that depends on nothing but these numbers."""
    if n == 0:
        return []
    spread = [hi] if n == 1 else [lo + (hi - lo) * i // (n - 1) for i in range(n)]
    random.Random(n * 1000003 + lo * 1009 + hi).shuffle(spread)
    return spread


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def _paged(g, lengths, hkv, fill=True):
    """A paged cache in which every sequence owns scattered blocks for its length, and its block table."""
    need = [(n + BLOCK - 1) // BLOCK for n in lengths]
    total = sum(need) + 3
    order = torch.randperm(total, generator=g, device=DEV).to(torch.int32)
    table = torch.full((len(lengths), max(need)), -1, dtype=torch.int32, device=DEV)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = order[at:at + n]
        at += n
    shape = (total, BLOCK, hkv, D)
    k, v = (_randn(g, *shape) if fill else torch.zeros(shape, dtype=BF16, device=DEV) for _ in range(2))
    return k, v, table


def _slots(table, seq, pos):
    seq, pos = torch.tensor(seq, device=DEV), torch.tensor(pos, device=DEV)
    return (table[seq, pos // BLOCK].long() * BLOCK + pos % BLOCK).to(torch.int32), pos.to(torch.int64)


def _qkv_views(qkv, hq, hkv):
    q, k, v = qkv.split([hq * D, hkv * D, hkv * D], dim=-1)
    return q.view(-1, hq, D), k.view(-1, hkv, D), v.view(-1, hkv, D)


def _cos_sin():
    return rope_table(D, MAX_POS, THETA).to(DEV)


def _layer(g, c, std=0.02):
    H, I, hq, hkv = c["hidden"], c["inter"], c["hq"], c["hkv"]
    return dict(input_norm=_norm_w(g, H), post_norm=_norm_w(g, H), q_norm=_norm_w(g, D), k_norm=_norm_w(g, D),
                qkv=_randn(g, (hq + 2 * hkv) * D, H, scale=std), o=_randn(g, H, hq * D, scale=std),
                gate_up=_randn(g, 2 * I, H, scale=std), down=_randn(g, H, I, scale=std))


def prepare(case, seed):
    g = _gen(seed)
    return {"case": case, **globals()["_prepare_" + case["kind"]](case, g)}


def run(state):
    return globals()["_run_" + state["case"]["kind"]](state)


def exact(case, seed):
    f = globals().get("_exact_" + case["kind"])
    return None if f is None else f(prepare(case, seed))


def work(case):
    b, f = globals()["_work_" + case["kind"]](case)
    return {"bytes": b, "flops": f}


def tolerance(case):
    if case["kind"] == "matmul" and case["dtype"] == "fp32":
        return {"rel": 4e-6}      # fp32 sums over K products: 1.1e-6 from the 64-bit product at K = 4096
    return {"rel": {"decode_step": 0.03, "decode_layer": 0.012, "post_attn": 0.012, "elementwise": 0.008,
                    "pre_attn": 0.012}.get(case["kind"], 0.01), "differ": 0.008}


# --------------------------------------------------------------------------------------- 64-bit forms of the parts

def _rms64(x, w):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x, cos_sin, positions):
    cs = cos_sin.view(cos_sin.shape[0], -1)[positions].double().unsqueeze(1)
    cos, sin = cs.chunk(2, dim=-1)
    a, b = x.chunk(2, dim=-1)
    return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)


def _attend64(q, k, v, causal=True):
    """q [lq, Hq, D], k / v [lk, Hkv, D] in 64 bits; query i sees keys up to lk - lq + i."""
    lq, hq, d = q.shape
    lk, hkv, _ = k.shape
    out = torch.empty_like(q)
    limit = (lk - lq + torch.arange(lq, device=q.device))[:, None]
    masked = (torch.arange(lk, device=q.device)[None, :] > limit) if causal else None
    for h in range(hq):
        s = torch.mm(q[:, h].contiguous(), k[:, h * hkv // hq].t().contiguous()) * d ** -0.5
        if masked is not None:
            s.masked_fill_(masked, float("-inf"))
        out[:, h] = torch.mm(torch.softmax(s, dim=-1), v[:, h * hkv // hq].contiguous())
    return out


def _gather(cache, table_row, n):
    blocks = table_row[:(n + BLOCK - 1) // BLOCK].long()
    return cache[blocks].reshape(-1, *cache.shape[2:])[:n].double()


def _silu_mul64(x):
    gate, up = x.chunk(2, dim=-1)
    return torch.nn.functional.silu(gate) * up


# ------------------------------------------------------------------------------------- one decoder layer, decoding

def _prepare_decode_layer(c, g):
    lens = _lengths(c["batch"], c["lo"], c["hi"])
    k, v, table = _paged(g, lens, c["hkv"])
    slots, pos = _slots(table, list(range(len(lens))), [n - 1 for n in lens])
    return dict(L=_layer(g, c), x=_randn(g, c["batch"], c["hidden"]), residual=_randn(g, c["batch"], c["hidden"]),
                k=k, v=v, table=table, slots=slots, pos=pos, lens=lens, ctx=_i32(lens), cs=_cos_sin())


def _run_decode_layer(s):
    c, L = s["case"], s["L"]
    qkv, res = hip.add_rms_norm_matmul(s["x"], s["residual"], L["input_norm"], EPS, L["qkv"])
    q, k, v = _qkv_views(qkv, c["hq"], c["hkv"])
    o = qk_norm_rope_kv_decode_attention(q, k, v, s["pos"], L["q_norm"], L["k_norm"], EPS, s["cs"], s["k"], s["v"],
                                         s["slots"], s["ctx"], s["table"], D ** -0.5)
    h = hip.matmul(o.view(o.shape[0], -1), L["o"].t())
    h, res = hip.add_rms_norm_matmul(h, res, L["post_norm"], EPS, L["gate_up"], silu=True)
    return {"h": hip.matmul(h, L["down"].t()), "residual": res, "o": o, "k_cache": s["k"], "v_cache": s["v"]}


def _decode_attend64(s, q, k, v):
    """Attention of one new token per sequence; its k and v (64 bits) stand for the cache's last row."""
    o = []
    for i, n in enumerate(s["lens"]):
        kk, vv = _gather(s["k"], s["table"][i], n), _gather(s["v"], s["table"][i], n)
        kk[n - 1], vv[n - 1] = k[i], v[i]
        o.append(_attend64(q[i:i + 1], kk, vv))
    return torch.cat(o)


def _exact_decode_layer(s):
    c, L = s["case"], {n: w.double() for n, w in s["L"].items()}
    res = s["x"].double() + s["residual"].double()
    q, k, v = _qkv_views(_rms64(res, L["input_norm"]) @ L["qkv"].t(), c["hq"], c["hkv"])
    q = _rope64(_rms64(q, L["q_norm"]), s["cs"], s["pos"])
    k = _rope64(_rms64(k, L["k_norm"]), s["cs"], s["pos"])
    o = _decode_attend64(s, q, k, v)
    res = res + o.reshape(o.shape[0], -1) @ L["o"].t()
    h = _silu_mul64(_rms64(res, L["post_norm"]) @ L["gate_up"].t()) @ L["down"].t()
    return {"h": h, "residual": res, "o": o, "k_cache": None, "v_cache": None}


def _params(c):
    return (c["hq"] + 2 * c["hkv"]) * D * c["hidden"] + c["hidden"] * c["hq"] * D + 3 * c["inter"] * c["hidden"]


def _work_decode_layer(c):
    tokens = sum(_lengths(c["batch"], c["lo"], c["hi"]))
    return (2 * _params(c) + tokens * c["hkv"] * D * 4 + c["batch"] * c["hidden"] * 8,
            2 * c["batch"] * _params(c) + 4 * tokens * c["hq"] * D)


# ------------------------------------------------------------------------------------------ the whole decode step

def _prepare_decode_step(c, g):
    cfg = Qwen3Config()
    dims = {"hidden": cfg.hidden_size, "inter": cfg.intermediate_size, "hq": cfg.num_attention_heads,
            "hkv": cfg.num_key_value_heads}
    model = Qwen3(Qwen3Config(vocab_size=1, num_hidden_layers=0), DEV)   # then the weights, as a loader sets them
    model.cfg = Qwen3Config(num_hidden_layers=c["layers"])
    model.embed = _randn(g, cfg.vocab_size, cfg.hidden_size, scale=0.02)
    model.layers = [_layer(g, dims) for _ in range(c["layers"])]
    lens = _lengths(c["batch"], c["lo"], c["hi"])
    k, _, table = _paged(g, lens, dims["hkv"], fill=False)
    model.allocate_kv_cache(k.shape[0]).normal_(generator=g)
    slots, pos = _slots(table, list(range(len(lens))), [n - 1 for n in lens])
    ctx = Context(False, slots, context_lens=_i32(lens), block_tables=table)
    ids = torch.randint(0, cfg.vocab_size, (c["batch"],), generator=g, device=DEV)
    static = ids.clone()

    def step():
        h = model.forward(static, pos, ctx, "hip", attention="hip")
        logits = model.logits(h, backend="hip", as_float=False)
        return h, logits, hip.greedy_sample(logits)

    with torch.inference_mode():
        step()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = step()
        graph.replay()
    return dict(model=model, ids=ids, static=static, pos=pos, ctx=ctx, graph=graph, out=out)


def _run_decode_step(s):
    s["static"].copy_(s["ids"])
    s["graph"].replay()
    h, logits, _ = s["out"]   # without the tokens: a tie of two bf16 logits falls either way in 32 rows
    return {"h": h, "logits": logits}


def _work_decode_step(c):
    tokens = sum(_lengths(c["batch"], c["lo"], c["hi"]))
    b, f = c["layers"] * 2 * _params(SMALL), c["layers"] * 2 * c["batch"] * _params(SMALL)
    b += c["layers"] * tokens * SMALL["hkv"] * D * 4 + 2 * VOCAB * SMALL["hidden"] + 2 * c["batch"] * VOCAB
    return b, f + c["layers"] * 4 * tokens * SMALL["hq"] * D + 2 * c["batch"] * VOCAB * SMALL["hidden"]


# ----------------------------------------------------------------------------------------------- decode attention

def _prepare_decode_attention(c, g):
    lens = _lengths(c["batch"], c["lo"], c["hi"])
    k, v, table = _paged(g, lens, c["hkv"])
    return dict(q=_randn(g, c["batch"], 1, c["hq"], D), k=k, v=v, table=table, lens=lens, ctx=_i32(lens))


def _run_decode_attention(s):
    return flash_attn_with_kvcache(s["q"], s["k"], s["v"], s["ctx"], s["table"], D ** -0.5, causal=True)


def _exact_decode_attention(s):
    return torch.stack([_attend64(s["q"][i].double(), _gather(s["k"], s["table"][i], n),
                                  _gather(s["v"], s["table"][i], n)) for i, n in enumerate(s["lens"])])


def _work_decode_attention(c):
    tokens = sum(_lengths(c["batch"], c["lo"], c["hi"]))
    return tokens * c["hkv"] * D * 4 + c["batch"] * c["hq"] * D * 4, 4 * tokens * c["hq"] * D


# -------------------------------------------------------------------------------------------------------- LM head

def _prepare_lm_head(c, g):
    return dict(x=_randn(g, c["rows"], c["hidden"]), w=_randn(g, c["vocab"], c["hidden"], scale=0.02))


def _run_lm_head(s):
    logits = hip.matmul(s["x"], s["w"].t())
    return {"logits": logits, "tokens": hip.greedy_sample(logits)}


def _exact_lm_head(s):
    return {"logits": s["x"].double() @ s["w"].double().t(), "tokens": None}


def _work_lm_head(c):
    m, n, k = c["rows"], c["vocab"], c["hidden"]
    return 2 * (m * k + n * k + m * n) + 8 * m, 2 * m * n * k


# ----------------------------------------------------------------------------------------------- prefill attention

def _prepare_prefill_attention(c, g):
    lens = _lengths(c["seqs"], c["lo"], c["hi"])
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    T = cu[-1]
    return dict(q=_randn(g, T, c["hq"], D), k=_randn(g, T, c["hkv"], D),
                v=_randn(g, T, (c["hq"] + 2 * c["hkv"]) * D)[:, -c["hkv"] * D:].view(T, c["hkv"], D),
                lens=lens, cu=_i32(cu), longest=max(lens))


def _run_prefill_attention(s):
    return flash_attn_varlen_func(s["q"], s["k"], s["v"], s["longest"], s["cu"], s["longest"], s["cu"], D ** -0.5,
                                  causal=True)


def _exact_prefill_attention(s):
    out, at = [], 0
    for n in s["lens"]:
        out.append(_attend64(*(s[x][at:at + n].double() for x in "qkv")))
        at += n
    return torch.cat(out)


def _work_prefill_attention(c):
    lens = _lengths(c["seqs"], c["lo"], c["hi"])
    return (4 * sum(lens) * (c["hq"] + c["hkv"]) * D, sum(2 * n * (n + 1) for n in lens) * c["hq"] * D)


# --------------------------------------------------------- attention over the paged cache: decodes and a prompt chunk

def _mixed_lengths(c):
    return ([1] * c["decodes"] + [c["chunk"]], _lengths(c["decodes"], c["lo"], c["hi"]) + [c["prefix"] + c["chunk"]])


def _prepare_mixed_attention(c, g):
    lq, lk = _mixed_lengths(c)
    k, v, table = _paged(g, lk, c["hkv"])
    cu_q, cu_k, seq, at = [0], [0], [], []
    for i, (a, b) in enumerate(zip(lq, lk)):
        cu_q.append(cu_q[-1] + a)
        cu_k.append(cu_k[-1] + b)
        seq += [i] * a
        at += range(b - a, b)
    slots, pos = _slots(table, seq, at)
    qkv = _randn(g, cu_q[-1], (c["hq"] + 2 * c["hkv"]) * D)
    return dict(qkv=qkv, qw=_norm_w(g, D), kw=_norm_w(g, D), cs=_cos_sin(), pos=pos, slots=slots, k=k, v=v,
                table=table, lq=lq, lk=lk, cu_q=_i32(cu_q), cu_k=_i32(cu_k))


def _run_mixed_attention(s):
    q, k, v = _qkv_views(s["qkv"], s["case"]["hq"], s["case"]["hkv"])
    q, _ = hip.qk_norm_rope_kv(q, k, v, s["pos"], s["qw"], s["kw"], EPS, s["cs"], s["k"], s["v"], s["slots"], False)
    o = flash_attn_varlen_func(q, s["k"], s["v"], max(s["lq"]), s["cu_q"], max(s["lk"]), s["cu_k"], D ** -0.5,
                               causal=True, block_table=s["table"])
    return {"o": o, "q": q, "k_cache": s["k"], "v_cache": s["v"]}


def _exact_mixed_attention(s):
    q, k, v = _qkv_views(s["qkv"].double(), s["case"]["hq"], s["case"]["hkv"])
    q = _rope64(_rms64(q, s["qw"]), s["cs"], s["pos"])
    k = _rope64(_rms64(k, s["kw"]), s["cs"], s["pos"])
    out, at = [], 0
    for i, (a, b) in enumerate(zip(s["lq"], s["lk"])):
        kk, vv = _gather(s["k"], s["table"][i], b), _gather(s["v"], s["table"][i], b)
        kk[b - a:], vv[b - a:] = k[at:at + a], v[at:at + a]
        out.append(_attend64(q[at:at + a], kk, vv))
        at += a
    return {"o": torch.cat(out), "q": q, "k_cache": None, "v_cache": None}


def _work_mixed_attention(c):
    lq, lk = _mixed_lengths(c)
    seen = sum(sum(range(b - a + 1, b + 1)) for a, b in zip(lq, lk))
    return (sum(lq) * (3 * c["hq"] + 4 * c["hkv"]) * D * 2 + sum(lk) * c["hkv"] * D * 4, 4 * seen * c["hq"] * D)


# ------------------------------------------------------------------------- a prefill layer before its attention

def _prepare_pre_attn(c, g):
    T = c["tokens"]
    k, v, table = _paged(g, [T], c["hkv"], fill=False)
    slots, pos = _slots(table, [0] * T, list(range(T)))
    return dict(L=_layer(g, c), x=_randn(g, T, c["hidden"]), residual=_randn(g, T, c["hidden"]), k=k, v=v,
                slots=slots, pos=pos, cs=_cos_sin())


def _run_pre_attn(s):
    c, L = s["case"], s["L"]
    h, res = hip.fused_add_rms_norm(s["x"], s["residual"], L["input_norm"], EPS)
    q, k, v = _qkv_views(hip.matmul(h, L["qkv"].t()), c["hq"], c["hkv"])
    q, k = hip.qk_norm_rope_kv(q, k, v, s["pos"], L["q_norm"], L["k_norm"], EPS, s["cs"], s["k"], s["v"], s["slots"],
                               True)
    return {"q": q, "k": k, "v": v, "residual": res, "k_cache": s["k"], "v_cache": s["v"]}


def _exact_pre_attn(s):
    c, L = s["case"], {n: w.double() for n, w in s["L"].items()}
    res = s["x"].double() + s["residual"].double()
    q, k, v = _qkv_views(_rms64(res, L["input_norm"]) @ L["qkv"].t(), c["hq"], c["hkv"])
    q = _rope64(_rms64(q, L["q_norm"]), s["cs"], s["pos"])
    k = _rope64(_rms64(k, L["k_norm"]), s["cs"], s["pos"])
    caches = [torch.zeros(s["k"].shape, dtype=torch.float64, device=DEV) for _ in "kv"]
    for cache, rows in zip(caches, (k, v)):
        cache.view(-1, c["hkv"], D)[s["slots"].long()] = rows
    return {"q": q, "k": k, "v": v, "residual": res, "k_cache": caches[0], "v_cache": caches[1]}


def _work_pre_attn(c):
    T, n = c["tokens"], (c["hq"] + 2 * c["hkv"]) * D
    return 2 * T * (3 * c["hidden"] + n + 3 * c["hkv"] * D) + 2 * n * c["hidden"], 2 * T * n * c["hidden"]


# -------------------------------------------------------------------------- a prefill layer after its attention

def _prepare_post_attn(c, g):
    T = c["tokens"]
    return dict(L=_layer(g, c), o=_randn(g, T, c["hq"] * D), residual=_randn(g, T, c["hidden"]))


def _run_post_attn(s):
    L = s["L"]
    h, res = hip.matmul_add_rms_norm(s["o"], L["o"], s["residual"], L["post_norm"], EPS)
    h = hip.matmul_silu_and_mul(h, L["gate_up"])
    y, out = hip.matmul_add_rms_norm(h, L["down"], res, L["input_norm"], EPS)
    return {"h": h, "y": y, "residual": out}


def _exact_post_attn(s):
    L = {n: w.double() for n, w in s["L"].items()}
    res = s["o"].double() @ L["o"].t() + s["residual"].double()
    h = _silu_mul64(_rms64(res, L["post_norm"]) @ L["gate_up"].t())
    res = h @ L["down"].t() + res
    return {"h": h, "y": _rms64(res, L["input_norm"]), "residual": res}


def _work_post_attn(c):
    T, H, I, n = c["tokens"], c["hidden"], c["inter"], c["hq"] * D
    params = H * n + 3 * I * H
    return 2 * (T * (n + 3 * H + I) + params), 2 * T * params


# ------------------------------------------------------------------------------------ the memory-bound kernels alone

def _prepare_elementwise(c, g):
    T, hq, hkv = c["tokens"], c["hq"], c["hkv"]
    quarter = [T * i // 4 for i in range(5)]
    lens = [max(1, b - a) for a, b in zip(quarter, quarter[1:])]
    k, v, table = _paged(g, lens, hkv, fill=False)
    seq = [i for i in range(4) for _ in range(quarter[i], quarter[i + 1])]
    slots, pos = _slots(table, seq, [t - quarter[i] for t, i in enumerate(seq)])
    return dict(qkv=_randn(g, T, (hq + 2 * hkv) * D + 64), qw=_norm_w(g, D), kw=_norm_w(g, D), w=_norm_w(g, c["hidden"]),
                x=_randn(g, T, c["hidden"]), residual=_randn(g, T, c["hidden"]),
                gate_up=_randn(g, T, 2 * c["inter"]), k=k, v=v, slots=slots, pos=pos, cs=_cos_sin())


def _run_elementwise(s):
    c = s["case"]
    h, res = hip.fused_add_rms_norm(s["x"], s["residual"], s["w"], EPS)
    q, k, v = _qkv_views(s["qkv"][:, :-64], c["hq"], c["hkv"])
    q, _ = hip.qk_norm_rope_kv(q, k, v, s["pos"], s["qw"], s["kw"], EPS, s["cs"], s["k"], s["v"], s["slots"], False)
    return {"h": h, "residual": res, "q": q, "k_cache": s["k"], "v_cache": s["v"], "y": hip.rms_norm(s["x"], s["w"], EPS),
            "act": hip.silu_and_mul(s["gate_up"])}


def _exact_elementwise(s):
    c = s["case"]
    res = s["x"].double() + s["residual"].double()
    q, k, v = _qkv_views(s["qkv"][:, :-64].double(), c["hq"], c["hkv"])
    caches = [torch.zeros(s["k"].shape, dtype=torch.float64, device=DEV) for _ in "kv"]
    for cache, rows in zip(caches, (_rope64(_rms64(k, s["kw"]), s["cs"], s["pos"]), v)):
        cache.view(-1, c["hkv"], D)[s["slots"].long()] = rows
    return {"h": _rms64(res, s["w"]), "residual": res, "q": _rope64(_rms64(q, s["qw"]), s["cs"], s["pos"]),
            "k_cache": caches[0], "v_cache": caches[1], "y": _rms64(s["x"], s["w"]),
            "act": _silu_mul64(s["gate_up"].double())}


def _work_elementwise(c):
    T, H, I, hq, hkv = c["tokens"], c["hidden"], c["inter"], c["hq"], c["hkv"]
    b = T * (2 * 6 * H + 2 * 2 * hq * D + 8 * hkv * D + 4 * D + 12 + 2 * 3 * I)
    return b, T * (10 * H + 10 * (hq + hkv) * D + 5 * I)


# ------------------------------------------------------------------------------------------------ the plain product

def _prepare_matmul(c, g):
    dt = torch.float32 if c["dtype"] == "fp32" else BF16
    a = _randn(g, c["m"], c["k"], scale=c["k"] ** -0.5, dtype=dt)
    b = _randn(g, c["k"], c["n"], dtype=dt) if c["b_rows"] == "k" else _randn(g, c["n"], c["k"], dtype=dt).t()
    return dict(a=a, b=b)


def _run_matmul(s):
    return hip.matmul(s["a"], s["b"], s["case"]["precision"])


def _tf32(x):
    """x rounded to a 10-bit mantissa, to nearest even (finite values)."""
    u = x.view(torch.int32)
    u = u + 0xfff + ((u >> 13) & 1)
    return (u & ~0x1fff).view(torch.float32)


def _exact_matmul(s):
    a, b = s["a"], s["b"]
    if s["case"]["dtype"] == "fp32" and s["case"]["precision"] == "tf32":
        a, b = _tf32(a.contiguous()), _tf32(b.contiguous())
    return a.double() @ b.double()


def _work_matmul(c):
    m, n, k = c["m"], c["n"], c["k"]
    return (4 if c["dtype"] == "fp32" else 2) * (m * k + k * n + m * n), 2 * m * n * k
