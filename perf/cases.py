"""The measured work of the paged-KV serving path: decode and prefill attention of a layer,
decoder layers, and whole decode steps, each through the entry points a program calls.

Kinds of case (field "kind"):
  decode   ops.paged_decode with RoPE and the append folded in (what Attention.forward calls
           for a decode step) on the pools of `layers` layers, replayed as one HIP graph, the
           way the runner replays its decode steps.
  prefill  ops.rope_kv_append (q = None) and ops.varlen_prefill with cos/sin on one layer (what
           Attention.forward calls for a prefill), launched eagerly, as the runner's prefills
           are; with `prefix` > 0 the prompts continue a cached prefix.
  layer    DecoderLayer.forward of `layers` layers, each on the hidden states and the residual
           stream of the one before: a decode step (a replayed graph) or a prefill (eager).
  model    ModelRunner.forward of a whole model, a decode step as a replayed graph: logits.

Lengths belong to the case (field "lens"), values and block tables to the seed.
"""
import math

import numpy as np
import torch
import torch.nn.functional as F

from needle_amd import ops
from needle_amd.model.config import ModelConfig
from needle_amd.model.qwen2 import DecoderLayer, build_model, fuse_projections
from needle_amd.model.runner import Batch, ModelRunner

DEVICE = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
NAMES = {"bf16": "bfloat16", "fp16": "float16", "fp32": "float32"}
ROPE_THETA = 1000000.0

# heads, kv heads, head_dim
QWEN_05B = (14, 2, 64)
QWEN_7B = (28, 4, 128)
LLAMA_8B = (32, 8, 128)
LLAMA_MHA = (32, 32, 128)

# name: hidden, heads, kv heads, ffn, q/k/v bias
WIDTHS = {
    "qwen2-0.5b": (896, 14, 2, 4864, True),
    "qwen2-7b": (3584, 28, 4, 18944, True),
    "llama3-8b": (4096, 32, 8, 14336, False),
}


def _attn(name, kind, heads, **more):
    return dict(name=name, kind=kind, heads=heads[0], kv_heads=heads[1], head_dim=heads[2], **more)


def listed():
    return [
        # A small batch of short chats: one decode step's attention over the 24 layers of a
        # 0.5B model (the smallest decode, a few microseconds per layer).
        _attn("decode-0.5b-8-seqs", "decode", QWEN_05B, dtype="bf16", page=16, seqs=8, lo=32,
              hi=512, layers=24, lens=1001),
        # One user far into a long document: a single sequence has to fill the GPU.
        _attn("decode-one-long", "decode", LLAMA_8B, dtype="fp16", page=16, seqs=1, lo=20011,
              hi=20011, layers=8, lens=1),
        # The throughput batch of the benchmark: 64 mid-length sequences, one layer.
        _attn("decode-8b-64-seqs", "decode", LLAMA_8B, dtype="bf16", page=16, seqs=64, lo=512,
              hi=4096, layers=1, lens=1002),
        # Long contexts of very different lengths with large pages.
        _attn("decode-long-page-64", "decode", LLAMA_8B, dtype="bf16", page=64, seqs=48, lo=1024,
              hi=32768, layers=1, lens=1005),
        # A float32 model (--dtype float32) at a serving batch.
        _attn("decode-fp32-12-seqs", "decode", QWEN_7B, dtype="fp32", page=16, seqs=12, lo=100,
              hi=4000, layers=4, lens=12),
        # One short prompt of an odd length, in float16: the smallest prefill.
        _attn("prefill-one-short", "prefill", QWEN_05B, dtype="fp16", page=16, seqs=1, lo=77,
              hi=77, prefix=0, lens=5),
        # The benchmark's packed prompts.
        _attn("prefill-7b-16-prompts", "prefill", QWEN_7B, dtype="bf16", page=16, seqs=16, lo=128,
              hi=2048, prefix=0, lens=1003),
        # Follow-up turns: a few hundred new tokens after long cached conversations.
        _attn("prefill-after-prefix", "prefill", LLAMA_8B, dtype="bf16", page=32, seqs=3, lo=100,
              hi=600, prefix=16000, lens=8),
        # Prompts of a float32 model.
        _attn("prefill-fp32-6-prompts", "prefill", QWEN_05B, dtype="fp32", page=16, seqs=6, lo=64,
              hi=1024, prefix=0, lens=6),
        # A decode step of one 7B-sized decoder layer: norms, projections, attention, MLP.
        dict(name="layer-decode-7b", kind="layer", width="qwen2-7b", dtype="bf16", page=16, layers=1,
             decode=True, seqs=16, lo=64, hi=1024, lens=16),
        # A prefill forward of 0.5B-sized layers at the engine's usual few thousand tokens.
        dict(name="layer-prefill-0.5b", kind="layer", width="qwen2-0.5b", dtype="bf16", page=16,
             layers=4, decode=False, seqs=7, lo=64, hi=1024, lens=7),
        # A whole decode step of the end-to-end benchmark's model at its usual running batch.
        dict(name="model-decode-0.5b", kind="model", width="qwen2-0.5b", dtype="bf16", page=16,
             layers=24, seqs=9, lo=64, hi=1400, lens=9),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "layer",
                       "layer", "model"])
    lens = rng.randrange(1 << 20)
    if kind == "decode":
        heads = rng.choice([QWEN_05B, QWEN_7B, LLAMA_8B, LLAMA_8B, LLAMA_MHA])
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        hi = _log_int(rng, 40, 32768)
        lo = max(1, int(hi / rng.uniform(1, 16)))
        seqs = _log_int(rng, 1, 128)
        # K and V bytes of a step, held below the largest listed case's
        row = 2 * heads[1] * heads[2] * (4 if dtype == "fp32" else 2)
        seqs = max(1, min(seqs, int(1.5e9 / (row * (lo + hi)))))
        step = row * seqs * (lo + hi)
        layers = max(1, min(rng.choice([1, 2, 8, 24]), int(1.5e9 / step)))
        return dict(kind=kind, heads=heads[0], kv_heads=heads[1], head_dim=heads[2], dtype=dtype,
                    page=rng.choice([16, 16, 16, 32, 64, 128]), seqs=seqs, lo=lo, hi=hi,
                    layers=layers, lens=lens)
    if kind == "prefill":
        heads = rng.choice([QWEN_05B, QWEN_7B, LLAMA_8B, LLAMA_MHA])
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        hi = _log_int(rng, 3, 1024 if dtype == "fp32" else 2048)
        lo = max(1, int(hi / rng.uniform(1, 16)))
        prefix = rng.choice([0, 0, _log_int(rng, 64, 2048 if dtype == "fp32" else 16384)])
        seqs = _log_int(rng, 1, 16)
        seqs = max(1, min(seqs, int(1.6e11 / (4 * heads[0] * heads[2] * hi * (prefix + hi)))))
        return dict(kind=kind, heads=heads[0], kv_heads=heads[1], head_dim=heads[2], dtype=dtype,
                    page=rng.choice([16, 16, 16, 32, 64]), seqs=seqs, lo=lo, hi=hi, prefix=prefix,
                    lens=lens)
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    hi = _log_int(rng, 40, 2048)
    lo = max(1, int(hi / rng.uniform(1, 16)))
    if kind == "layer":
        width = rng.choice(sorted(WIDTHS))
        decode = rng.random() < 0.6
        seqs, layers = _log_int(rng, 1, 96 if decode else 4), rng.choice([1, 2])
        if not decode:
            # tokens held below the largest listed prefill's multiply-adds
            most = {"qwen2-0.5b": 10000, "qwen2-7b": 700, "llama3-8b": 700}[width] // layers
            hi = min(hi, most // seqs)
            lo = min(lo, hi)
        return dict(kind=kind, width=width, dtype=dtype, page=16, layers=layers, decode=decode,
                    seqs=seqs, lo=lo, hi=hi, lens=lens)
    return dict(kind=kind, width="qwen2-0.5b", dtype=dtype, page=16, layers=rng.choice([6, 12, 24]),
                seqs=_log_int(rng, 1, 64), lo=lo, hi=hi, lens=lens)


# ---------------------------------------------------------------------------- inputs

def _is_decode(case):
    return case["kind"] in ("decode", "model") or bool(case.get("decode"))


def _heads(case):
    if "heads" in case:
        return case["heads"], case["kv_heads"], case["head_dim"]
    hidden, h, hkv, _ffn, _bias = WIDTHS[case["width"]]
    return h, hkv, hidden // h


def _lengths(case):
    """(cached tokens, new tokens) of every sequence: spread over their logarithm."""
    r = np.random.default_rng(case["lens"])
    n = np.exp(r.uniform(math.log(case["lo"]), math.log(case["hi"] + 1), case["seqs"]))
    n = np.clip(n.astype(np.int64), case["lo"], case["hi"]).tolist()
    if _is_decode(case):
        return n, [1] * len(n)
    p = case.get("prefix", 0)
    return (r.integers(p // 4, p, size=len(n), endpoint=True).tolist() if p else [0] * len(n)), n


def _inputs(case, seed):
    """Everything that is drawn from the seed, as plain tensors on the GPU."""
    dtype, page = DTYPES[case["dtype"]], case["page"]
    h, hkv, d = _heads(case)
    ctx, new = _lengths(case)
    layers = case.get("layers", 1)
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)

    def randn(*shape, std=1.0):
        return torch.randn(shape, generator=gen, device=DEVICE, dtype=dtype).mul_(std)

    blocks = [-(-(c + n) // page) for c, n in zip(ctx, new)]
    num_blocks = sum(blocks) + 2
    perm = np.random.default_rng(seed).permutation(num_blocks - 1).tolist()
    table = np.full((len(ctx), max(blocks)), num_blocks - 1, dtype=np.int32)
    at = 0
    for i, b in enumerate(blocks):
        table[i, :b] = perm[at:at + b]
        at += b
    pos = np.concatenate([np.arange(c, c + n) for c, n in zip(ctx, new)])
    total = len(pos)
    s = {"case": case, "ctx": ctx, "new": new,
         "table": torch.from_numpy(table).to(DEVICE),
         "lens": torch.tensor(ctx, dtype=torch.int32, device=DEVICE),
         "cu": torch.tensor(np.concatenate([[0], np.cumsum(new)]), dtype=torch.int32,
                            device=DEVICE),
         "positions": torch.from_numpy(pos).to(DEVICE),
         "pools": [randn(2, num_blocks, hkv, page, d) for _ in range(layers)]}
    inv = 1.0 / (ROPE_THETA ** (torch.arange(0, d, 2, device=DEVICE).float() / d))
    angle = torch.outer(s["positions"].float(), inv)
    angle = torch.cat([angle, angle], dim=-1)
    s["cos"], s["sin"] = angle.cos().to(dtype), angle.sin().to(dtype)
    if "width" not in case:
        # the projections' outputs: views of one fused q/k/v row per token
        qkv = randn(total, (h + 2 * hkv) * d)
        q, k, v = qkv.split([h * d, hkv * d, hkv * d], dim=-1)
        s["q"], s["k"], s["v"] = (q.view(total, h, d), k.view(total, hkv, d),
                                  v.view(total, hkv, d))
        return s
    hidden, _h, _hkv, ffn, bias = WIDTHS[case["width"]]
    vocab = 151936 if case["kind"] == "model" else 32
    config = ModelConfig(model_type="qwen2" if bias else "llama", hidden_size=hidden,
                         num_hidden_layers=layers, num_attention_heads=h, num_key_value_heads=hkv,
                         intermediate_size=ffn, vocab_size=vocab, max_position_embeddings=4096,
                         rms_norm_eps=1e-6, rope_theta=ROPE_THETA)
    with torch.device(DEVICE):
        if case["kind"] == "model":
            m = build_model(config)
        else:
            m = torch.nn.ModuleList([DecoderLayer(config, i, bias) for i in range(layers)])
    m = m.to(dtype).eval()
    with torch.no_grad():
        for name, p in m.named_parameters():
            if "norm" in name:
                p.copy_(1.0 + randn(*p.shape, std=0.1))
            elif "embed" in name:   # the stream's scale next to what a layer adds to it
                p.copy_(randn(*p.shape))
            else:
                p.copy_(randn(*p.shape, std=0.02))
    s["module"], s["config"] = m, config
    if case["kind"] == "model":
        s["ids"] = torch.randint(0, vocab, (total,), generator=gen, device=DEVICE)
    else:
        s["hidden"], s["residual"] = randn(total, hidden, std=0.5), randn(total, hidden)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "layer":
        fuse_projections(s["module"])
    elif kind == "model":
        s["runner"] = ModelRunner(s["config"], case["page"], NAMES[case["dtype"]], DEVICE,
                                  model=s["module"])
        s["runner"].kv_caches = s["pools"]
    elif kind == "decode":
        h, hkv, d = _heads(case)
        need = ops.decode_workspace_bytes(case["seqs"], h, hkv, d, s["table"].shape[1],
                                          case["page"])
        s["workspace"] = ops.decode_workspace(need, torch.device(DEVICE))
    if _is_decode(case):
        # the serving loop's decode steps are graphs, captured once and replayed
        with torch.no_grad():
            _step(s)
            torch.cuda.synchronize()
            s["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["graph"]):
                s["result"] = _step(s)
        torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------------- one pass

def _step(s):
    case = s["case"]
    kind, pools = case["kind"], s["pools"]
    h, hkv, d = _heads(case)
    scale = 1.0 / math.sqrt(d)
    if kind == "decode":
        outs = [ops.paged_decode(s["q"], pool, s["table"], s["lens"], scale, h, hkv, d,
                                 workspace=s["workspace"], new_k=s["k"], new_v=s["v"],
                                 cos=s["cos"], sin=s["sin"]) for pool in pools]
        return {"out": outs, "pool": pools}
    if kind == "prefill":
        pool, most = pools[0], max(s["new"])
        ops.rope_kv_append(None, s["k"], s["v"], s["cos"], s["sin"], pool, s["table"], s["lens"],
                           s["cu"])
        out = ops.varlen_prefill(s["q"], pool, s["table"], s["cu"], s["lens"], most, scale, h,
                                 hkv, d, max_context_len=max(s["ctx"]), cos=s["cos"],
                                 sin=s["sin"])
        return {"out": out, "pool": pool}
    decode = _is_decode(case)
    if kind == "layer":
        x, residual = s["hidden"], s["residual"]
        for layer, pool in zip(s["module"], pools):
            x, residual = layer(x, s["positions"], pool, s["table"], s["cu"], s["lens"],
                                max(s["new"]), not decode, s["cos"], s["sin"], residual)
        return {"hidden": x, "residual": residual, "pool": pools}
    logits = s["runner"].forward(Batch(s["ids"], s["positions"], s["cu"], 1, s["table"],
                                       s["lens"], False))
    return {"logits": logits, "pool": pools}


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["result"]
    with torch.no_grad():
        return _step(state)


# ---------------------------------------------------------------------------- exact values

def _rope(x, cos, sin):
    half = x.shape[-1] // 2
    rot = torch.cat([-x[..., half:], x[..., :half]], dim=-1)
    return x * cos.unsqueeze(1) + rot * sin.unsqueeze(1)


def _attend(s, q, k, v, pool, cos, sin):
    """(attention output, pool after the append) in float64; q, k, v as projected."""
    page = pool.shape[3]
    hkv, d = k.shape[1], k.shape[2]
    g = q.shape[1] // hkv
    q, k = _rope(q, cos, sin), _rope(k, cos, sin)
    pool = pool.double()
    out = torch.empty_like(q)
    at = 0
    for i, (c, n) in enumerate(zip(s["ctx"], s["new"])):
        p = torch.arange(c, c + n, device=DEVICE)
        blk = s["table"][i].long()
        pool[0, blk[p // page], :, p % page] = k[at:at + n]
        pool[1, blk[p // page], :, p % page] = v[at:at + n]
        every = torch.arange(c + n, device=DEVICE)
        kv = pool[:, blk[every // page], :, every % page]        # [c + n, 2, hkv, d]
        keys, values = kv.permute(1, 2, 0, 3).contiguous()       # [hkv, c + n, d] each
        qi = q[at:at + n].view(n, hkv, g, d).permute(1, 2, 0, 3).reshape(hkv, g * n, d)
        w = torch.matmul(qi, keys.transpose(1, 2).contiguous()).mul_(1.0 / math.sqrt(d))
        w = w.view(hkv, g, n, c + n).masked_fill_(every > p[:, None], -math.inf)
        w = torch.softmax(w, dim=-1).view(hkv, g * n, c + n)
        o = torch.matmul(w, values).view(hkv, g, n, d)
        out[at:at + n] = o.permute(2, 0, 1, 3).reshape(n, hkv * g, d)
        at += n
    return out, pool


def _norm(x, weight, eps=1e-6):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * weight


def _linear(x, m):
    return F.linear(x, m.weight.double(), None if m.bias is None else m.bias.double())


def _layer(s, layer, x, residual, pool, cos, sin):
    h, hkv, d = _heads(s["case"])
    t = x.shape[0]
    residual = x if residual is None else x + residual
    x = _norm(residual, layer.input_layernorm.weight.double())
    a = layer.self_attn
    o, pool = _attend(s, _linear(x, a.q_proj).view(t, h, d), _linear(x, a.k_proj).view(t, hkv, d),
                      _linear(x, a.v_proj).view(t, hkv, d), pool, cos, sin)
    residual = residual + _linear(o.reshape(t, h * d), a.o_proj)
    x = _norm(residual, layer.post_attention_layernorm.weight.double())
    m = layer.mlp
    return _linear(F.silu(_linear(x, m.gate_proj)) * _linear(x, m.up_proj), m.down_proj), \
        residual, pool


@torch.no_grad()
def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    cos, sin = s["cos"].double(), s["sin"].double()
    if kind in ("decode", "prefill"):
        q, k, v = (s[n].double() for n in ("q", "k", "v"))
        got = [_attend(s, q, k, v, pool, cos, sin) for pool in s["pools"]]
        outs, pools = [o for o, _ in got], [p for _, p in got]
        if kind == "prefill":
            return {"out": outs[0], "pool": pools[0]}
        return {"out": outs, "pool": pools}
    m = s["module"]
    layers = m.model.layers if kind == "model" else m
    if kind == "model":
        x, residual = m.model.embed_tokens.weight.double()[s["ids"]], None
        # the model holds its own cos/sin tables in the model dtype
        rope = m.model.rotary_emb
        cos = rope.cos_cached[s["positions"]].double()
        sin = rope.sin_cached[s["positions"]].double()
    else:
        x, residual = s["hidden"].double(), s["residual"].double()
    pools = []
    for layer, pool in zip(layers, s["pools"]):
        x, residual, p = _layer(s, layer, x, residual, pool, cos, sin)
        pools.append(p)
    if kind == "layer":
        return {"hidden": x, "residual": residual, "pool": pools}
    x = _norm(x + residual, m.model.norm.weight.double())
    return {"logits": _linear(x, m.lm_head), "pool": pools}


# ---------------------------------------------------------------------------- work, tolerance

def work(case):
    h, hkv, d = _heads(case)
    e = 4 if case["dtype"] == "fp32" else 2
    ctx, new = _lengths(case)
    total, layers = sum(new), case.get("layers", 1)
    pairs = sum(n * c + n * (n + 1) // 2 for c, n in zip(ctx, new))
    cached = sum(ctx) * hkv * d * 2 * e
    table = 4 * sum(-(-(c + n) // case["page"]) for c, n in zip(ctx, new))
    # q, k, v and cos/sin rows in, the output and the appended rows out
    rows = total * ((h + 2 * hkv) * d + 2 * d + h * d + 2 * hkv * d) * e
    flops = 4 * h * d * pairs
    if "width" in case:
        hidden, _h, _hkv, ffn, _bias = WIDTHS[case["width"]]
        weights = hidden * (2 * h * d + 2 * hkv * d + 3 * ffn)
        flops += 2 * total * weights
        # hidden states and residual stream in and out once per run, K/V rows appended per layer
        once = 4 * total * hidden * e
        per_layer = weights * e + cached + table + total * 2 * hkv * d * e
        if case["kind"] == "model":
            vocab = 151936
            return {"bytes": layers * per_layer + (vocab * hidden + total * vocab) * e + once,
                    "flops": layers * flops + 2 * total * hidden * vocab}
        return {"bytes": layers * per_layer + once, "flops": layers * flops}
    return {"bytes": layers * (cached + rows + table), "flops": layers * flops}


def tolerance(case):
    """About four times the distance from the float64 values measured for each kind.  A model's
    or a layer stack's rounding differences travel through what follows (bf16: 0.006 to 0.014
    from exact); attention alone is 0.003 (bf16), 0.0004 (fp16), 4e-7 (fp32) away."""
    if "width" in case:
        return {"rel": {"bf16": 3e-2, "fp16": 5e-3}[case["dtype"]]}
    return {"rel": {"bf16": 1e-2, "fp16": 1.5e-3, "fp32": 2e-6}[case["dtype"]]}
