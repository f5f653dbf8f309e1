"""The work a serving process gives this framework, as cases that can be timed: decoder layers, attention over long
contexts, experts, recurrent mixers and sampling, through the entry points the model code itself calls
(``models``' modules and ``vllm_distributed_amd.ops``), with the sizes of ``models/configs`` and of ``bench.py``.

kinds
  layer      embedding -> one Llama decoder layer -> final norm over a paged cache.  Batches of decoded rows are replayed
             from a captured graph, as the model runner replays them; batches with prompts run eagerly.
  attention  this step's keys and values into the paged cache, then attention over it: decoded rows, or prompt portions
  latent     the same over DeepSeek's latent cache
  experts    a sparse block (router, experts, weighted sum) in bf16 or with 4-bit AWQ experts
  recurrence the sequence mixers with per-request state: gated delta rule, linear attention, state-space scan
  sample     one token per row under temperature, top-k, top-p and min-p
"""
import math
import random

import torch

DEV = "cuda"
BLOCK = 64                      # tokens per cache block on the GPU

# hidden, feed-forward, query heads, key heads, rope base (models/configs/llama-3-8b.json, llama-3-70b.json)
DENSE = {"8b": (4096, 14336, 32, 8, 500000.0), "70b": (8192, 28672, 64, 8, 500000.0)}
VOCAB = 32000                   # rows of the embedding table that the cases carry
# hidden, expert width, experts, chosen (deepseek-v2-lite.json, mixtral-8x7b.json, qwen3-coder-480b-a35b.json)
EXPERTS = {"v2-lite": (2048, 1408, 64, 6), "8x7b": (4096, 14336, 8, 2), "480b": (6144, 2560, 160, 8)}
RANK, ROPE = 512, 64            # deepseek-v2-lite.json: width of the latent, of the rotated shared key part


def listed():
    return [
        # one user's stream on an 8B model: launches and weight streaming, the latency of a token
        {"name": "layer_decode_1", "kind": "layer", "model": "8b", "decodes": 1, "context": 1000, "prompts": 0, "tokens": 0},
        # 256 streams on a 70B model (bench.py's second point)
        {"name": "layer_decode_256", "kind": "layer", "model": "70b", "decodes": 256, "context": 160, "prompts": 0, "tokens": 0},
        # 2048 streams on a 70B model (bench.py's headline point)
        {"name": "layer_decode_2048", "kind": "layer", "model": "70b", "decodes": 2048, "context": 150, "prompts": 0, "tokens": 0},
        # prompts of unequal length beside running streams, one scheduler step of an 8B model
        {"name": "layer_mixed_8k", "kind": "layer", "model": "8b", "decodes": 61, "context": 700, "prompts": 5, "tokens": 8131},
        # long conversations, one new token each
        {"name": "attention_decode_long", "kind": "attention", "heads": 32, "kv_heads": 8, "dim": 128, "rows": 48, "new": 1,
         "context": 9000, "cache": "bf16"},
        # latent attention of 128 streams, one rank's 16 heads
        {"name": "latent_decode", "kind": "latent", "heads": 16, "rows": 128, "new": 1, "context": 3100},
        # a prompt step through sparse experts
        {"name": "experts_prompt", "kind": "experts", "model": "v2-lite", "weights": "bf16", "tokens": 6001},
        # 16 streams through 4-bit experts (the documented deployment's model)
        {"name": "experts_decode_awq", "kind": "experts", "model": "480b", "weights": "awq", "tokens": 16},
        # prompts through the gated delta rule (a decay per key channel)
        {"name": "delta_rule_prompt", "kind": "recurrence", "op": "delta_channel", "heads": 16, "groups": 16, "dim": 128,
         "vdim": 128, "rows": 5, "tokens": 8017},
        # prompts through gated linear attention (a decay per key channel)
        {"name": "linear_attention_prompt", "kind": "recurrence", "op": "linear_channel", "heads": 16, "groups": 16, "dim": 128,
         "vdim": 128, "rows": 3, "tokens": 6007},
        # 128 decoded rows through a state-space layer: states in and out
        {"name": "state_space_decode", "kind": "recurrence", "op": "state_space", "heads": 16, "groups": 2, "dim": 128,
         "vdim": 128, "rows": 128, "tokens": 128},
        # a sampled token for each of 256 streams, Llama-3's vocabulary
        {"name": "sample_256", "kind": "sample", "rows": 256, "vocab": 128256, "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "attention", "latent", "experts", "recurrence", "recurrence", "recurrence", "sample"])
    if kind == "layer":
        model = rng.choice(["8b", "70b"])
        if rng.random() < 0.6:
            rows = _log_int(rng, 1, 1800)
            return {"kind": kind, "model": model, "decodes": rows, "context": _log_int(rng, 100, 4000 if rows <= 64 else 300),
                    "prompts": 0, "tokens": 0}
        tokens = _log_int(rng, 128, 8000 if model == "8b" else 2000)
        return {"kind": kind, "model": model, "decodes": rng.choice([0, rng.randint(1, 64)]), "context": rng.randint(100, 900),
                "prompts": min(rng.randint(1, 8), tokens // 32), "tokens": tokens}
    if kind == "attention":
        heads, kv, dim = rng.choice([(32, 8, 128), (64, 8, 128), (16, 2, 128), (32, 8, 64), (16, 8, 256)])
        cache = rng.choice(["bf16", "bf16", "fp8"])
        if rng.random() < 0.6:
            rows = _log_int(rng, 1, 256)
            return {"kind": kind, "heads": heads, "kv_heads": kv, "dim": dim, "rows": rows, "new": 1,
                    "context": _log_int(rng, 200, min(32000, 400000 // rows)), "cache": cache}
        new = _log_int(rng, 32, 4096)
        return {"kind": kind, "heads": heads, "kv_heads": kv, "dim": dim, "rows": max(1, min(8, 8192 // new) - rng.randint(0, 3)),
                "new": new, "context": new + rng.choice([0, 0, rng.randint(1, 4000)]), "cache": cache}
    if kind == "latent":
        heads = rng.choice([16, 16, 128])
        if rng.random() < 0.7:
            rows = _log_int(rng, 1, 128)
            return {"kind": kind, "heads": heads, "rows": rows, "new": 1,
                    "context": _log_int(rng, 200, min(16000, 400000 // rows if heads == 16 else 80000 // rows))}
        new = _log_int(rng, 32, 1500 if heads == 16 else 300)
        return {"kind": kind, "heads": heads, "rows": rng.randint(1, 3), "new": new, "context": new + rng.randint(0, 500)}
    if kind == "experts":
        model, weights = rng.choice([("v2-lite", "bf16"), ("v2-lite", "bf16"), ("8x7b", "bf16"), ("480b", "awq")])
        return {"kind": kind, "model": model, "weights": weights,
                "tokens": _log_int(rng, 1, {"v2-lite": 6000, "8x7b": 1500, "480b": 64}[model])}
    if kind == "recurrence":
        op = rng.choice(["delta_channel", "delta_head", "linear_channel", "linear_head", "state_space"])
        heads = rng.choice([8, 16, 32])
        dim, vdim = rng.choice([(128, 128), (128, 128), (64, 64), (64, 128)])
        groups = {"state_space": max(heads // 8, 1), "delta_head": rng.choice([heads, heads // 2])}.get(op, heads)
        out = {"kind": kind, "op": op, "heads": heads, "groups": groups, "dim": dim, "vdim": vdim}
        if rng.random() < 0.35:
            rows = _log_int(rng, 1, 256)
            return dict(out, rows=rows, tokens=rows)
        rows = _log_int(rng, 1, 24)
        return dict(out, rows=rows, tokens=rows * 20 + _log_int(rng, 100, 7500 if heads < 32 else 4000))
    return {"kind": kind, "rows": _log_int(rng, 1, 320), "vocab": rng.choice([32000, 50257, 102400, 128256]),
            "dtype": rng.choice(["bf16", "fp32"])}


# ------------------------------------------------------------------ shapes and plain inputs
def _split(total, parts):
    """``total`` cut into ``parts`` unequal positive pieces, the same for the same arguments."""
    r = random.Random(total * 31 + parts)
    w = [r.uniform(0.3, 1.7) for _ in range(parts)]
    out = [max(1, int(total * v / sum(w))) for v in w]
    out[0] += total - sum(out)
    if out[0] < 1:
        out = [total // parts + (i < total % parts) for i in range(parts)]
    return out


def _contexts(mean, rows):
    """``rows`` context lengths about ``mean``, the same for the same arguments."""
    r = random.Random(mean * 17 + rows)
    return [max(1, int(mean * r.uniform(0.5, 1.5))) for _ in range(rows)] if rows > 1 else [mean]


def _gen(seed):
    return torch.Generator(DEV).manual_seed(int(seed) * 7 + 3)


def _normal(g, *shape, std=1.0, dtype=torch.bfloat16):
    """Random values, filled a slice at a time where the tensor is large."""
    out = torch.empty(shape, dtype=dtype, device=DEV)
    return out.normal_(0.0, std, generator=g)


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def _lengths(case):
    """(rows each sequence brings, its length with them), decoded sequences first."""
    kind = case["kind"]
    if kind == "layer":
        ctx = _contexts(case["context"], case["decodes"]) if case["decodes"] else []
        pre = _split(case["tokens"], case["prompts"]) if case["prompts"] else []
        return [1] * len(ctx) + pre, ctx + pre
    if kind in ("attention", "latent"):
        if case["new"] == 1:
            ctx = _contexts(case["context"], case["rows"])
            return [1] * case["rows"], ctx
        new = _split(case["new"] * case["rows"], case["rows"])
        return new, [n + case["context"] - case["new"] for n in new]
    new = _split(case["tokens"], case["rows"]) if case["tokens"] > case["rows"] else [1] * case["rows"]
    return new, [n + (100 if n == 1 or i % 2 else 0) for i, n in enumerate(new)]    # every other prompt goes on from a state


def _paging(g, new, lens):
    """Cache blocks in no order, and where each sequence's tokens are."""
    per = [-(-n // BLOCK) for n in lens]
    total = sum(per) + 1
    order = torch.randperm(total, generator=g, device=DEV).to(torch.int32)
    first = torch.tensor([0] + per[:-1], device=DEV).cumsum(0)
    width = max(per)
    col = torch.arange(width, device=DEV)
    table = order[(first[:, None] + col).clamp(max=total - 1)]
    table = torch.where(col < _i32(per)[:, None], table, torch.zeros_like(table)).contiguous()
    qsl = torch.tensor([0] + new, device=DEV).cumsum(0).to(torch.int32)
    seq = torch.repeat_interleave(torch.arange(len(new), device=DEV), _i32(new))
    pos = torch.arange(sum(new), device=DEV) - qsl[seq].long() + (_i32(lens) - _i32(new))[seq]
    slots = (table[seq, pos // BLOCK].long() * BLOCK + pos % BLOCK).to(torch.int32)
    return {"blocks": total, "table": table, "qsl": qsl, "seq": seq.to(torch.int32), "pos": pos.to(torch.int32), "slots": slots,
            "lens": _i32(lens)}


def _history(p, values):
    """``values [blocks * BLOCK, ...]`` as each sequence's tokens in order: index of every (sequence, position)."""
    return lambda i, n: values[(p["table"][i, torch.arange(n, device=DEV) // BLOCK].long() * BLOCK
                                + torch.arange(n, device=DEV) % BLOCK)]


# ------------------------------------------------------------------ a dense decoder layer
def _layer_inputs(case, seed):
    h, f, hq, hkv, _ = DENSE[case["model"]]
    d, g = 128, _gen(seed)
    new, lens = _lengths(case)
    p = _paging(g, new, lens)
    n = p["blocks"] * BLOCK
    w = {"table": _normal(g, VOCAB, h), "qkv": _normal(g, (hq + 2 * hkv) * d, h, std=h ** -0.5),
         "o": _normal(g, h, hq * d, std=(hq * d) ** -0.5), "gate_up": _normal(g, 2 * f, h, std=h ** -0.5),
         "down": _normal(g, h, f, std=2.0 * f ** -0.5)}
    for name in ("n1", "n2", "n3"):
        w[name] = (1.0 + 0.1 * _normal(g, h, dtype=torch.float32)).bfloat16()
    ids = torch.randint(0, VOCAB, (sum(new),), generator=g, device=DEV, dtype=torch.int32)
    return {"new": new, "lens": lens, "p": p, "w": w, "ids": ids, "k": _normal(g, n, hkv, d), "v": _normal(g, n, hkv, d)}


def _layer_prepare(case, seed):
    from vllm_distributed_amd import ops
    from vllm_distributed_amd.models.layers.attention import AttentionMetadata, RMSNorm, set_forward_context
    from vllm_distributed_amd.models.layers.linear import pad_dense_weight_rows
    from vllm_distributed_amd.models.llama import LlamaDecoderLayer
    from vllm_distributed_amd.ops import hip
    h, f, hq, hkv, base = DENSE[case["model"]]
    x = _layer_inputs(case, seed)
    p, w, d = x["p"], x["w"], 128
    cfg = {"model_type": "llama", "hidden_size": h, "intermediate_size": f, "num_attention_heads": hq,
           "num_key_value_heads": hkv, "rms_norm_eps": 1e-5, "hidden_act": "silu", "num_hidden_layers": 1}
    longest = max(x["lens"])
    with torch.device(DEV):
        layer = LlamaDecoderLayer(cfg, 0, torch.bfloat16,
                                  ops.build_cos_sin_cache(d, -(-longest // BLOCK) * BLOCK, base, None).to(DEV))
        norm = RMSNorm(h, 1e-5, torch.bfloat16)
    for mod, name in ((layer.self_attn.qkv_proj, "qkv"), (layer.self_attn.o_proj, "o"), (layer.mlp.gate_up_proj, "gate_up"),
                      (layer.mlp.down_proj, "down"), (layer.input_layernorm, "n1"), (layer.post_attention_layernorm, "n2"),
                      (norm, "n3")):
        mod.weight.data = w[name]
    pad_dense_weight_rows(layer, 128)
    kc = torch.zeros(ops.k_cache_shape(p["blocks"], hkv, d, BLOCK), dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros(ops.v_cache_shape(p["blocks"], hkv, d, BLOCK), dtype=torch.bfloat16, device=DEV)
    ops.reshape_and_cache(x["k"], x["v"], kc, vc, torch.arange(p["blocks"] * BLOCK, device=DEV, dtype=torch.int32))
    layer.self_attn.attn.bind_kv_cache(kc, vc)
    nd, npre = case["decodes"], case["prompts"]
    most = max(x["lens"][:nd]) if nd else 0
    md = AttentionMetadata(
        num_decodes=nd, num_decode_tokens=nd, num_prefills=npre, num_prefill_tokens=case["tokens"], slot_mapping=p["slots"],
        block_table=p["table"], seq_lens=p["lens"], query_start_loc=p["qsl"], max_query_len=max(x["new"]), max_seq_len=longest,
        prefill_query_start_loc=(p["qsl"][nd:] - nd).contiguous() if npre else None,
        max_prefill_query_len=max(x["new"][nd:]) if npre else 0, max_decode_seq_len=most, prefill_fresh=npre > 0,
        decode_workspace=torch.empty(hip.decode_workspace_floats(nd, hq, d, hkv, most), dtype=torch.float32, device=DEV)
        if nd else None)

    @torch.inference_mode()
    def step():
        set_forward_context(md, p["pos"])
        hidden, residual = layer(p["pos"], ops.embedding(x["ids"], w["table"]), None)
        set_forward_context(None)
        if hidden is None:
            return norm(residual), residual
        return norm(hidden, residual)

    # (the modules own the weights now: the plain copies go)
    state = {"kind": "layer", "step": step, "caches": (kc, vc), "graph": None, "out": None}
    for name in ("qkv", "o", "gate_up", "down"):
        del w[name]
    x["k"] = x["v"] = None
    if npre == 0:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):
                step()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["out"] = step()
    return state


def _layer_run(s):
    if s["graph"] is not None:
        s["graph"].replay()
        hidden, residual = s["out"]
    else:
        hidden, residual = s["step"]()
    return {"hidden": hidden, "residual": residual, "k_cache": s["caches"][0], "v_cache": s["caches"][1]}


def _rms64(x, w, eps=1e-5):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w.double()


def _rope64(x, pos, base):
    d = x.shape[-1]
    a = pos.double()[:, None] * float(base) ** (-torch.arange(0, d, 2, device=DEV, dtype=torch.float64) / d)
    cos, sin = a.cos()[:, None], a.sin()[:, None]
    lo, hi = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([lo * cos - hi * sin, hi * cos + lo * sin], -1)


def _attend64(q, k, v, scale):
    """Causal attention of the last ``q.shape[0]`` positions, heads one at a time."""
    nq, hq, d = q.shape
    n, hkv = k.shape[0], k.shape[1]
    out = torch.empty_like(q)
    mask = torch.arange(n, device=DEV)[None] > torch.arange(n - nq, n, device=DEV)[:, None] if nq > 1 else None
    if nq == 1:
        s = torch.einsum("hgd,nhd->hgn", q[0].view(hkv, -1, d), k) * scale
        return torch.einsum("hgn,nhd->hgd", s.softmax(-1), v).reshape(1, hq, d)
    for j in range(hq):
        s = (q[:, j] @ k[:, j * hkv // hq].t()).mul_(scale).masked_fill_(mask, float("-inf"))
        out[:, j] = s.softmax(-1) @ v[:, j * hkv // hq]
    return out


def _layer_exact(case, seed):
    h, f, hq, hkv, base = DENSE[case["model"]]
    x = _layer_inputs(case, seed)
    p, w, d = x["p"], x["w"], 128
    res = w["table"][x["ids"].long()].double()
    qkv = _rms64(res, w["n1"]) @ w["qkv"].double().t()
    q, k, v = qkv.split([hq * d, hkv * d, hkv * d], -1)
    q = _rope64(q.reshape(-1, hq, d), p["pos"], base)
    k = _rope64(k.reshape(-1, hkv, d), p["pos"], base)
    v = v.reshape(-1, hkv, d)
    past_k, past_v = _history(p, x["k"]), _history(p, x["v"])
    out = torch.empty_like(q)
    at = 0
    for i, (n, ln) in enumerate(zip(x["new"], x["lens"])):
        kk = torch.cat([past_k(i, ln - n).double(), k[at:at + n]])
        vv = torch.cat([past_v(i, ln - n).double(), v[at:at + n]])
        out[at:at + n] = _attend64(q[at:at + n], kk, vv, d ** -0.5)
        at += n
    res = res + out.reshape(-1, hq * d) @ w["o"].double().t()
    g, u = (_rms64(res, w["n2"]) @ w["gate_up"].double().t()).split(f, -1)
    res = res + (torch.nn.functional.silu(g) * u) @ w["down"].double().t()
    return {"hidden": _rms64(res, w["n3"]), "residual": res, "k_cache": None, "v_cache": None}


# ------------------------------------------------------------------ attention over a paged cache
def _attention_inputs(case, seed):
    g = _gen(seed)
    new, lens = _lengths(case)
    p = _paging(g, new, lens)
    n, t, hq, hkv, d = p["blocks"] * BLOCK, sum(new), case["heads"], case["kv_heads"], case["dim"]
    return {"new": new, "lens": lens, "p": p, "q": _normal(g, t, hq, d, std=1.3), "k": _normal(g, n, hkv, d),
            "v": _normal(g, n, hkv, d), "k_new": _normal(g, t, hkv, d), "v_new": _normal(g, t, hkv, d)}


def _attention_prepare(case, seed):
    from vllm_distributed_amd import ops
    x = _attention_inputs(case, seed)
    p, hkv, d = x["p"], case["kv_heads"], case["dim"]
    dt = torch.float8_e4m3fn if case["cache"] == "fp8" else torch.bfloat16
    kc = torch.zeros(ops.k_cache_shape(p["blocks"], hkv, d, BLOCK), dtype=dt, device=DEV)
    vc = torch.zeros(ops.v_cache_shape(p["blocks"], hkv, d, BLOCK), dtype=dt, device=DEV)
    ops.reshape_and_cache(x["k"], x["v"], kc, vc, torch.arange(p["blocks"] * BLOCK, device=DEV, dtype=torch.int32))
    x["k"] = x["v"] = None
    return {"kind": "attention", "x": x, "caches": (kc, vc), "decode": case["new"] == 1, "scale": d ** -0.5}


def _attention_run(s):
    from vllm_distributed_amd import ops
    x, p, (kc, vc) = s["x"], s["x"]["p"], s["caches"]
    ops.reshape_and_cache(x["k_new"], x["v_new"], kc, vc, p["slots"])
    longest = max(x["lens"])
    if s["decode"]:
        out = ops.paged_attention_decode(x["q"], kc, vc, p["table"], p["lens"], s["scale"], longest)
    else:
        out = ops.paged_attention(x["q"], kc, vc, p["table"], p["qsl"], p["lens"], s["scale"], max(x["new"]), longest)
    # (an 8-bit cache is handed over as its bytes)
    return {"out": out, "k_cache": _whole(kc), "v_cache": _whole(vc)}


def _whole(cache):
    return cache.view(torch.uint8) if cache.dtype == torch.float8_e4m3fn else cache


def _attention_exact(case, seed):
    x = _attention_inputs(case, seed)
    p = x["p"]
    f8 = case["cache"] == "fp8"

    def kept(t):            # what the cache keeps of a value
        return t.float().clamp(-448, 448).to(torch.float8_e4m3fn).double() if f8 else t.double()
    past_k, past_v = _history(p, x["k"]), _history(p, x["v"])
    out = torch.empty(x["q"].shape, dtype=torch.float64, device=DEV)
    at = 0
    for i, (n, ln) in enumerate(zip(x["new"], x["lens"])):
        kk = torch.cat([kept(past_k(i, ln - n)), kept(x["k_new"][at:at + n])])
        vv = torch.cat([kept(past_v(i, ln - n)), kept(x["v_new"][at:at + n])])
        out[at:at + n] = _attend64(x["q"][at:at + n].double(), kk, vv, case["dim"] ** -0.5)
        at += n
    return {"out": out, "k_cache": None, "v_cache": None}


# ------------------------------------------------------------------ latent attention
def _latent_inputs(case, seed):
    g = _gen(seed)
    new, lens = _lengths(case)
    p = _paging(g, new, lens)
    t, dk = sum(new), RANK + ROPE
    return {"new": new, "lens": lens, "p": p, "q": _normal(g, t, case["heads"], dk, std=0.8),
            "rows": _normal(g, p["blocks"] * BLOCK, dk), "latent": _normal(g, t, dk)}


LATENT_SCALE = (128 + ROPE) ** -0.5


def _latent_prepare(case, seed):
    from vllm_distributed_amd import ops
    x = _latent_inputs(case, seed)
    p = x["p"]
    kc = torch.zeros(ops.k_cache_shape(p["blocks"], 1, RANK + ROPE, BLOCK), dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros(ops.v_cache_shape(p["blocks"], 1, RANK, BLOCK), dtype=torch.bfloat16, device=DEV)
    ops.mla_cache_write(x["rows"], kc, vc, torch.arange(p["blocks"] * BLOCK, device=DEV, dtype=torch.int32))
    x["rows"] = None
    decode = case["new"] == 1
    return {"kind": "latent", "x": x, "caches": (kc, vc), "seq": None if decode else p["seq"],
            "keys": p["lens"] if decode else p["pos"] + 1}


def _latent_run(s):
    from vllm_distributed_amd import ops
    x, p, (kc, vc) = s["x"], s["x"]["p"], s["caches"]
    ops.mla_cache_write(x["latent"], kc, vc, p["slots"])
    out = ops.mla_attention(x["q"], kc, vc, p["table"], s["seq"], s["keys"], LATENT_SCALE, max(x["lens"]))
    return {"out": out, "k_cache": kc, "v_cache": vc}


def _latent_exact(case, seed):
    x = _latent_inputs(case, seed)
    past = _history(x["p"], x["rows"])
    out = torch.empty(x["q"].shape[:2] + (RANK,), dtype=torch.float64, device=DEV)
    at = 0
    for i, (n, ln) in enumerate(zip(x["new"], x["lens"])):
        rows = torch.cat([past(i, ln - n).double(), x["latent"][at:at + n].double()])
        mask = torch.arange(ln, device=DEV)[None] > torch.arange(ln - n, ln, device=DEV)[:, None]
        for lo in range(0, n, 64):
            q = x["q"][at + lo:at + min(lo + 64, n)].double()
            sc = torch.einsum("thd,nd->thn", q, rows) * LATENT_SCALE
            sc = sc.masked_fill(mask[lo:lo + 64, None], float("-inf"))
            out[at + lo:at + min(lo + 64, n)] = sc.softmax(-1) @ rows[:, :RANK]
        at += n
    return {"out": out, "k_cache": None, "v_cache": None}


# ------------------------------------------------------------------ sparse experts
def _expert_inputs(case, seed):
    """Rows that, as in a trained model, lie towards the router rows of the experts they are for; some experts are
    asked for more than others."""
    h, inter, e, k = EXPERTS[case["model"]]
    g, t = _gen(seed), case["tokens"]
    router = _normal(g, e, h, std=h ** -0.5)
    wish = 1.0 / (torch.arange(e, device=DEV, dtype=torch.float32) + 0.5 * e)
    chosen = torch.multinomial(wish[torch.randperm(e, generator=g, device=DEV)].expand(t, e), k, generator=g)
    pull = 8.0 + 4.0 * torch.rand(t, k, generator=g, device=DEV)
    x = torch.randn(t, h, generator=g, device=DEV)
    for j in range(k):
        x += pull[:, j:j + 1] * router[chosen[:, j]].float()
    out = {"x": x.bfloat16(), "router": router}
    if case["weights"] == "awq":
        for name, n, kk in (("13", 2 * inter, h), ("2", h, inter)):
            out["qw" + name] = torch.randint(-2 ** 31, 2 ** 31, (e, n // 16, kk // 128, 64, 4), generator=g, device=DEV,
                                             dtype=torch.int32)
            scale = kk ** -0.5 / 4.6 * (0.5 + torch.rand(e, n // 16, kk // 128, 16, generator=g, device=DEV))
            zero = torch.randint(6, 10, scale.shape, generator=g, device=DEV).float() + 128.0
            out["sz" + name] = torch.stack([scale, zero], -1).bfloat16()
    else:
        out["w13"] = _normal(g, e, 2 * inter, h, std=h ** -0.5)
        out["w2"] = _normal(g, e, h, inter, std=inter ** -0.5)
    return out


def _experts_prepare(case, seed):
    from vllm_distributed_amd.models.layers.linear import QuantSpec
    from vllm_distributed_amd.models.layers.moe import FusedMoE
    h, inter, e, k = EXPERTS[case["model"]]
    x = _expert_inputs(case, seed)
    awq = case["weights"] == "awq"
    with torch.device(DEV):
        block = FusedMoE(h, inter, e, k, True, torch.bfloat16, allocate_experts=False)
    block.gate.weight.data = x["router"]
    if awq:
        block.quant = QuantSpec("awq", 128)
        for name in ("qw13", "sz13", "qw2", "sz2"):
            setattr(block, name, x[name])
    else:
        block.w13, block.w2 = (torch.nn.Parameter(x[n], requires_grad=False) for n in ("w13", "w2"))
    return {"kind": "experts", "block": block, "x": x["x"]}


@torch.inference_mode()
def _experts_run(s):
    return s["block"](s["x"])


def _w4_64(qw, sz):
    """Dense rows of one expert's packed weights (the layout is ops/quant.py's)."""
    w = qw.long()
    v = torch.stack([(w >> (4 * ((e >> 1) + 4 * (e & 1)))) & 15 for e in range(8)], -1)     # nt kb lane word e
    nt, kb = qw.shape[:2]
    q = v.view(nt, kb, 4, 16, 4, 8).permute(0, 3, 1, 2, 4, 5).reshape(nt, 16, kb, 128).double()
    s, z = sz[..., 0].double().permute(0, 2, 1), sz[..., 1].double().permute(0, 2, 1) - 128.0
    return ((q - z[..., None]) * s[..., None]).reshape(nt * 16, kb * 128)


def _experts_exact(case, seed):
    h, inter, e, k = EXPERTS[case["model"]]
    x = _expert_inputs(case, seed)
    xd = x["x"].double()
    probs, idx = (xd @ x["router"].double().t()).softmax(-1).topk(k, -1)
    probs = probs / probs.sum(-1, keepdim=True)
    out = torch.zeros_like(xd)
    for j in range(e):
        t, c = torch.nonzero(idx == j, as_tuple=True)
        if t.numel() == 0:
            continue
        w13, w2 = ((_w4_64(x["qw13"][j], x["sz13"][j]), _w4_64(x["qw2"][j], x["sz2"][j])) if case["weights"] == "awq"
                   else (x["w13"][j].double(), x["w2"][j].double()))
        gate, up = (xd[t] @ w13.t()).split(inter, -1)
        out.index_add_(0, t, (torch.nn.functional.silu(gate) * up) @ w2.t() * probs[t, c, None])
    return out


# ------------------------------------------------------------------ mixers with per-request state
def _recurrence_inputs(case, seed):
    g = _gen(seed)
    new, lens = _lengths(case)
    t, h, gr, d, vd, op = sum(new), case["heads"], case["groups"], case["dim"], case["vdim"], case["op"]
    out = {"new": new, "lens": lens}
    cols = h * vd + 2 * gr * d
    out["x"] = _normal(g, t, cols + h * vd)[:, :cols]          # the layer's fused projection is wider: rows are strided
    out["state"] = _normal(g, len(new) + 1, h, d, vd, std=0.3, dtype=torch.float32)
    out["slots"] = torch.randperm(len(new) + 1, generator=g, device=DEV)[:len(new)].to(torch.int32)
    channels = h * d if op == "delta_channel" else h
    if op in ("delta_channel", "delta_head", "state_space"):
        step = torch.exp(torch.empty(channels, device=DEV).uniform_(math.log(1e-3), math.log(1e-1), generator=g))
        out["dt"] = _normal(g, t, channels, std=0.5)
        out["dt_bias"] = step + torch.log(-torch.expm1(-step))          # softplus of it is the step
        out["a_log"] = torch.log(torch.empty(h, device=DEV).uniform_(1.0, 16.0, generator=g))
        out["beta"] = _normal(g, t, h)
        out["skip"] = 1.0 + 0.1 * torch.randn(h, generator=g, device=DEV)
    elif op == "linear_channel":
        out["decay"] = torch.sigmoid(2.0 + torch.randn(t, h * d, generator=g, device=DEV)) ** (1.0 / 16.0)
    else:
        out["decay"] = 1.0 - 2.0 ** -(2.0 + 6.0 * torch.arange(h, device=DEV, dtype=torch.float32) / max(h - 1, 1))
    return out


def _recurrence_prepare(case, seed):
    x = _recurrence_inputs(case, seed)
    return {"kind": "recurrence", "case": case, "x": x, "qsl": torch.tensor([0] + x["new"]).cumsum(0).to(torch.int32).to(DEV),
            "lens": _i32(x["lens"]), "most": max(x["new"])}


def _recurrence_run(s):
    from vllm_distributed_amd import ops
    c, x, op = s["case"], s["x"], s["case"]["op"]
    at = (x["state"], x["slots"], s["qsl"], s["lens"])
    if op in ("delta_channel", "delta_head"):
        out = ops.gated_delta_rule(x["x"], c["heads"], c["groups"], c["dim"], c["vdim"], x["beta"], x["dt"], x["dt_bias"],
                                   x["a_log"], *at, 1e-6, s["most"])
    elif op == "state_space":
        out = ops.selective_scan(x["x"], x["dt"], c["heads"], c["groups"], c["vdim"], c["dim"], x["a_log"], x["dt_bias"],
                                 x["skip"], *at, s["most"])
    elif op == "linear_channel":
        out = ops.decay_linear_attention(x["x"], c["heads"], c["dim"], c["vdim"], x["decay"], *at, False, s["most"],
                                         c["dim"] ** -0.5)
    else:
        out = ops.decay_linear_attention(x["x"], c["heads"], c["dim"], c["vdim"], x["decay"], *at, True, s["most"])
    return {"out": out, "state": x["state"]}


def _recurrence_exact(case, seed):
    x = _recurrence_inputs(case, seed)
    h, gr, d, vd, op = case["heads"], case["groups"], case["dim"], case["vdim"], case["op"]
    xd = x["x"].double()
    t = xd.shape[0]
    beta = q_scale = skip = None
    if op == "state_space":
        v, k, q = xd.split([h * vd, gr * d, gr * d], -1)
    else:
        q, k, v = xd.split([gr * d, gr * d, h * vd], -1)
    q, k, v = q.reshape(t, gr, d), k.reshape(t, gr, d), v.reshape(t, h, vd)
    if op.startswith("delta"):
        q = q * torch.rsqrt(q.pow(2).sum(-1, keepdim=True) + 1e-6) * d ** -0.5
        k = k * torch.rsqrt(k.pow(2).sum(-1, keepdim=True) + 1e-6)
        beta = torch.sigmoid(x["beta"].double())
    if op == "linear_head":
        q, k, v = (torch.nn.functional.silu(z) for z in (q, k, v))
    if "dt" in x:
        step = torch.nn.functional.softplus(x["dt"].double() + x["dt_bias"].double(), threshold=60.0).reshape(t, h, -1)
        decay = torch.exp(-torch.exp(x["a_log"].double()).view(1, h, 1) * step)
        if op == "state_space":
            skip = x["skip"].double().view(1, h, 1) * v
            v = v * step
    elif op == "linear_channel":
        decay, q_scale = x["decay"].double().view(t, h, d), d ** -0.5
    else:
        decay = x["decay"].double().view(1, h, 1).expand(t, h, 1)
    q, k = q.repeat_interleave(h // gr, 1), k.repeat_interleave(h // gr, 1)
    new, lens = x["new"], x["lens"]
    order = sorted(range(len(new)), key=lambda i: -new[i])      # the longest first: the running ones are a prefix
    first = [sum(new[:i]) for i in range(len(new))]
    first_t = torch.tensor([first[i] for i in order], device=DEV)
    slots = x["slots"].long()[order]
    fresh = torch.tensor([lens[i] == new[i] for i in order], device=DEV)
    S = x["state"].double()[slots].masked_fill(fresh.view(-1, 1, 1, 1), 0.0)
    out = torch.empty(t, h, vd, dtype=torch.float64, device=DEV)
    n = len(new)
    for r in range(max(new)):
        while new[order[n - 1]] <= r:
            n -= 1
        at = first_t[:n] + r
        kr, Sn = k[at].unsqueeze(3), S[:n]
        Sn *= decay[at].unsqueeze(3)
        u = v[at].unsqueeze(2)
        if beta is not None:
            u = beta[at].view(n, h, 1, 1) * (u - kr.transpose(2, 3) @ Sn)
        Sn += kr * u
        out[at] = (q[at].unsqueeze(2) @ Sn).squeeze(2)
    if q_scale is not None:
        out *= q_scale
    if skip is not None:
        out += skip
    state = x["state"].double()
    state[slots] = S
    return {"out": out.reshape(t, h * vd), "state": state}


# ------------------------------------------------------------------ sampling
def _sample_prepare(case, seed):
    g, b, v = _gen(seed), case["rows"], case["vocab"]
    logits = torch.randn(b, v, generator=g, device=DEV) * 2.2
    sharp = torch.randint(0, v, (b, 12), generator=g, device=DEV)           # a few likely continuations
    logits.scatter_(1, sharp, 9.0 + 4.0 * torch.rand(b, 12, generator=g, device=DEV))
    pick = torch.arange(b, device=DEV)
    return {"kind": "sample", "logits": logits.to(torch.bfloat16 if case["dtype"] == "bf16" else torch.float32),
            "temperature": torch.where(pick % 8 == 7, 0.0, 0.6 + 0.6 * torch.rand(b, generator=g, device=DEV)),
            "top_k": torch.where(pick % 3 == 0, 50, torch.where(pick % 3 == 1, 0, 20)).to(torch.int32),
            "top_p": torch.where(pick % 4 == 0, 1.0, 0.95 - 0.05 * (pick % 2)).float(),
            "min_p": torch.where(pick % 5 == 0, 0.05, 0.0).float(),
            "uniform": torch.rand(b, generator=g, device=DEV).clamp(1e-6, 1 - 1e-6)}


def _sample_run(s):
    from vllm_distributed_amd import ops
    return ops.sample(s["logits"], s["temperature"], s["top_k"], s["top_p"], s["min_p"], s["uniform"])


# ------------------------------------------------------------------ what is asked of this file
_PREPARE = {"layer": _layer_prepare, "attention": _attention_prepare, "latent": _latent_prepare, "experts": _experts_prepare,
            "recurrence": _recurrence_prepare, "sample": _sample_prepare}
_RUN = {"layer": _layer_run, "attention": _attention_run, "latent": _latent_run, "experts": _experts_run,
        "recurrence": _recurrence_run, "sample": _sample_run}
_EXACT = {"layer": _layer_exact, "attention": _attention_exact, "latent": _latent_exact, "experts": _experts_exact,
          "recurrence": _recurrence_exact}


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["kind"]](state)


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed) if case["kind"] in _EXACT else None


def _pairs(new, lens):
    """(query, key) pairs of causal attention."""
    return sum(n * (ln - n) + n * (n + 1) // 2 for n, ln in zip(new, lens))


def work(case):
    kind = case["kind"]
    if kind == "sample":
        return {"bytes": case["rows"] * case["vocab"] * (2 if case["dtype"] == "bf16" else 4), "flops": 0}
    if kind == "experts":
        h, inter, e, k = EXPERTS[case["model"]]
        t = case["tokens"]
        used = min(e, e * (1.0 - (1.0 - k / e) ** t))                       # experts that some row is for
        size = 0.5 + 4.0 / 128 if case["weights"] == "awq" else 2.0
        return {"bytes": used * 3 * h * inter * size + e * h * 2 + 4 * t * h, "flops": 2.0 * t * (3 * h * inter * k + e * h)}
    new, lens = _lengths(case)
    t, keys, pairs = sum(new), sum(lens), _pairs(new, lens)
    if kind == "layer":
        h, f, hq, hkv, _ = DENSE[case["model"]]
        params = h * (2 * hq + 2 * hkv) * 128 + 3 * h * f
        return {"bytes": 2 * params + 4 * keys * hkv * 128 + 6 * t * h, "flops": 2.0 * t * params + 4.0 * pairs * hq * 128}
    if kind == "attention":
        hq, hkv, d = case["heads"], case["kv_heads"], case["dim"]
        return {"bytes": 2 * keys * hkv * d * (1 if case["cache"] == "fp8" else 2) + 4 * t * hq * d + 4 * t * hkv * d,
                "flops": 4.0 * pairs * hq * d}
    if kind == "latent":
        hq = case["heads"]
        return {"bytes": 2 * keys * (RANK + ROPE) + 2 * t * hq * (2 * RANK + ROPE), "flops": 2.0 * pairs * hq * (2 * RANK + ROPE)}
    h, gr, d, vd, op = case["heads"], case["groups"], case["dim"], case["vdim"], case["op"]
    wide = {"delta_channel": 2 * h * d, "linear_channel": 4 * h * d}.get(op, 2 * h)
    return {"bytes": t * (2 * (h * vd + 2 * gr * d) + wide + 4 * h * vd) + 8 * len(new) * h * d * vd,
            "flops": t * h * d * vd * (6.0 if op.startswith("delta") else 4.0)}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return {"rel": 0.0, "differ": 0.01}     # whole numbers: a row whose draw falls on the border of two tokens
    if kind == "recurrence":
        return {"rel": 1e-5, "max": 1e-3}       # 32-bit sums over up to thousands of rows
    if kind == "attention":
        return {"rel": 0.01, "max": 0.2, "differ": 0.01}
    if kind == "experts":
        return {"rel": 0.03, "max": 0.5}        # as below, and a weighted sum of up to eight rows, kept in 16 bits or in 32
    return {"rel": 0.012, "max": 0.25}          # 16-bit values between the matrix products
