"""The work a serving program has this library do, as cases that can be timed and checked.

Six kinds of call, each through the public entry points and over the sizes that serving meets:

* ``decode_attention``: one new token per request, its K/V stored and attended over the paged
  cache (``BaseAttention.write_kv``, ``AttentionBatch.forward``), for one request up to 256,
  short contexts to long ones, pages of 1 and 16 tokens;
* ``prefill_attention``: causal prefill of a ragged batch, with and without a cached prefix;
* ``decode_layer``: a decoder layer's projections and norms for 1 to 256 decode rows (QKV with
  QK-norm, RoPE and K/V store; o_proj with its residual norm; gate_up with SiLU x mul; down with
  its residual norm);
* ``prefill_ops``: the layer passes between the library GEMMs of a prefill (residual norm,
  QK-norm / RoPE / K/V store, SiLU x mul);
* ``sample``: joint top-k / top-p sampling of a batch of logits rows;
* ``model``: a whole decode step or prefill of the Qwen3 model, logits returned.

Decode calls are short and a serving program replays them from a HIP graph; cases with ``graph``
hold such a graph (captured in ``prepare``, re-planned where the engine re-plans), the others
launch eagerly. ``layers`` is how many layers share the plan in one pass, as in a forward.
Request lengths come from the case itself (``lengths``), values from the seed.
"""
from __future__ import annotations

import dataclasses
import math
import random

import torch

from llm_infer_rust_amd import ops
from llm_infer_rust_amd.backend import (Attention, AttentionMetadata, AttentionSpec, BatchPhase,
                                        DecodeHostMetadata)
from llm_infer_rust_amd.kv_cache import BaseAttention, KVCacheLayout, KVCachePool
from llm_infer_rust_amd.model import Qwen3Config, Qwen3Model
from llm_infer_rust_amd.sampling import Sampler, SamplingParams

D = 128  # head dim
EPS = 1e-6
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
WIDTHS = {"8b": Qwen3Config.qwen3_8b(), "0.6b": Qwen3Config.qwen3_0_6b()}
VOCAB = 151936


def _decode(name, rows, lo, hi, hq, hkv, page, layers, graph, dtype="bf16", lengths=2):
    c = dict(kind="decode_attention", rows=rows, lo=lo, hi=hi, q_heads=hq, kv_heads=hkv,
             page=page, layers=layers, graph=graph, dtype=dtype, lengths=lengths)
    return dict(c, name=name) if name else c


def _prefill(name, requests, lo, hi, prefix_lo, prefix_hi, hq, hkv, page, dtype="bf16",
             lengths=3):
    c = dict(kind="prefill_attention", requests=requests, lo=lo, hi=hi, prefix_lo=prefix_lo,
             prefix_hi=prefix_hi, q_heads=hq, kv_heads=hkv, page=page, dtype=dtype,
             lengths=lengths)
    return dict(c, name=name) if name else c


def _layer(name, rows, width, layers, graph, dtype="bf16"):
    c = dict(kind="decode_layer", rows=rows, width=width, layers=layers, graph=graph,
             dtype=dtype)
    return dict(c, name=name) if name else c


def _ops(name, tokens, width, dtype="bf16"):
    c = dict(kind="prefill_ops", tokens=tokens, width=width, dtype=dtype)
    return dict(c, name=name) if name else c


def _sample(name, rows, vocab, mix, dtype="bf16"):
    c = dict(kind="sample", rows=rows, vocab=vocab, mix=mix, dtype=dtype)
    return dict(c, name=name) if name else c


def _model(name, phase, rows, lo, hi, width, layers, lengths=5):
    c = dict(kind="model", phase=phase, rows=rows, lo=lo, hi=hi, width=width, layers=layers,
             lengths=lengths)
    return dict(c, name=name) if name else c


def listed():
    return [
        # One interactive user: a single request of an odd length, replayed layers.
        _decode("decode_attn_single", 1, 1337, 1337, 32, 8, 16, 8, True),
        # Isolated paged decode, batch 64, ragged contexts over single-token pages.
        _decode("decode_attn_page1", 64, 512, 4096, 16, 8, 1, 1, False),
        # A full serving batch in the middle of its outputs, pages of 16.
        _decode("decode_attn_serving", 256, 1248, 1312, 32, 8, 16, 1, True),
        # A batch of fresh prompts, no cached prefix.
        _prefill("prefill_ragged", 8, 256, 2048, 0, 0, 16, 8, 16),
        # Prompts that continue long cached prefixes.
        _prefill("prefill_cached", 16, 64, 512, 1024, 8192, 32, 8, 16, lengths=4),
        # The layer around the attention for one user ...
        _layer("layer_one_row", 1, "8b", 1, True),
        # ... for a small model under a middling, odd batch in fp16 ...
        _layer("layer_small_model", 45, "0.6b", 4, True, "fp16"),
        # ... and for a full serving batch.
        _layer("layer_serving", 256, "8b", 1, True),
        # The sampler behind a full serving batch, one parameter set.
        _sample("sample_serving", 256, VOCAB, "joint"),
        # The sampler for a handful of users with settings of their own.
        _sample("sample_few", 5, VOCAB, "mixed"),
        # A full prefill chunk (8,192 tokens): the passes between its GEMMs.
        _ops("prefill_ops", 8192, "8b"),
        # A whole decode step of a moderately loaded server (four layers and the head).
        _model("model_decode", "decode", 24, 300, 1500, "8b", 4),
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5))))))


def draw(rng: random.Random):
    kind = rng.choice(["decode_attention", "prefill_attention", "decode_layer", "prefill_ops",
                       "sample", "model"])
    dtype = "bf16" if rng.random() < 0.75 else "fp16"
    seed = rng.randrange(1 << 20)
    if kind == "decode_attention":
        hq, hkv = rng.choice([(16, 8), (32, 8), (32, 8), (8, 8), (32, 4)])
        rows = _log_int(rng, 1, 256)
        # at most 1.4 GB of K/V in a pass, as the full serving batch reads
        most = max(16, 340_000 * 8 // hkv // rows)
        hi = _log_int(rng, 16, min(32768, most))
        lo = max(1, round(hi * rng.choice([0.1, 0.5, 1.0])))
        layers = 8 if rows * hi <= 16384 else 1
        return _decode(None, rows, lo, hi, hq, hkv, rng.choice([1, 16, 16]), layers,
                       rng.random() < 0.75, dtype, seed)
    if kind == "prefill_attention":
        hq, hkv = rng.choice([(16, 8), (32, 8)])
        requests = _log_int(rng, 1, 16)
        hi = _log_int(rng, 17, min(2048, 8192 // requests))
        lo = max(1, round(hi * rng.choice([0.1, 0.5, 1.0])))
        cached = rng.random() < 0.5
        # at most 400 GFLOP in a pass
        most = int(3.5e11 / (4 * hq * D * requests * hi))
        prefix = _log_int(rng, 16, max(17, min(8192, most))) if cached else 0
        return _prefill(None, requests, lo, hi, prefix // 4, prefix, hq, hkv, 16, dtype, seed)
    if kind == "decode_layer":
        width = rng.choice(["8b", "8b", "0.6b"])
        rows = _log_int(rng, 1, 256)
        return _layer(None, rows, width, 1 if width == "8b" else 4, True, dtype)
    if kind == "prefill_ops":
        return _ops(None, _log_int(rng, 16, 8192), rng.choice(["8b", "0.6b"]), dtype)
    if kind == "sample":
        rows = _log_int(rng, 1, 256)
        vocab = rng.choice([VOCAB, VOCAB, _log_int(rng, 1000, VOCAB)])
        return _sample(None, rows, vocab, rng.choice(["joint", "mixed", "greedy", "top_p"]),
                       rng.choice(["bf16", "bf16", "fp16", "fp32"]))
    width = rng.choice(["8b", "0.6b"])
    if rng.random() < 0.7:
        hi = _log_int(rng, 64, 2048)
        return _model(None, "decode", _log_int(rng, 1, 64), max(1, hi // 4), hi, width, 2, seed)
    hi = _log_int(rng, 17, 512)
    return _model(None, "prefill", _log_int(rng, 1, 4), max(1, hi // 2), hi, width, 2, seed)


# ------------------------------------------------------------------ inputs (plain torch)
def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, dtype, scale=1.0):
    t = torch.empty(*shape, dtype=dtype, device="cuda").normal_(0.0, 1.0, generator=g)
    return t if scale == 1.0 else t.mul_(scale)


def _gamma(g, n, dtype):
    return torch.empty(n, dtype=torch.float32, device="cuda").uniform_(
        0.5, 1.5, generator=g).to(dtype)


def _uniform_lengths(seed: int, n: int, lo: int, hi: int) -> list[int]:
    r = random.Random(seed)
    return [r.randint(lo, hi) for _ in range(n)]


def _paged(g, lengths, page, hkv, dtype, layers):
    """Random-page KV pools (one per layer) and the block table; page 0 is reserved."""
    per = [-(-n // page) for n in lengths]
    pages = sum(per)
    perm = torch.randperm(pages, generator=g, device="cuda").to(torch.int32) + 1
    table = torch.full((len(lengths), max(per)), -1, dtype=torch.int32, device="cuda")
    off = 0
    for b, n in enumerate(per):
        table[b, :n] = perm[off:off + n]
        off += n
    pools = [tuple(_randn(g, pages + 1, page, hkv, D, dtype=dtype) for _ in range(2))
             for _ in range(layers)]
    return table, pools


def _last_slots(table, lengths, page):
    last = torch.tensor(lengths, dtype=torch.int64, device="cuda") - 1
    rows = torch.arange(len(lengths), device="cuda")
    return table[rows, last // page].to(torch.int64) * page + last % page


def _bind(kc, vc) -> BaseAttention:
    cache = BaseAttention()
    cache.set_reserved_write_slot(0)
    cache.bind_kv_cache(kc, vc)
    return cache


def _captured(fn, keep=()):
    """fn's launches in a HIP graph (warmed up first on a side stream; ``keep``: buffers that fn
    updates in place, put back to what they were). Returns the graph and fn's captured outputs."""
    before = [t.clone() for t in keep]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    for t, b in zip(keep, before):
        t.copy_(b)
    return graph, out


# ------------------------------------------------------------------ decode attention
def _decode_inputs(case, seed):
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    b, hq, hkv, page = case["rows"], case["q_heads"], case["kv_heads"], case["page"]
    lengths = _uniform_lengths(case["lengths"], b, case["lo"], case["hi"])
    table, pools = _paged(g, lengths, page, hkv, dt, case["layers"])
    qkv = _randn(g, case["layers"], b, (hq + 2 * hkv) * D, dtype=dt)
    return lengths, table, pools, qkv


def _heads(qkv, hq, hkv):
    t = qkv.size(0)
    return (qkv[:, :hq * D].view(t, hq, D), qkv[:, hq * D:(hq + hkv) * D].view(t, hkv, D),
            qkv[:, (hq + hkv) * D:].view(t, hkv, D))


def _decode_prepare(case, seed):
    lengths, table, pools, qkv = _decode_inputs(case, seed)
    b, hq, hkv, page = case["rows"], case["q_heads"], case["kv_heads"], case["page"]
    loc = _last_slots(table, lengths, page)
    attn = Attention.new("mi355x", AttentionSpec(hq, hkv, D, DTYPES[case["dtype"]],
                                                 torch.device("cuda")))
    attn.bind_cache_layout(page)
    lens = torch.tensor(lengths, dtype=torch.int32, device="cuda")
    host = DecodeHostMetadata(lengths)
    meta = AttentionMetadata(BatchPhase.DECODE, decode_host=host, write_loc=loc,
                             block_table=table, cache_seqlens=lens)
    caches = [_bind(kc, vc) for kc, vc in pools]
    state = dict(kind=case["kind"], attn=attn, meta=meta, caches=caches, keep=(table, loc, qkv))
    if case["graph"]:
        state["plan"] = attn.prepare_decode_graph(meta)
    batch = attn.prepare(meta, b)

    def layers():
        out = []
        for cache, rows in zip(caches, qkv):
            q, k, v = _heads(rows, hq, hkv)
            cache.write_kv(k, v, loc)
            out.append(batch.forward(q, k, v, cache))
        return out

    state["pools"] = pools
    if case["graph"]:
        state["graph"], state["out"] = _captured(layers)
    else:
        state["fn"] = layers
    return state


def _attend64(q, k, v, causal_from=None):
    """q [n, hq, D] over k/v [t, hkv, D] in 64 bits; query i sees keys up to causal_from + i."""
    n, hq, _ = q.shape
    t, hkv, _ = k.shape
    qd = q.double().view(n, hkv, hq // hkv, D).permute(1, 2, 0, 3).reshape(hkv, -1, D)
    kd = k.double().transpose(0, 1).contiguous()
    s = torch.matmul(qd, kd.transpose(1, 2).contiguous()) / math.sqrt(D)
    if causal_from is not None:
        pos = torch.arange(n, device=q.device) + causal_from
        hidden = torch.arange(t, device=q.device)[None, :] > pos[:, None]
        s.view(hkv, hq // hkv, n, t).masked_fill_(hidden, float("-inf"))
    p = torch.softmax(s, -1)
    o = torch.matmul(p, v.double().transpose(0, 1).contiguous())
    return o.view(hkv, hq // hkv, n, D).permute(2, 0, 1, 3).reshape(n, hq * D)


def _request_slots(table, b, length, page):
    pos = torch.arange(length, device="cuda")
    return table[b, pos // page].to(torch.int64) * page + pos % page


def _decode_exact(case, seed):
    lengths, table, pools, qkv = _decode_inputs(case, seed)
    hq, hkv, page = case["q_heads"], case["kv_heads"], case["page"]
    loc = _last_slots(table, lengths, page)
    outs = []
    for (kc, vc), rows in zip(pools, qkv):
        q, k, v = _heads(rows, hq, hkv)
        kf, vf = kc.view(-1, hkv, D), vc.view(-1, hkv, D)
        kf[loc], vf[loc] = k, v
        out = [_attend64(q[b:b + 1], kf[s], vf[s]) for b, n in enumerate(lengths)
               for s in (_request_slots(table, b, n, page),)]
        outs.append(torch.cat(out))
    return {"out": outs, "caches": None}


# ------------------------------------------------------------------ prefill attention
def _prefill_lengths(case):
    new = _uniform_lengths(case["lengths"], case["requests"], case["lo"], case["hi"])
    pre = _uniform_lengths(case["lengths"] + 1, case["requests"], case["prefix_lo"],
                           case["prefix_hi"])
    return new, pre


def _bounds(new):
    out = [0]
    for n in new:
        out.append(out[-1] + n)
    return out


def _prefill_inputs(case, seed):
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    new, pre = _prefill_lengths(case)
    hq, hkv = case["q_heads"], case["kv_heads"]
    qkv = _randn(g, sum(new), (hq + 2 * hkv) * D, dtype=dt)
    lengths = [n + p for n, p in zip(new, pre)]
    table, pools = _paged(g, lengths, case["page"], hkv, dt, 1)
    if case["prefix_hi"]:  # the new tokens' K/V are in the cache when attention runs
        _, k, v = _heads(qkv, hq, hkv)
        b = _bounds(new)
        for r, (n, p) in enumerate(zip(new, pre)):
            s = _request_slots(table, r, n + p, case["page"])[p:]
            pools[0][0].view(-1, hkv, D)[s] = k[b[r]:b[r + 1]]
            pools[0][1].view(-1, hkv, D)[s] = v[b[r]:b[r + 1]]
    return new, pre, table, pools[0], qkv


def _prefill_meta(new, pre, table, loc=None):
    b = _bounds(new)
    return AttentionMetadata(
        BatchPhase.PREFILL, write_loc=loc,
        cu_seqlens_q=torch.tensor(b, dtype=torch.int32, device="cuda"),
        prefix_lens=torch.tensor(pre, dtype=torch.int32, device="cuda"), block_table=table,
        host_cu_seqlens_q=b, host_prefix_lens=list(pre))


def _prefill_prepare(case, seed):
    new, pre, table, (kc, vc), qkv = _prefill_inputs(case, seed)
    hq, hkv = case["q_heads"], case["kv_heads"]
    attn = Attention.new("mi355x", AttentionSpec(hq, hkv, D, DTYPES[case["dtype"]],
                                                 torch.device("cuda")))
    attn.bind_cache_layout(case["page"])
    meta = _prefill_meta(new, pre, table)
    return dict(kind=case["kind"], batch=attn.prepare(meta, sum(new)), attn=attn, meta=meta,
                heads=_heads(qkv, hq, hkv), cache=_bind(kc, vc))


def _prefill_exact(case, seed):
    new, pre, table, (kc, vc), qkv = _prefill_inputs(case, seed)
    hq, hkv = case["q_heads"], case["kv_heads"]
    q, k, v = _heads(qkv, hq, hkv)
    b, out = _bounds(new), []
    for r, (n, p) in enumerate(zip(new, pre)):
        ks, vs = k[b[r]:b[r + 1]], v[b[r]:b[r + 1]]
        if p:
            s = _request_slots(table, r, n + p, case["page"])
            ks, vs = kc.view(-1, hkv, D)[s], vc.view(-1, hkv, D)[s]
        out.append(_attend64(q[b[r]:b[r + 1]], ks, vs, causal_from=p))
    return torch.cat(out)


# ------------------------------------------------------------------ one layer's own passes
SLOTS = 1024  # K/V slots of the small pools that the layer cases store into


def _tables(max_positions: int, theta: float):
    inv = torch.exp(torch.arange(0, D, 2, dtype=torch.float32) * (-(math.log(theta) / D)))
    f = torch.arange(max_positions, dtype=torch.float32)[:, None] * inv[None]
    return f.cos(), f.sin()


def _layer_weights(g, cfg, dt):
    h, f = cfg.hidden_size, cfg.intermediate_size
    shapes = dict(qkv=(cfg.qkv_width, h), o=(h, cfg.num_attention_heads * D), gate_up=(2 * f, h),
                  down=(h, f))
    w = {k: _randn(g, *s, dtype=dt, scale=0.02) for k, s in shapes.items()}
    for k, n in (("q_norm", D), ("k_norm", D), ("norm1", h), ("norm2", h)):
        w[k] = _gamma(g, n, dt)
    return w


def _layer_inputs(case, seed):
    g, dt, cfg = _gen(seed), DTYPES[case["dtype"]], WIDTHS[case["width"]]
    rows, layers = case["rows"], []
    for _ in range(case["layers"]):
        layers.append(dict(
            w=_layer_weights(g, cfg, dt), x=_randn(g, rows, cfg.hidden_size, dtype=dt),
            attn=_randn(g, rows, cfg.num_attention_heads * D, dtype=dt, scale=0.5),
            residual=_randn(g, rows, cfg.hidden_size, dtype=dt),
            pool=[torch.zeros(SLOTS, 1, cfg.num_kv_heads, D, dtype=dt, device="cuda")
                  for _ in range(2)]))
    positions = torch.randint(0, 2048, (rows,), generator=g, device="cuda")
    loc = torch.randperm(SLOTS - 1, generator=g, device="cuda")[:rows] + 1
    return cfg, layers, positions, loc


def _layer_prepare(case, seed):
    cfg, layers, positions, loc = _layer_inputs(case, seed)
    rope = ops.HalfSplitRope(2048, D, cfg.rope_theta, "cuda")
    caches = [_bind(*layer["pool"]) for layer in layers]

    def run():
        out = []
        for layer, cache in zip(layers, caches):
            w, residual = layer["w"], layer["residual"]
            qkv = ops.linear_qk_norm_rope_store(
                layer["x"], w["qkv"], cfg.num_attention_heads, cfg.num_kv_heads, w["q_norm"],
                w["k_norm"], EPS, positions, rope, cache, loc)
            x, residual = ops.linear_add_rms_norm(layer["attn"], w["o"], residual, w["norm1"],
                                                  EPS)
            act = ops.linear_silu_mul(x, w["gate_up"])
            y, residual = ops.linear_add_rms_norm(act, w["down"], residual, w["norm2"], EPS)
            out.append([qkv, x, act, y, residual] + layer["pool"])
        return out

    state = dict(kind=case["kind"], keep=(layers, positions, loc, rope, caches))
    if case["graph"]:
        state["graph"], state["out"] = _captured(run, [layer["residual"] for layer in layers])
    else:
        state["fn"] = run
    return state


def _rms64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _linear64(x, w):
    return torch.cat([x @ part.double().t() for part in w.split(16384)], 1)


def _qk_rope64(qkv, hq, hkv, wq, wk, positions, cos, sin):
    """q and k normalised and rotated, v as it is, laid out as the packed rows."""
    q, k, v = _heads(qkv, hq, hkv)
    c, s = (t.double().to(qkv.device)[positions][:, None] for t in (cos, sin))
    out = []
    for x, w in ((q, wq), (k, wk)):
        x = _rms64(x, w)
        a, b = x[..., :D // 2], x[..., D // 2:]
        out.append(torch.cat([a * c - b * s, b * c + a * s], -1))
    return torch.cat([t.flatten(1) for t in (*out, v)], 1), out[1], v


def _silu_mul64(gate_up):
    g, u = gate_up.chunk(2, 1)
    return torch.nn.functional.silu(g) * u


def _layer_exact(case, seed):
    cfg, layers, positions, loc = _layer_inputs(case, seed)
    hq, hkv = cfg.num_attention_heads, cfg.num_kv_heads
    cos, sin = _tables(2048, cfg.rope_theta)
    out = []
    for layer in layers:
        w = layer["w"]
        qkv, k, v = _qk_rope64(_linear64(layer["x"].double(), w["qkv"]), hq, hkv, w["q_norm"],
                               w["k_norm"], positions, cos, sin)
        pools = []
        for pool, rows in zip(layer["pool"], (k, v)):
            pool = pool.double()
            pool.view(-1, hkv, D)[loc] = rows
            pools.append(pool)
        r = layer["residual"].double() + _linear64(layer["attn"].double(), w["o"])
        x = _rms64(r, w["norm1"])
        act = _silu_mul64(_linear64(x, w["gate_up"]))
        r = r + _linear64(act, w["down"])
        out.append([qkv, x, act, _rms64(r, w["norm2"]), r] + pools)
    return out


# ------------------------------------------------------------------ prefill passes
def _ops_inputs(case, seed):
    g, dt, cfg = _gen(seed), DTYPES[case["dtype"]], WIDTHS[case["width"]]
    t, h = case["tokens"], cfg.hidden_size
    pool = [torch.zeros(t + 1, 1, cfg.num_kv_heads, D, dtype=dt, device="cuda")
            for _ in range(2)]
    return dict(cfg=cfg, x=_randn(g, t, h, dtype=dt), residual=_randn(g, t, h, dtype=dt),
                norm=_gamma(g, h, dt), q_norm=_gamma(g, D, dt), k_norm=_gamma(g, D, dt),
                qkv=_randn(g, t, cfg.qkv_width, dtype=dt),
                gate_up=_randn(g, t, 2 * cfg.intermediate_size, dtype=dt), pool=pool,
                positions=torch.randint(0, 2048, (t,), generator=g, device="cuda"),
                loc=torch.randperm(t, generator=g, device="cuda") + 1)


def _ops_prepare(case, seed):
    state = _ops_inputs(case, seed)
    cfg = state["cfg"]
    return dict(state, kind=case["kind"], rope=ops.HalfSplitRope(2048, D, cfg.rope_theta, "cuda"),
                cache=_bind(*state["pool"]))


def _ops_run(s):
    cfg = s["cfg"]
    x, residual = ops.add_rms_norm(s["x"], s["residual"], s["norm"], EPS)
    q, k, v = _heads(s["qkv"], cfg.num_attention_heads, cfg.num_kv_heads)
    ops.qk_norm_rope_store(q, k, v, s["q_norm"], s["k_norm"], EPS, s["positions"], s["rope"],
                           s["cache"], s["loc"])
    return [x, residual, s["qkv"], *s["pool"], ops.silu_and_mul(s["gate_up"])]


def _ops_exact(case, seed):
    s = _ops_inputs(case, seed)
    cfg = s["cfg"]
    hkv = cfg.num_kv_heads
    r = s["x"].double() + s["residual"].double()
    qkv, k, v = _qk_rope64(s["qkv"].double(), cfg.num_attention_heads, hkv, s["q_norm"],
                           s["k_norm"], s["positions"], *_tables(2048, cfg.rope_theta))
    pools = []
    for pool, rows in zip(s["pool"], (k, v)):
        pool = pool.double()
        pool.view(-1, hkv, D)[s["loc"]] = rows
        pools.append(pool)
    return [_rms64(r, s["norm"]), r, qkv, *pools, _silu_mul64(s["gate_up"].double())]


# ------------------------------------------------------------------ sampling
MIXED = (SamplingParams(0.7, 50, 0.9), SamplingParams(0.0), SamplingParams(1.0, -1, 0.95),
         SamplingParams(0.8, 40, 1.0), SamplingParams(1.0))


def _sample_params(case):
    mix = {"joint": (SamplingParams(0.7, 50, 0.9),), "greedy": (SamplingParams(0.0),),
           "top_p": (SamplingParams(0.8, -1, 0.9),), "mixed": MIXED}[case["mix"]]
    return [mix[i % len(mix)] for i in range(case["rows"])]


def _sample_prepare(case, seed):
    g = _gen(seed)
    logits = _randn(g, case["rows"], case["vocab"], dtype=DTYPES[case["dtype"]], scale=2.5)
    # a few likely tokens per row, as a trained head has
    top = torch.randint(0, case["vocab"], (case["rows"], 16), generator=g, device="cuda")
    logits.scatter_(1, top, _randn(g, case["rows"], 16, dtype=logits.dtype, scale=2.0) + 13.0)
    return dict(kind=case["kind"], logits=logits, params=_sample_params(case),
                sampler=Sampler(seed))


# ------------------------------------------------------------------ whole model
def _model_cfg(case):
    return dataclasses.replace(WIDTHS[case["width"]], num_layers=case["layers"],
                               max_position_embeddings=4096)


def _model_inputs(case, seed):
    """Weights by parameter name, the paged cache, and the step's ids. Decode: one new token per
    request at position length - 1. Prefill: whole prompts, no cached prefix."""
    g, dt, cfg = _gen(seed), torch.bfloat16, _model_cfg(case)
    weights = {"embed": _randn(g, cfg.vocab_size, cfg.hidden_size, dtype=dt, scale=0.02),
               "norm": _gamma(g, cfg.hidden_size, dt)}
    weights["head"] = (weights["embed"] if cfg.tie_word_embeddings else
                       _randn(g, cfg.vocab_size, cfg.hidden_size, dtype=dt, scale=0.02))
    layers = [_layer_weights(g, cfg, dt) for _ in range(cfg.num_layers)]
    lengths = _uniform_lengths(case["lengths"], case["rows"], case["lo"], case["hi"])
    table, pools = _paged(g, lengths, 16, cfg.num_kv_heads, dt, cfg.num_layers)
    if case["phase"] == "decode":
        positions = torch.tensor(lengths, dtype=torch.int64, device="cuda") - 1
        loc = _last_slots(table, lengths, 16)
    else:
        positions = torch.cat([torch.arange(n, device="cuda") for n in lengths])
        loc = torch.cat([_request_slots(table, b, n, 16) for b, n in enumerate(lengths)])
    ids = torch.randint(0, cfg.vocab_size, positions.shape, generator=g, device="cuda")
    return cfg, weights, layers, lengths, table, pools, positions, loc, ids


def _model_prepare(case, seed):
    cfg, weights, layers, lengths, table, pools, positions, loc, ids = _model_inputs(case, seed)
    model = Qwen3Model(cfg, torch.bfloat16, "cuda")
    model.embed_tokens, model.norm, model.lm_head = (weights["embed"], weights["norm"],
                                                     weights["head"])
    for i, (layer, w) in enumerate(zip(model.layers, layers)):
        layer.qkv_proj, layer.o_proj, layer.gate_up_proj, layer.down_proj = (
            w["qkv"], w["o"], w["gate_up"], w["down"])
        layer.q_norm, layer.k_norm = w["q_norm"], w["k_norm"]
        layer.input_layernorm, layer.post_attention_layernorm = w["norm2"], w["norm1"]
    pages = pools[0][0].size(0) - 1
    pool = KVCachePool(KVCacheLayout(cfg.num_layers, pages, 16, cfg.num_kv_heads, D),
                       torch.bfloat16, "cuda")
    for i, (kc, vc) in enumerate(pools):
        pool.buffer[0, i].copy_(kc)
        pool.buffer[1, i].copy_(vc)
    model.bind_kv_cache(pool, reserved_slot=0)
    state = dict(kind=case["kind"], model=model, pool=pool, ids=ids, positions=positions, loc=loc)
    if case["phase"] == "decode":
        lens = torch.tensor(lengths, dtype=torch.int32, device="cuda")
        host = DecodeHostMetadata(lengths)
        meta = AttentionMetadata(BatchPhase.DECODE, decode_host=host, write_loc=loc,
                                 block_table=table, cache_seqlens=lens)
        state["plan"] = model.attention.prepare_decode_graph(meta)
        state["host"], state["meta"] = host, meta
        batch = model.attention.prepare(meta, len(lengths))
        logits = torch.empty(len(lengths), cfg.vocab_size, dtype=torch.bfloat16, device="cuda")
        state["graph"], state["out"] = _captured(
            lambda: model.forward(ids, positions, batch, loc, logits_out=logits))
    else:
        state["meta"] = _prefill_meta(lengths, [0] * len(lengths), table, loc)
        state["last"] = torch.tensor(_bounds(lengths)[1:], device="cuda") - 1
    return state


def _model_run(s):
    if "graph" in s:  # the engine's decode step: re-plan at the host lengths, then the replay
        s["plan"].prepare_replay(s["host"])
        s["graph"].replay()
        return s["out"]
    batch = s["model"].attention.prepare(s["meta"], s["ids"].size(0))
    return s["model"].forward(s["ids"], s["positions"], batch, s["loc"], s["last"])


def _model_exact(case, seed):
    cfg, weights, layers, lengths, table, pools, positions, loc, ids = _model_inputs(case, seed)
    hq, hkv = cfg.num_attention_heads, cfg.num_kv_heads
    cos, sin = _tables(4096, cfg.rope_theta)
    decode = case["phase"] == "decode"
    b = _bounds([1] * len(lengths) if decode else lengths)
    r = weights["embed"][ids].double()
    x = _rms64(r, layers[0]["norm2"])
    for i, (w, (kc, vc)) in enumerate(zip(layers, pools)):
        qkv, k, v = _qk_rope64(_linear64(x, w["qkv"]), hq, hkv, w["q_norm"], w["k_norm"],
                               positions, cos, sin)
        q = qkv[:, :hq * D].view(-1, hq, D)
        kc, vc = kc.view(-1, hkv, D).double(), vc.view(-1, hkv, D).double()
        kc[loc], vc[loc] = k, v
        rows = []
        for n, length in enumerate(lengths):
            s = _request_slots(table, n, length, 16)
            rows.append(_attend64(q[b[n]:b[n + 1]], kc[s], vc[s],
                                  causal_from=length - 1 if decode else 0))
        r = r + _linear64(torch.cat(rows), w["o"])
        act = _silu_mul64(_linear64(_rms64(r, w["norm1"]), w["gate_up"]))
        r = r + _linear64(act, w["down"])
        x = _rms64(r, layers[i + 1]["norm2"] if i + 1 < len(layers) else weights["norm"])
    if not decode:
        x = x[torch.tensor(b[1:], device="cuda") - 1]
    return _linear64(x, weights["head"])


# ------------------------------------------------------------------ the interface
def prepare(case, seed):
    return {"decode_attention": _decode_prepare, "prefill_attention": _prefill_prepare,
            "decode_layer": _layer_prepare, "prefill_ops": _ops_prepare,
            "sample": _sample_prepare, "model": _model_prepare}[case["kind"]](case, seed)


def run(state):
    kind = state["kind"]
    if kind == "prefill_attention":
        return state["batch"].forward(*state["heads"], state["cache"])
    if kind == "prefill_ops":
        return _ops_run(state)
    if kind == "sample":
        return state["sampler"].sample_batch_device(state["logits"], state["params"])
    if kind == "model":
        return _model_run(state)
    if "graph" in state:
        state["graph"].replay()
        out = state["out"]
    else:
        out = state["fn"]()
    if kind == "decode_attention":
        return {"out": out, "caches": state["pools"]}
    return out


def exact(case, seed):
    if case["kind"] == "sample":
        return None  # token ids
    return {"decode_attention": _decode_exact, "prefill_attention": _prefill_exact,
            "decode_layer": _layer_exact, "prefill_ops": _ops_exact,
            "model": _model_exact}[case["kind"]](case, seed)


def _layer_work(cfg, rows):
    h, f = cfg.hidden_size, cfg.intermediate_size
    hq, hkv = cfg.num_attention_heads, cfg.num_kv_heads
    weights = cfg.qkv_width * h + h * hq * D + 3 * h * f
    moved = rows * (h + cfg.qkv_width + 2 * hkv * D + hq * D + 3 * h)
    return 2 * (weights + moved), 2 * rows * weights


def work(case):
    kind = case["kind"]
    if kind == "decode_attention":
        n = sum(_uniform_lengths(case["lengths"], case["rows"], case["lo"], case["hi"]))
        hq, hkv, rows = case["q_heads"], case["kv_heads"], case["rows"]
        one = (2 * n * hkv * D * 2 + 4 * -(-n // case["page"]) + rows * 2 * hq * D * 2
               + rows * (2 * hkv * D * 2 * 2 + 8))
        return {"bytes": one * case["layers"], "flops": 4 * n * hq * D * case["layers"]}
    if kind == "prefill_attention":
        new, pre = _prefill_lengths(case)
        hq, hkv = case["q_heads"], case["kv_heads"]
        tokens, keys = sum(new), sum(new) + sum(pre)
        return {"bytes": 2 * D * (2 * tokens * hq + 2 * keys * hkv),
                "flops": 4 * hq * D * sum(n * p + n * (n + 1) // 2 for n, p in zip(new, pre))}
    if kind == "decode_layer":
        b, f = _layer_work(WIDTHS[case["width"]], case["rows"])
        return {"bytes": b * case["layers"], "flops": f * case["layers"]}
    if kind == "prefill_ops":
        cfg, t = WIDTHS[case["width"]], case["tokens"]
        heads = cfg.num_attention_heads + cfg.num_kv_heads
        per = (4 * cfg.hidden_size + 2 * heads * D + 3 * cfg.num_kv_heads * D
               + 3 * cfg.intermediate_size)
        return {"bytes": 2 * t * per, "flops": 10 * t * per}
    if kind == "sample":
        size = 4 if case["dtype"] == "fp32" else 2
        return {"bytes": case["rows"] * (case["vocab"] * size + 20),
                "flops": 4 * case["rows"] * case["vocab"]}
    cfg = _model_cfg(case)
    lengths = _uniform_lengths(case["lengths"], case["rows"], case["lo"], case["hi"])
    decode = case["phase"] == "decode"
    tokens = len(lengths) if decode else sum(lengths)
    b, f = _layer_work(cfg, tokens)
    hq, hkv, h = cfg.num_attention_heads, cfg.num_kv_heads, cfg.hidden_size
    seen = sum(lengths) if decode else sum(n * (n + 1) // 2 for n in lengths)
    b += 2 * sum(lengths) * hkv * D * 2 if decode else 0
    f += 4 * seen * hq * D
    head = cfg.vocab_size * h
    return {"bytes": cfg.num_layers * b + 2 * (head + len(lengths) * cfg.vocab_size),
            "flops": cfg.num_layers * f + 2 * len(lengths) * head}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        # a draw may turn where a cutoff falls between two tokens of almost equal probability
        return {"rel": 0.0, "differ": 0.01}
    # Relative errors against 64 bits as measured: attention 2.1e-3 in bf16, a layer's last
    # outputs 4.5e-3 in bf16 and 5e-4 in fp16, the prefill passes 2.3e-3, four layers and the
    # head 1.4e-2. About four times that (the model: what two such results can differ by).
    fp16 = case.get("dtype") == "fp16"
    if kind == "model":
        return {"rel": 0.025, "max": 0.35}
    if fp16:
        return {"rel": 2e-3, "max": 0.02}
    return {"rel": 1.8e-2, "max": 0.15} if kind == "decode_layer" else {"rel": 9e-3, "max": 0.1}
