"""The work whose speed matters to a user of this framework, as cases that can be timed and checked.

Five kinds of case, each through the entry points that a serving program calls, on the model shapes of
nanoserve_amd.model (random weights, scattered cache blocks):

  decode_attn  attention of one-token rows over their cache pages (paged_attention_decode), either called once
               or, as in a decode step, for several layers replayed from a graph
  chunk_attn   attention of prefill chunks (paged_attention_prefill), with decode rows beside them where
               dec_rows > 0 (paged_attention_mixed); steps that the engine would replay from a graph (several
               layers) are replayed here too
  layer        everything between the attention of one layer and that of the next: O projection, residual,
               RMSNorm, SwiGLU MLP, residual, RMSNorm, QKV projection, RoPE and the K/V write. Decode-sized
               steps are replayed from a graph (several layers, each on inputs of its own), larger ones run
               eagerly, as the engine's executor does both
  step         one decode step of a whole model through DecodeGraphRunner: staging, replay, greedy tokens
  prompts      one eager forward of a whole model over fresh prompts (Qwen2Model.forward_batch)

Lengths are drawn between a case's bounds by a generator that is seeded with the bounds, so they belong to the case;
values come from the seed.
"""
import dataclasses
import math
import random

import torch

from nanoserve_amd.hip_graphs import DecodeGraphRunner, capture
from nanoserve_amd.kernels.linear import linear_residual_rms_norm, linear_rope_qkv, linear_silu_mul
from nanoserve_amd.kernels.paged_attention import (pair_rows, paged_attention_decode, paged_attention_mixed,
                                                   paged_attention_prefill, prefill_seq_info)
from nanoserve_amd.kv_cache import PagedKVCache
from nanoserve_amd.model import QWEN25_0_5B, QWEN25_1_5B, QWEN25_3B, Qwen2Model, SeqInput

MODELS = {"0.5b": QWEN25_0_5B, "1.5b": QWEN25_1_5B, "3b": QWEN25_3B}
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
PAGE = 16
GRAPH_ROWS = 512    # steps of up to this many rows replay a graph in the engine
SMALL_VOCAB = 2048  # of the layer cases' models: they don't reach the LM head


def listed():
    return [
        # one user's decode: a single short row, called directly; launch and latency are all there is
        {"name": "decode_attn_one_row", "kind": "decode_attn", "model": "1.5b", "dtype": "bf16", "seqs": 1, "share": 1,
         "ctx_lo": 300, "ctx_hi": 300, "layers": 1, "graph": False},
        # a full decode batch of mixed contexts, eight layers of it in one replay
        {"name": "decode_attn_32_rows", "kind": "decode_attn", "model": "0.5b", "dtype": "bf16", "seqs": 32, "share": 1,
         "ctx_lo": 512, "ctx_hi": 4096, "layers": 8, "graph": True},
        # long documents: few rows, contexts up to the models' 32k positions
        {"name": "decode_attn_long", "kind": "decode_attn", "model": "3b", "dtype": "bf16", "seqs": 12, "share": 1,
         "ctx_lo": 9000, "ctx_hi": 32000, "layers": 4, "graph": True},
        # the fp32 correctness configuration: four 128-token prompts, whose tokens run as decode rows
        {"name": "decode_attn_fp32_prompts", "kind": "decode_attn", "model": "0.5b", "dtype": "fp32", "seqs": 4,
         "share": 128, "ctx_lo": 1, "ctx_hi": 1, "layers": 1, "graph": False},
        # a mixed step's attention: a 1536-token chunk on 512 cached tokens beside 16 decode rows
        {"name": "mixed_attn_chunk", "kind": "chunk_attn", "model": "1.5b", "seqs": 1, "new_lo": 1536, "new_hi": 1536,
         "ctx_lo": 512, "ctx_hi": 512, "dec_rows": 16, "dec_lo": 256, "dec_hi": 2048, "layers": 1},
        # several long prompts at once, ragged, some of them continued
        {"name": "prefill_attn_ragged_long", "kind": "chunk_attn", "model": "3b", "seqs": 3, "new_lo": 900,
         "new_hi": 4400, "ctx_lo": 0, "ctx_hi": 6000, "dec_rows": 0, "dec_lo": 1, "dec_hi": 1, "layers": 1},
        # one user's decode through the layers
        {"name": "layer_1_row", "kind": "layer", "model": "0.5b", "rows": 1, "layers": 4},
        # the full decode batch
        {"name": "layer_32_rows", "kind": "layer", "model": "1.5b", "rows": 32, "layers": 4},
        # speculative verification: 24 sequences of 5 rows
        {"name": "layer_120_rows", "kind": "layer", "model": "1.5b", "rows": 120, "layers": 4},
        # the mixed step: a 1536-token chunk, 16 decode rows and a padding row
        {"name": "layer_1553_rows", "kind": "layer", "model": "1.5b", "rows": 1553, "layers": 1},
        # the headline: a whole decode step at batch 32
        {"name": "step_32_rows", "kind": "step", "model": "1.5b", "rows": 32, "ctx_lo": 1024, "ctx_hi": 1151},
        # time to the first token: five ragged prompts in one eager forward
        {"name": "prompts_ragged", "kind": "prompts", "model": "0.5b", "seqs": 5, "new_lo": 60, "new_hi": 900},
    ]


def _log(rng, lo, hi):
    """An integer between lo and hi, spread over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    model = rng.choice(sorted(MODELS))
    kind = rng.choices(["decode_attn", "chunk_attn", "layer", "step", "prompts"], [0.3, 0.25, 0.35, 0.05, 0.05])[0]
    if kind == "decode_attn":
        if rng.random() < 0.15:     # fp32: prompts of the correctness configuration, or plain rows
            share = rng.choice([1, _log(rng, 8, 160)])
            lo = 1 if share > 1 else _log(rng, 16, 1024)
            return {"kind": kind, "model": model, "dtype": "fp32", "seqs": rng.randint(1, 4) if share > 1 else rng.randint(1, 16),
                    "share": share, "ctx_lo": lo, "ctx_hi": lo if share > 1 else 2 * lo, "layers": 1, "graph": False}
        hi = _log(rng, 32, 32000)
        lo = max(1, int(hi * rng.uniform(0.1, 1.0)))
        share = rng.choice([1, 1, 1, 3, 5])
        seqs = min(_log(rng, 1, 128 // share), max(1, 300000 // hi))
        return {"kind": kind, "model": model, "dtype": "bf16", "seqs": seqs, "share": share, "ctx_lo": lo, "ctx_hi": hi,
                "layers": 4, "graph": True}
    if kind == "chunk_attn":
        seqs = rng.choice([1, 1, 2, 3, 5, 8])
        hi = _log(rng, 16, 6000 // seqs)
        ctx, dec = rng.choice([0, _log(rng, 16, 12000)]), rng.choice([0, 0, rng.randint(1, 48)])
        return {"kind": kind, "model": model, "seqs": seqs, "new_lo": max(1, int(hi * rng.uniform(0.2, 1.0))), "new_hi": hi,
                "ctx_lo": ctx // 3, "ctx_hi": ctx, "dec_rows": dec, "dec_lo": 32, "dec_hi": _log(rng, 64, 4096),
                "layers": 4 if seqs * hi + dec <= GRAPH_ROWS else 1}
    if kind == "layer":
        rows = rng.choice([_log(rng, 1, 64), _log(rng, 65, 512), _log(rng, 513, 6000)])
        return {"kind": kind, "model": model, "rows": rows, "layers": 4 if rows <= GRAPH_ROWS else 1}
    if kind == "step":
        hi = _log(rng, 64, 2000)
        return {"kind": kind, "model": rng.choice(["0.5b", "1.5b"]), "rows": _log(rng, 1, 32),
                "ctx_lo": max(1, int(hi * rng.uniform(0.2, 1.0))), "ctx_hi": hi}
    hi = _log(rng, 30, 900)
    return {"kind": kind, "model": "0.5b", "seqs": rng.randint(1, 5), "new_lo": max(1, int(hi * rng.uniform(0.1, 1.0))),
            "new_hi": hi}


# ------------------------------------------------------------------------------------------------ inputs
def _lengths(n, lo, hi, tag):
    r = random.Random(f"{tag} {n} {lo} {hi}")
    return [r.randint(lo, hi) for _ in range(n)]


def _pages(tokens):
    return -(-tokens // PAGE)


def _tables(lengths, first, tag):
    """Scattered block lists for sequences of these lengths (ids from `first` on), and the next free id."""
    need = [_pages(n) for n in lengths]
    ids = list(range(first, first + sum(need)))
    random.Random(f"{tag} {len(ids)}").shuffle(ids)
    out = []
    for n in need:
        out.append(ids[:n])
        ids = ids[n:]
    return out, first + sum(need)


def _padded(tables, rows_each=1):
    """int32 [rows, width] on the GPU, zeros past each table's end, every table rows_each times."""
    width = max(len(t) for t in tables)
    flat = torch.tensor([t + [0] * (width - len(t)) for t in tables], dtype=torch.int32)
    return flat.repeat_interleave(rows_each, 0).cuda()


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, std=1.0, dtype=torch.bfloat16):
    return torch.empty(*shape, device="cuda", dtype=torch.float32).normal_(0.0, std, generator=g).to(dtype)


def _weights(cfg, g):
    """Weights of cfg's shape under their checkpoint names: matrices N(0, 0.02), norm weights around 1. As in a trained
    model, the residual stream is large beside what one layer adds to it (embeddings N(0, 1), the two matrices that
    write to it scaled by their number): its roundings then pass through the layers without growing."""
    H, inter = cfg.hidden_size, cfg.intermediate_size
    out_std = 0.02 / math.sqrt(2 * cfg.n_layers)
    nq, nk = cfg.n_heads * cfg.head_dim, cfg.n_kv_heads * cfg.head_dim
    sd = {"model.embed_tokens.weight": _normal(g, cfg.vocab_size, H)}
    for i in range(cfg.n_layers):
        p = f"model.layers.{i}."
        for name, n in (("input_layernorm", H), ("post_attention_layernorm", H)):
            sd[p + name + ".weight"] = (1.0 + _normal(g, n, std=0.1, dtype=torch.float32)).bfloat16()
        for name, n in (("q", nq), ("k", nk), ("v", nk)):
            sd[p + f"self_attn.{name}_proj.weight"] = _normal(g, n, H, std=0.02)
            sd[p + f"self_attn.{name}_proj.bias"] = _normal(g, n, std=0.02)
        sd[p + "self_attn.o_proj.weight"] = _normal(g, H, nq, std=out_std)
        sd[p + "mlp.gate_proj.weight"] = _normal(g, inter, H, std=0.02)
        sd[p + "mlp.up_proj.weight"] = _normal(g, inter, H, std=0.02)
        sd[p + "mlp.down_proj.weight"] = _normal(g, H, inter, std=out_std)
    sd["model.norm.weight"] = (1.0 + _normal(g, H, std=0.1, dtype=torch.float32)).bfloat16()
    return sd


def _decode_lengths(case):
    """(tokens cached per sequence, context length of every row)."""
    first = _lengths(case["seqs"], case["ctx_lo"], case["ctx_hi"], "decode")
    return [c + case["share"] - 1 for c in first], [c + j for c in first for j in range(case["share"])]


def _decode_inputs(case, seed):
    cfg, dt, g = MODELS[case["model"]], DTYPES[case["dtype"]], _gen(seed)
    kept, lens = _decode_lengths(case)
    tables, n_blocks = _tables(kept, 1, "decode")
    layers = []
    for _ in range(case["layers"]):
        pool = (n_blocks, PAGE, cfg.n_kv_heads, cfg.head_dim)
        layers.append((_normal(g, len(lens), cfg.n_heads, cfg.head_dim, std=1.5, dtype=dt),
                       _normal(g, *pool, dtype=dt), _normal(g, *pool, dtype=dt)))
    return cfg, layers, tables, lens


def _chunk_lengths(case):
    new = _lengths(case["seqs"], case["new_lo"], case["new_hi"], "new")
    ctx = _lengths(case["seqs"], case["ctx_lo"], case["ctx_hi"], "ctx")
    dec = _lengths(case["dec_rows"], min(case["dec_lo"], case["dec_hi"]), case["dec_hi"], "dec")
    return new, ctx, dec


def _chunk_inputs(case, seed):
    """The step's rows: the decode rows first, as the scheduler places them, then the chunks."""
    cfg, g = MODELS[case["model"]], _gen(seed)
    new, ctx, dec = _chunk_lengths(case)
    dec_tables, n = _tables(dec, 1, "dec")
    tables, n = _tables([a + b for a, b in zip(new, ctx)], n, "chunk")
    pool = (n, PAGE, cfg.n_kv_heads, cfg.head_dim)
    layers = [(_normal(g, len(dec) + sum(new), cfg.n_heads, cfg.head_dim, std=1.5), _normal(g, *pool), _normal(g, *pool))
              for _ in range(case["layers"])]
    return cfg, layers, new, ctx, dec, tables, dec_tables


def _layer_inputs(case, seed):
    cfg = dataclasses.replace(MODELS[case["model"]], n_layers=case["layers"], vocab_size=SMALL_VOCAB)
    g, rows = _gen(seed), case["rows"]
    sd = _weights(cfg, g)
    acts = [(_normal(g, rows, cfg.n_heads * cfg.head_dim, std=0.5), _normal(g, rows, cfg.hidden_size))
            for _ in range(cfg.n_layers)]
    pos = torch.randint(0, 2048, (rows,), device="cuda", generator=g)
    inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, cfg.head_dim, 2, dtype=torch.float, device="cuda") / cfg.head_dim))
    f = torch.cat([pos[:, None].float() * inv] * 2, dim=-1)
    slots = torch.randperm(_pages(rows) * PAGE, device="cuda", generator=g)[:rows]
    return cfg, sd, acts, f.cos().bfloat16(), f.sin().bfloat16(), slots


def _step_inputs(case, seed):
    cfg, g = MODELS[case["model"]], _gen(seed)
    ctx = _lengths(case["rows"], case["ctx_lo"], case["ctx_hi"], "step")     # tokens cached before the step
    tables, n_blocks = _tables([c + 1 for c in ctx], 1, "step")              # block 0 is the runner's own
    sd = _weights(cfg, g)
    pool = (cfg.n_layers, n_blocks, PAGE, cfg.n_kv_heads, cfg.head_dim)
    k, v = _normal(g, *pool), _normal(g, *pool)
    tokens = torch.randint(0, cfg.vocab_size, (case["rows"],), device="cuda", generator=g).tolist()
    return cfg, sd, k, v, tokens, ctx, tables


def _prompt_inputs(case, seed):
    cfg, g = MODELS[case["model"]], _gen(seed)
    new = _lengths(case["seqs"], case["new_lo"], case["new_hi"], "prompts")
    tables, n_blocks = _tables(new, 0, "prompts")
    sd = _weights(cfg, g)
    tokens = torch.randint(0, cfg.vocab_size, (sum(new),), device="cuda", generator=g)
    return cfg, sd, tokens, new, tables, n_blocks


# ------------------------------------------------------------------------------------------------ the calls
def _replayed(fn):
    """fn recorded into a graph, as the runners record their steps. The result holds fn, and with it every tensor
    that fn reads: the graph itself keeps addresses only."""
    graph, out = capture(fn, torch.cuda.graph_pool_handle())

    def replay(inputs_of=fn):
        graph.replay()
        return out
    return replay


def _prepare_decode_attn(case, seed):
    cfg, layers, tables, lens = _decode_inputs(case, seed)
    share = case["share"]
    bt, cl, scale = _padded(tables, share), torch.tensor(lens, dtype=torch.int32).cuda(), cfg.head_dim ** -0.5
    pairs = None
    if 1 < share <= 8 and case["dtype"] == "bf16":     # rows that share a table run in pairs (speculative lane)
        host = torch.zeros(len(lens), dtype=torch.int32)
        pair_rows([t for t in tables for _ in range(share)], host)
        pairs = host.cuda()

    def call():
        return [paged_attention_decode(q, k, v, bt, cl, scale, pairs=pairs) for q, k, v in layers]
    return _replayed(call) if case["graph"] else call


def _prepare_chunk_attn(case, seed):
    cfg, layers, new, ctx, dec, tables, dec_tables = _chunk_inputs(case, seed)
    starts = [len(dec) + sum(new[:i]) for i in range(len(new))]
    info, bt, scale = prefill_seq_info(starts, new, ctx, "cuda"), _padded(tables), cfg.head_dim ** -0.5
    max_new, max_kv = max(new), max(a + b for a, b in zip(new, ctx))
    if dec:
        dec_bt, dec_cl = _padded(dec_tables), torch.tensor(dec, dtype=torch.int32).cuda()
        rows = torch.arange(len(dec), device="cuda")

    def call():
        if not dec:
            return [paged_attention_prefill(q, k, v, bt, info, max_new, max_kv, scale) for q, k, v in layers]
        return [paged_attention_mixed(q, k, v, bt, info, max_new, max_kv, dec_bt, dec_cl, rows, scale,
                                      out=torch.empty_like(q)) for q, k, v in layers]
    return _replayed(call) if sum(new) + len(dec) <= GRAPH_ROWS else call


def _prepare_layer(case, seed):
    cfg, sd, acts, cos, sin, slots = _layer_inputs(case, seed)
    model, eps = Qwen2Model(cfg, sd), cfg.rms_norm_eps
    caches = [[torch.zeros(_pages(case["rows"]), PAGE, cfg.n_kv_heads, cfg.head_dim, device="cuda", dtype=torch.bfloat16)
               for _ in range(2)] for _ in acts]

    def call():
        out = []
        for w, (o, x), (kc, vc) in zip(model.layers, acts, caches):
            h, x = linear_residual_rms_norm(o, w.o_p or w.o_w, x, w.ln2, eps)
            a = linear_silu_mul(h, w.gate_up_p or w.gate_up_w)
            h, x = linear_residual_rms_norm(a, w.down_p or w.down_w, x, w.ln1, eps)
            q, k, v = linear_rope_qkv(h, w.qkv_p or w.qkv_w, w.qkv_b, cos, sin, cfg.n_heads, cfg.n_kv_heads,
                                      cfg.head_dim, kc, vc, slots)
            out.append((x, q, k, v, kc, vc))
        return out
    return _replayed(call) if case["rows"] <= GRAPH_ROWS else call


def _prepare_step(case, seed):
    cfg, sd, k, v, tokens, ctx, tables = _step_inputs(case, seed)
    model = Qwen2Model(cfg, sd)
    pool = PagedKVCache(cfg, k.shape[1])
    pool.k.copy_(k)
    pool.v.copy_(v)
    del k, v
    runner = DecodeGraphRunner(model, pool, max_seq_len=max(ctx) + 64)
    slots = [t[c // PAGE] * PAGE + c % PAGE for t, c in zip(tables, ctx)]
    lens, n = [c + 1 for c in ctx], len(ctx)

    def call():
        logits = runner.run(tokens, ctx, slots, tables, lens)
        runner.greedy_tokens(n)
        return logits
    call()      # records the bucket's graph, as the engine does at start-up
    return call


def _prepare_prompts(case, seed):
    cfg, sd, tokens, new, tables, n_blocks = _prompt_inputs(case, seed)
    model, pool = Qwen2Model(cfg, sd), PagedKVCache(cfg, n_blocks)
    pos = torch.tensor([j for n in new for j in range(n)]).cuda()
    slots = torch.tensor([t[j // PAGE] * PAGE + j % PAGE for t, n in zip(tables, new) for j in range(n)]).cuda()

    def call():
        seqs = [SeqInput(n, block_table=t) for n, t in zip(new, tables)]
        return model.forward_batch(tokens, pos, seqs, logits="last", paged=pool, slot_mapping=slots)
    return call


def prepare(case, seed):
    return {"decode_attn": _prepare_decode_attn, "chunk_attn": _prepare_chunk_attn, "layer": _prepare_layer,
            "step": _prepare_step, "prompts": _prepare_prompts}[case["kind"]](case, seed)


def run(state):
    return state()


# ------------------------------------------------------------------------------------------------ work, tolerance
def _layer_params(cfg):
    H, nq, nk = cfg.hidden_size, cfg.n_heads * cfg.head_dim, cfg.n_kv_heads * cfg.head_dim
    return (nq + 2 * nk) * H + H * nq + 3 * H * cfg.intermediate_size


def work(case):
    cfg = MODELS[case["model"]]
    nq, nk, H = cfg.n_heads * cfg.head_dim, cfg.n_kv_heads * cfg.head_dim, cfg.hidden_size
    if case["kind"] == "decode_attn":
        size = torch.finfo(DTYPES[case["dtype"]]).bits // 8
        kept, lens = _decode_lengths(case)
        nbytes = sum(kept) * 2 * nk * size + 2 * len(lens) * nq * size + 4 * sum(map(_pages, kept)) + 4 * len(lens)
        return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * 4 * nq * sum(lens)}
    if case["kind"] == "chunk_attn":
        new, ctx, dec = _chunk_lengths(case)
        rows, keys = sum(new) + len(dec), sum(new) + sum(ctx) + sum(dec)
        seen = sum(n * c + n * (n + 1) // 2 for n, c in zip(new, ctx)) + sum(dec)
        return {"bytes": case["layers"] * (keys * 2 * nk * 2 + 2 * rows * nq * 2), "flops": case["layers"] * 4 * nq * seen}
    if case["kind"] == "layer":
        rows, params = case["rows"], _layer_params(cfg)
        acts = rows * (nq + 2 * H) + rows * (nq + 4 * nk) + 2 * rows * cfg.head_dim
        return {"bytes": case["layers"] * 2 * (params + acts), "flops": case["layers"] * 2 * rows * params}
    weights = cfg.n_layers * _layer_params(cfg)
    if case["kind"] == "step":
        ctx, head = _lengths(case["rows"], case["ctx_lo"], case["ctx_hi"], "step"), cfg.vocab_size * H
        return {"bytes": 2 * (weights + head + case["rows"] * cfg.vocab_size) + sum(c + 1 for c in ctx) * cfg.n_layers * 4 * nk,
                "flops": 2 * case["rows"] * (weights + head) + 4 * nq * cfg.n_layers * sum(c + 1 for c in ctx)}
    new, head = _lengths(case["seqs"], case["new_lo"], case["new_hi"], "prompts"), cfg.vocab_size * H
    return {"bytes": 2 * (weights + head) + sum(new) * cfg.n_layers * 4 * nk + 2 * len(new) * cfg.vocab_size,
            "flops": 2 * sum(new) * weights + 2 * len(new) * head + 4 * nq * cfg.n_layers * sum(n * (n + 1) // 2 for n in new)}


def tolerance(case):
    """About four times what the paths are off their 64-bit values (fp32 sums more: 2e-7 was seen), and for whole
    models, whose layers each add the rounding of the residual stream, about twice (1.3e-2 was seen)."""
    if case["kind"] in ("decode_attn", "chunk_attn"):
        return {"rel": 5e-6} if case.get("dtype") == "fp32" else {"rel": 1e-2}
    return {"rel": 1.5e-2} if case["kind"] == "layer" else {"rel": 3e-2}


# ------------------------------------------------------------------------------------------------ 64 bits
def _attend64(q, k, v, pos):
    """q [T, n_heads, hd] at positions pos [T] over k, v [L, n_kv, hd], all 64-bit: query t sees keys 0 .. pos[t]."""
    T, nh, hd = q.shape
    L, nkv = k.shape[0], k.shape[1]
    hidden = torch.arange(L, device=q.device)[None, None, :] > pos[:, None, None]
    out = torch.empty_like(q)
    for g in range(nkv):
        heads = slice(g * nh // nkv, (g + 1) * nh // nkv)
        s = (q[:, heads].reshape(-1, hd) @ k[:, g].t()).view(T, -1, L) * hd ** -0.5
        p = torch.softmax(s.masked_fill(hidden, -math.inf), dim=-1)
        out[:, heads] = (p.view(-1, L) @ v[:, g]).view(T, -1, hd)
    return out


def _gathered(pool, table, n):
    """The first n tokens' rows of a block list, 64-bit [n, n_kv, hd]."""
    return pool[torch.tensor(table, device=pool.device)].flatten(0, 1)[:n].double()


def _rms64(x, w, eps):
    return w.double() * x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _rope64(x, cos, sin):
    half = x.shape[-1] // 2
    turned = torch.cat([-x[..., half:], x[..., :half]], dim=-1)
    return x * cos[:, None] + turned * sin[:, None]


def _qkv64(cfg, sd, i, h, cos, sin):
    q, k, v = (h @ sd[f"model.layers.{i}.self_attn.{n}_proj.weight"].double().t()
               + sd[f"model.layers.{i}.self_attn.{n}_proj.bias"].double() for n in "qkv")
    q, k, v = (t.view(h.shape[0], -1, cfg.head_dim) for t in (q, k, v))
    return _rope64(q, cos, sin), _rope64(k, cos, sin), v


def _mlp64(cfg, sd, i, o, x):
    """The residual stream after layer i's attention output o [rows, n_heads * hd] and its MLP."""
    p = f"model.layers.{i}."
    x = x + o @ sd[p + "self_attn.o_proj.weight"].double().t()
    h = _rms64(x, sd[p + "post_attention_layernorm.weight"], cfg.rms_norm_eps)
    a = torch.nn.functional.silu(h @ sd[p + "mlp.gate_proj.weight"].double().t())
    a = a * (h @ sd[p + "mlp.up_proj.weight"].double().t())
    return x + a @ sd[p + "mlp.down_proj.weight"].double().t()


def _model64(cfg, sd, tokens, pos, attend):
    """Final-normed hidden states of a whole forward; attend(i, q, k, v) is layer i's attention."""
    inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, cfg.head_dim, 2, dtype=torch.float64, device="cuda") / cfg.head_dim))
    f = torch.cat([pos[:, None].double() * inv] * 2, dim=-1)
    x = sd["model.embed_tokens.weight"][tokens].double()
    for i in range(cfg.n_layers):
        h = _rms64(x, sd[f"model.layers.{i}.input_layernorm.weight"], cfg.rms_norm_eps)
        x = _mlp64(cfg, sd, i, attend(i, *_qkv64(cfg, sd, i, h, f.cos(), f.sin())).flatten(1), x)
    return _rms64(x, sd["model.norm.weight"], cfg.rms_norm_eps)


def _exact_decode_attn(case, seed):
    cfg, layers, tables, lens = _decode_inputs(case, seed)
    share, outs = case["share"], []
    for q, k, v in layers:
        out = torch.empty_like(q, dtype=torch.float64)
        for s, t in enumerate(tables):
            rows = slice(s * share, (s + 1) * share)
            n = lens[rows][-1]
            out[rows] = _attend64(q[rows].double(), _gathered(k, t, n), _gathered(v, t, n),
                                  torch.tensor(lens[rows], device="cuda") - 1)
        outs.append(out)
    return outs


def _exact_chunk_attn(case, seed):
    cfg, layers, new, ctx, dec, tables, dec_tables = _chunk_inputs(case, seed)
    outs = []
    for q, k, v in layers:
        out, start = torch.empty_like(q, dtype=torch.float64), 0
        for n, c, t in list(zip([1] * len(dec), [d - 1 for d in dec], dec_tables)) + list(zip(new, ctx, tables)):
            out[start:start + n] = _attend64(q[start:start + n].double(), _gathered(k, t, n + c), _gathered(v, t, n + c),
                                             torch.arange(c, c + n, device="cuda"))
            start += n
        outs.append(out)
    return outs


def _exact_layer(case, seed):
    cfg, sd, acts, cos, sin, slots = _layer_inputs(case, seed)
    outs = []
    for i, (o, x) in enumerate(acts):
        x = _mlp64(cfg, sd, i, o.double(), x.double())
        h = _rms64(x, sd[f"model.layers.{i}.input_layernorm.weight"], cfg.rms_norm_eps)
        q, k, v = _qkv64(cfg, sd, i, h, cos.double(), sin.double())
        caches = []
        for t in (k, v):
            c = torch.zeros(_pages(case["rows"]) * PAGE, cfg.n_kv_heads, cfg.head_dim, device="cuda", dtype=torch.float64)
            c[slots] = t
            caches.append(c.view(-1, PAGE, cfg.n_kv_heads, cfg.head_dim))
        outs.append((x, q, k, v, *caches))
    return outs


def _exact_step(case, seed):
    cfg, sd, kp, vp, tokens, ctx, tables = _step_inputs(case, seed)

    def attend(i, q, k, v):
        out = torch.empty_like(q)
        for r, (c, t) in enumerate(zip(ctx, tables)):
            kk, vv = (torch.cat([_gathered(pool[i], t, c), new[r:r + 1]]) for pool, new in ((kp, k), (vp, v)))
            out[r:r + 1] = _attend64(q[r:r + 1], kk, vv, torch.tensor([c], device="cuda"))
        return out
    h = _model64(cfg, sd, torch.tensor(tokens, device="cuda"), torch.tensor(ctx, device="cuda"), attend)
    return h @ sd["model.embed_tokens.weight"].double().t()


def _exact_prompts(case, seed):
    cfg, sd, tokens, new, _, _ = _prompt_inputs(case, seed)
    pos = torch.cat([torch.arange(n, device="cuda") for n in new])
    ends = torch.tensor(new).cumsum(0).tolist()

    def attend(i, q, k, v):
        return torch.cat([_attend64(q[e - n:e], k[e - n:e], v[e - n:e], pos[e - n:e]) for n, e in zip(new, ends)])
    h = _model64(cfg, sd, tokens, pos, attend)[[e - 1 for e in ends]]
    return h @ sd["model.embed_tokens.weight"].double().t()


def exact(case, seed):
    return {"decode_attn": _exact_decode_attn, "chunk_attn": _exact_chunk_attn, "layer": _exact_layer,
            "step": _exact_step, "prompts": _exact_prompts}[case["kind"]](case, seed)
