"""The calls of this framework whose time matters, as data: which sizes, which inputs, one
pass of each through the public entry points, the work a pass cannot do without, and the
same results in 64 bits.

A case is a dict of plain values; ``kind`` names the entry point:

  attention   block attention of new queries over the contiguous or paged block KV cache:
              ``AttentionBackend.flash_kvcache_attention`` (contiguous, every cached key
              visible) and ``ops.block_attn`` (page tables, block-causal masks, the cache
              write of the call's own keys and values)
  rows        the sparse layer's edges: ``fused_gather_input_rmsnorm_pair`` of the selected
              token rows, then ``scatter_rows`` of rows of that shape into the layer's cache
              and the current hidden states
  projections ``ops.qkv_rope_kv_write``: q / k / v projections, RoPE and the cache writes
  unmask      ``ops.unmask_step``: greedy tokens, confidences and the threshold rule
  model       ``BlockDiffusionLM`` over the static caches: one sub-block diffusion step

Inputs are drawn on the GPU from the seed; what a program fixes before it has any data
(lengths, page counts, selected-row counts) follows from the case alone.
"""
from __future__ import annotations

import math
import random

import torch

from fast_v2_amd import _ffi, ops
from fast_v2_amd.cuda_bench.fused_sparse_extension import fused_gather_input_rmsnorm_pair, get_fused_ops
from fast_v2_amd.e2e.model import BlockDiffusionConfig, RMSNorm, build_model
from fast_v2_amd.e2e.sampler import HipStaticAttention
from fast_v2_amd.utils.attention_backends import get_attention_backend

BLOCK = 32         # tokens of a diffusion block
HEAD_DIM = 128
PAGE = 32          # tokens of a cache page
VOCAB = 152064
MASK_ID = 152063
HEADS = ((28, 4), (12, 2))  # query / KV heads of the repository's two layouts
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _attention(name=None, **kw):
    case = dict(kind="attention", batch=1, q_len=8, q_heads=28, kv_heads=4, min_keys=544, max_keys=544,
                layout="contiguous", mask="all", write=False, dtype="bf16")
    case.update(kw)
    return _named(case, name)


def _named(case, name):
    if name is not None:
        case["name"] = name
    return case


def listed():
    return [
        # one user, an 8-token sub-block step early in a generation: the smallest call
        _attention("sub_block_1x544"),
        # the sub-block step of a batch of 16 at mixed lengths on pages, the generation's
        # most frequent attention call
        _attention("sub_block_16_paged", batch=16, min_keys=1056, max_keys=4128, layout="paged_hm"),
        # long contexts and a large batch in fp16, lengths that end inside a block
        _attention("sub_block_48_long", batch=48, min_keys=2000, max_keys=12011, layout="paged", dtype="fp16"),
        # a whole 32-token block over the static cache: a block's first step and its commit
        _attention("block_16", batch=16, q_len=BLOCK, min_keys=1056, max_keys=4128),
        # two short prompts of odd length, every prompt key visible (the prompt forward)
        _attention("prompt_2x157", batch=2, q_len=157, min_keys=157, max_keys=157),
        # one prompt of ordinary length, block-causal, its keys written by the call
        _attention("prompt_1x1500", q_len=1500, min_keys=1500, max_keys=1500, mask="block", write=True,
                   layout="paged"),
        # a batch of long prompts, the largest call
        _attention("prompt_4x4096", batch=4, q_len=4096, min_keys=4096, max_keys=4096, mask="block", write=True),
        # callers in fp32 (the reference's CPU-runnable layout): one block over 544 keys
        _attention("block_fp32_1x544", q_len=BLOCK, q_heads=12, kv_heads=2, dtype="fp32"),
        # a sparse layer that recomputes a quarter of 4096 tokens
        _named(dict(kind="rows", batch=1, seq=4096, rows=1024, hidden=3584, dtype="bf16"), "rows_1024_of_4096"),
        # the projections of a sub-block step of 16 sequences
        _named(dict(kind="projections", batch=16, seq=8, hidden=3584, q_heads=28, kv_heads=4, cache=1024,
                    dtype="bf16"), "projections_16x8"),
        # sampling of a sub-block step of 16 sequences
        _named(dict(kind="unmask", batch=16, positions=8, vocab=VOCAB, dtype="bf16"), "unmask_16x8"),
        # a two-layer model's sub-block step of 16 sequences with the full vocabulary, eager
        _named(dict(kind="model", batch=16, seq=8, layers=2, keys=1056), "model_step_16x8"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sub_block", "block", "prompt", "prompt", "fp32", "rows", "projections", "unmask", "model"])
    hq, hkv = rng.choice(HEADS)
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    layout = rng.choice(["contiguous", "paged", "paged_hm"])
    if kind in ("sub_block", "block"):
        batch = _log(rng, 1, 48)
        lo = _log(rng, 64, 6000)
        hi = lo + rng.randint(0, 2 * lo)
        batch = max(1, min(batch, 600_000 // (lo + hi)))
        return _attention(batch=batch, q_len=rng.choice([8, 8, 4, 16]) if kind == "sub_block" else BLOCK, q_heads=hq,
                          kv_heads=hkv, min_keys=lo, max_keys=hi, layout=layout, dtype=dtype)
    if kind == "prompt":
        q_len = _log(rng, 40, 6000)
        batch = max(1, min(16, _log(rng, 1, 16), 16000 // q_len))
        mask = rng.choice(["all", "block"])
        prefix = BLOCK * rng.choice([0, 0, rng.randint(1, 64)])
        pairs = 28_000_000 if mask == "all" else 45_000_000  # at most the largest listed call's products
        while batch * q_len * (q_len + prefix) > pairs:
            batch, q_len = (batch - 1, q_len) if batch > 1 else (1, q_len * 9 // 10)
        return _attention(batch=batch, q_len=q_len, q_heads=hq, kv_heads=hkv, min_keys=q_len + prefix,
                          max_keys=q_len + prefix, layout=layout, mask=mask, write=rng.choice([False, True]),
                          dtype=dtype)
    if kind == "fp32":
        hq, hkv = 12, 2
        lo = _log(rng, 64, 2000)
        return _attention(batch=rng.choice([1, 1, 2, 4]), q_len=rng.choice([8, BLOCK, BLOCK]), q_heads=hq,
                          kv_heads=hkv, min_keys=lo, max_keys=lo + rng.randint(0, lo // 2), dtype="fp32")
    if kind == "rows":
        seq = _log(rng, 256, 16000)
        return dict(kind="rows", batch=rng.choice([1, 1, 2]), seq=seq, rows=max(1, int(seq * rng.uniform(0.02, 0.5))),
                    hidden=rng.choice([3584, 1536]), dtype=dtype)
    if kind == "projections":
        batch = _log(rng, 1, 64)
        return dict(kind="projections", batch=batch, seq=rng.choice([8, 8, BLOCK]), hidden=hq * HEAD_DIM, q_heads=hq,
                    kv_heads=hkv, cache=1024, dtype=dtype)
    if kind == "unmask":
        return dict(kind="unmask", batch=_log(rng, 1, 64), positions=rng.choice([8, 8, 4, 16]),
                    vocab=rng.choice([VOCAB, VOCAB, 32001]), dtype=dtype)
    seq = rng.choice([8, BLOCK])
    return dict(kind="model", batch=_log(rng, 1, 128 // seq), seq=seq, layers=rng.choice([1, 2]),
                keys=_log(rng, 64, 2000))


# ---------------------------------------------------------------------------------------
# inputs

def _lengths(case):
    """Visible keys per sequence: spread over the case's range in a fixed shuffled order."""
    n, lo, hi = case["batch"], case["min_keys"], case["max_keys"]
    out = [lo + (hi - lo) * i // max(n - 1, 1) for i in range(n)]
    random.Random(n * 7919 + lo).shuffle(out)
    return out


def _gen(seed, device="cuda"):
    return torch.Generator(device=device).manual_seed(seed)


def _randn(g, *shape, dtype=torch.bfloat16, scale=1.0):
    t = torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)
    return (t * scale).to(dtype) if scale != 1.0 else t.to(dtype)


def _attention_inputs(case, seed):
    """Queries, the cache as a program holds it and the per-sequence K / V rows' positions."""
    g = _gen(seed)
    dt = DTYPES[case["dtype"]]
    b, hkv = case["batch"], case["kv_heads"]
    lens = _lengths(case)
    st = {"q": _randn(g, b, case["q_len"], case["q_heads"], HEAD_DIM, dtype=dt),
          "lens": torch.tensor(lens, dtype=torch.int32, device="cuda"), "table": None}
    if case["layout"] == "contiguous":
        shape = (b, (max(lens) + 31) // 32 * 32, hkv, HEAD_DIM)
    else:
        per = [(n + PAGE - 1) // PAGE for n in lens]
        perm = torch.randperm(sum(per), generator=g, device="cuda").to(torch.int32)
        table = torch.zeros(b, max(per), dtype=torch.int32, device="cuda")
        at = 0
        for i, n in enumerate(per):
            table[i, :n] = perm[at:at + n]
            at += n
        st["table"] = table
        shape = (sum(per), PAGE, hkv, HEAD_DIM)
    for name in ("k", "v"):
        t = _randn(g, *shape, dtype=dt)
        if case["layout"] == "paged_hm":  # each page stored [Hkv, PAGE, D]
            t = t.transpose(1, 2).contiguous().transpose(1, 2)
        st[name] = t
    if case["write"]:
        for name in ("k_new", "v_new"):
            st[name] = _randn(g, b, case["q_len"], hkv, HEAD_DIM, dtype=dt)
    return st


def _rows_inputs(case, seed):
    g = _gen(seed)
    dt = DTYPES[case["dtype"]]
    b, s, t, h = case["batch"], case["seq"], case["rows"], case["hidden"]
    hid = torch.randn(b, s, h, generator=g, device="cuda")
    big = torch.rand(b, s, h, generator=g, device="cuda") < 0.01  # the outlier channels of hidden states
    hid = torch.where(big, hid * 20.0, hid).to(dt)
    idx = torch.stack([torch.randperm(s, generator=g, device="cuda")[:t] for _ in range(b)])
    w = (1.0 + 0.02 * torch.randn(h, generator=g, device="cuda")).to(dt)
    return {"hidden": hid, "idx": idx, "weight": w, "values": _randn(g, b, t, h, dtype=dt),
            "cache": _randn(g, b, s, h, dtype=dt), "current": _randn(g, b, s, h, dtype=dt)}


def _rotary(first, count, dt):
    """cos / sin [1, count, D] of the positions from ``first`` (theta 1e6), fp32 then cast."""
    inv = 1.0 / (1_000_000.0 ** (torch.arange(0, HEAD_DIM, 2, dtype=torch.float32, device="cuda") / HEAD_DIM))
    f = torch.arange(first, first + count, device="cuda").float()[:, None] * inv[None]
    f = torch.cat((f, f), dim=-1)
    return f.cos().to(dt)[None], f.sin().to(dt)[None]


def _projection_inputs(case, seed):
    g = _gen(seed)
    dt = DTYPES[case["dtype"]]
    b, s, h = case["batch"], case["seq"], case["hidden"]
    nq, nkv = case["q_heads"] * HEAD_DIM, case["kv_heads"] * HEAD_DIM
    st = {"x": _randn(g, b, s, h, dtype=dt)}
    for name, n in (("q", nq), ("k", nkv), ("v", nkv)):
        st["w" + name] = _randn(g, n, h, dtype=dt, scale=0.02)
        st["b" + name] = _randn(g, n, dtype=dt, scale=0.1)
    at = case["cache"] - BLOCK
    st["cos"], st["sin"] = _rotary(at, s, dt)
    st["start"] = torch.full((b,), at, dtype=torch.int32, device="cuda")
    for name, rows in (("cache", case["cache"]), ("block", BLOCK)):
        for x in "kv":
            st[f"{x}_{name}"] = torch.zeros(b, rows, case["kv_heads"], HEAD_DIM, dtype=dt, device="cuda")
    return st


def _unmask_inputs(case, seed):
    g = _gen(seed)
    dt = DTYPES[case["dtype"]]
    b, n, v = case["batch"], case["positions"], case["vocab"]
    lg = torch.randn(b, n, v, generator=g, device="cuda") * 2.0
    # about half of the positions have one clear token, the others compete
    tok = torch.randint(0, v - 1, (b, n, 1), generator=g, device="cuda")
    lg.scatter_(2, tok, torch.rand(b, n, 1, generator=g, device="cuda") * 20.0 + 6.0)
    masked = torch.rand(b, n, generator=g, device="cuda") < 0.7
    ids = torch.where(masked, torch.full_like(tok[..., 0], MASK_ID), tok[..., 0])
    return {"logits": lg.to(dt), "ids": ids, "tokens": ids.clone(),
            "finished": torch.zeros(b, dtype=torch.bool, device="cuda")}


def _config(case):
    return BlockDiffusionConfig(num_hidden_layers=case["layers"])


def _model_shapes(cfg):
    h, i, kv = cfg.hidden_size, cfg.intermediate_size, cfg.num_key_value_heads * cfg.head_dim
    out = {"model.embed_tokens.weight": (cfg.vocab_size, h), "lm_head.weight": (cfg.vocab_size, h),
           "model.norm.weight": (h,)}
    for n in range(cfg.num_hidden_layers):
        p = f"model.layers.{n}."
        out.update({p + "self_attn.q_proj.weight": (h, h), p + "self_attn.q_proj.bias": (h,),
                    p + "self_attn.k_proj.weight": (kv, h), p + "self_attn.k_proj.bias": (kv,),
                    p + "self_attn.v_proj.weight": (kv, h), p + "self_attn.v_proj.bias": (kv,),
                    p + "self_attn.o_proj.weight": (h, h), p + "mlp.gate_proj.weight": (i, h),
                    p + "mlp.up_proj.weight": (i, h), p + "mlp.down_proj.weight": (h, i),
                    p + "input_layernorm.weight": (h,), p + "post_attention_layernorm.weight": (h,)})
    return out


def _model_inputs(case, seed):
    """Weights by parameter name, token ids and the caches' contents before the step: the
    committed prefix and the open block (the last BLOCK of ``keys``)."""
    g = _gen(seed)
    cfg = _config(case)
    weights = {}
    for name, shape in _model_shapes(cfg).items():
        t = torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(0.0, 0.02, generator=g)
        weights[name] = t + 1.0 if name.endswith("norm.weight") else t
    b, n = case["batch"], max(case["keys"], BLOCK)
    ids = torch.randint(0, cfg.vocab_size - 1, (b, case["seq"]), generator=g, device="cuda")
    shape = (cfg.num_hidden_layers, b, n, cfg.num_key_value_heads, HEAD_DIM)
    return weights, ids, _randn(g, *shape), _randn(g, *shape), n


def prepare(case, seed):
    kind = case["kind"]
    if kind == "attention":
        st = _attention_inputs(case, seed)
        st["plain"] = case["layout"] == "contiguous" and case["mask"] == "all" and not case["write"]
        st["backend"] = get_attention_backend("hip")
        st["scale"] = HEAD_DIM ** -0.5
        st["mode"] = _ffi.MASK_BLOCK_CAUSAL if case["mask"] == "block" else _ffi.MASK_SEQLEN
    elif kind == "rows":
        st = _rows_inputs(case, seed)
        norm = RMSNorm(case["hidden"], 1e-6).to("cuda", DTYPES[case["dtype"]])
        with torch.no_grad():
            norm.weight.copy_(st["weight"])
        st["norm"], st["ops"] = norm, get_fused_ops()
    elif kind == "projections":
        st = _projection_inputs(case, seed)
    elif kind == "unmask":
        st = _unmask_inputs(case, seed)
        st["scratch"] = ops.UnmaskScratch(case["batch"], case["positions"], st["logits"].device)
    else:
        weights, ids, k, v, n = _model_inputs(case, seed)
        cfg = _config(case)
        model = build_model(cfg, "cuda")
        with torch.no_grad():
            for name, p in model.named_parameters():
                p.copy_(weights[name])
        impl = HipStaticAttention()
        cache, block = impl.make_caches(case["batch"], (n + 255) // 256 * 256, cfg, torch.bfloat16, "cuda", True)
        impl.patch(model, block)
        for layer in range(cfg.num_hidden_layers):
            cache.key_cache[layer][:, :n].copy_(k[layer])
            cache.value_cache[layer][:, :n].copy_(v[layer])
            block.key_cache[layer].copy_(k[layer][:, n - BLOCK:])
            block.value_cache[layer].copy_(v[layer][:, n - BLOCK:])
            block.note_update(layer)
        cache.set_kv_write_start(n - BLOCK)
        cache.set_scratch_seqlens(n)
        cache.prepare_write_idx(BLOCK)
        at = 0 if case["seq"] == BLOCK else 8
        st = {"model": model, "ids": ids, "cache": cache, "block": block, "at": at,
              "pos": torch.arange(n - BLOCK + at, n - BLOCK + at + case["seq"], device="cuda")}
    st["case"] = case
    return st


# ---------------------------------------------------------------------------------------
# one pass

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "attention":
        if state["plain"]:
            return state["backend"].flash_kvcache_attention(state["q"], state["k"], state["v"], state["lens"],
                                                            scaling=state["scale"])
        out = ops.block_attn(state["q"], state["k"], state["v"], state["lens"], state["scale"],
                             mask_mode=state["mode"], mask_block=BLOCK, page_table=state["table"],
                             page_size=PAGE if state["table"] is not None else 0,
                             k_new=state.get("k_new"), v_new=state.get("v_new"))
        return [out, state["k"], state["v"]] if case["write"] else out
    if kind == "rows":
        selected, normed = fused_gather_input_rmsnorm_pair(state["hidden"], state["idx"], state["norm"])
        current = state["ops"].scatter_and_return_cuda(state["values"], state["idx"], state["cache"],
                                                       state["current"])
        return [selected, normed, state["cache"], current]
    if kind == "projections":
        s = state
        q = ops.qkv_rope_kv_write(s["x"], s["wq"], s["bq"], s["wk"], s["bk"], s["wv"], s["bv"], s["cos"], s["sin"],
                                  s["k_cache"], s["v_cache"], write_start=s["start"], k_block=s["k_block"],
                                  v_block=s["v_block"])
        return [q, s["k_cache"], s["v_cache"], s["k_block"], s["v_block"]]
    if kind == "unmask":
        tokens = state["tokens"].copy_(state["ids"])  # every step starts from its own ids
        sc = ops.unmask_step(state["logits"], tokens, MASK_ID, 0.9, row_offset=0, shift=1,
                             finished=state["finished"], scratch=state["scratch"])
        return [tokens, sc.row_tok, sc.row_conf, sc.counts]
    with torch.no_grad():
        logits = state["model"](state["ids"], state["cache"], use_block_cache=True,
                                block_past_key_values=state["block"], replace_position=state["at"],
                                cache_position=state["pos"], logits_to_keep=case["seq"])
    cache = state["cache"]
    return [logits] + cache.key_cache + cache.value_cache


# ---------------------------------------------------------------------------------------
# the work a pass cannot do without

def work(case):
    kind = case["kind"]
    elem = 4 if case.get("dtype") == "fp32" else 2
    if kind == "attention":
        b, s, hq, hkv = case["batch"], case["q_len"], case["q_heads"], case["kv_heads"]
        lens = _lengths(case)
        rows = 2 * b * s * hq * HEAD_DIM * elem + sum(lens) * hkv * HEAD_DIM * elem * 2
        if case["write"]:
            # the call's own rows are read where the caller has them and written to the cache
            rows += 2 * b * s * hkv * HEAD_DIM * elem
        if case["mask"] == "all":
            pairs = sum(n * s for n in lens)
        else:
            pairs = sum(min(n, ((n - s + i) // BLOCK + 1) * BLOCK) for n in lens for i in range(s))
        return {"bytes": rows, "flops": 4 * pairs * hq * HEAD_DIM}
    if kind == "rows":
        n, h = case["batch"] * case["rows"], case["hidden"]
        return {"bytes": n * h * elem * (3 + 3) + h * elem + 2 * n * 8, "flops": 4 * n * h}
    if kind == "projections":
        n, h = case["batch"] * case["seq"], case["hidden"]
        nq, nkv = case["q_heads"] * HEAD_DIM, case["kv_heads"] * HEAD_DIM
        return {"bytes": elem * (n * h + (nq + 2 * nkv) * (h + 1) + n * nq + n * 4 * nkv + 2 * case["seq"] * HEAD_DIM),
                "flops": 2 * n * h * (nq + 2 * nkv)}
    if kind == "unmask":
        n = case["batch"] * case["positions"]
        return {"bytes": n * case["vocab"] * elem + n * 28, "flops": 4 * n * case["vocab"]}
    cfg = _config(case)
    n = case["batch"] * case["seq"]
    keys = max(case["keys"], BLOCK)
    params = sum(math.prod(s) for p, s in _model_shapes(cfg).items() if "embed_tokens" not in p)
    kv = cfg.num_hidden_layers * case["batch"] * keys * cfg.num_key_value_heads * HEAD_DIM * 2
    return {"bytes": 2 * (params + kv + n * cfg.vocab_size + n * cfg.hidden_size),
            "flops": 2 * n * params + cfg.num_hidden_layers * 4 * n * keys * cfg.hidden_size}


def tolerance(case):
    # The figures are about four times the distance between the kernels and 64-bit
    # arithmetic: one or two roundings to the data type, and sums in fp32.
    kind, dtype = case["kind"], case.get("dtype", "bf16")
    if kind == "attention":
        if dtype == "fp32":
            return {"rel": 1.5e-6}
        return {"rel": 1e-2 if dtype == "bf16" else 1.2e-3}
    if kind in ("rows", "projections"):
        return {"rel": 1e-2 if dtype == "bf16" else 1.2e-3}
    if kind == "unmask":
        # confidences are probabilities rounded to the logits' type; a sum in another order
        # may move one across a rounding boundary, and a tie with it
        return {"rel": 8e-3 if dtype == "bf16" else 1e-3, "differ": 0.02}
    return {"rel": 4e-2}


# ---------------------------------------------------------------------------------------
# the same results in 64 bits

def _cache_rows(st, case, lens, b):
    """Flat indices of sequence b's positions in the [pages * PAGE] (or [L]) key rows."""
    pos = torch.arange(lens[b], device="cuda")
    if st["table"] is None:
        return pos
    return st["table"][b].long()[pos // PAGE] * PAGE + pos % PAGE


def _attend(q, k, v, scale, limit=None):
    """q [S, Hq, D], k / v [L, Hkv, D] in float64; keys at or past limit[i] hidden."""
    s, hq, _ = q.shape
    rep = hq // k.shape[1]
    out = torch.empty_like(q)
    for h in range(hq):
        w = q[:, h].contiguous() @ k[:, h // rep].t().contiguous() * scale
        if limit is not None:
            w.masked_fill_(torch.arange(k.shape[0], device="cuda")[None] >= limit[:, None], float("-inf"))
        out[:, h] = torch.softmax(w, dim=-1) @ v[:, h // rep].contiguous()
    return out


def _exact_attention(case, seed):
    st = _attention_inputs(case, seed)
    lens, s = _lengths(case), case["q_len"]
    out = torch.empty(st["q"].shape, dtype=torch.float64, device="cuda")
    paged = st["table"] is not None
    for b, n in enumerate(lens):
        rows = _cache_rows(st, case, lens, b)
        kv = []
        for x in "kv":
            if case["write"]:
                new = st[f"{x}_new"][b]
                if paged:
                    flat = rows[n - s:]
                    st[x][flat // PAGE, flat % PAGE] = new
                else:
                    st[x][b, n - s:n] = new
            kv.append((st[x][rows // PAGE, rows % PAGE] if paged else st[x][b, :n]).double())
        limit = None
        if case["mask"] == "block":
            limit = ((n - s + torch.arange(s, device="cuda")) // BLOCK + 1) * BLOCK
        out[b] = _attend(st["q"][b].double(), kv[0], kv[1], HEAD_DIM ** -0.5, limit)
    return [out, st["k"].double(), st["v"].double()] if case["write"] else out


def _rms(x, w, eps=1e-6):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w


def _exact_rows(case, seed):
    st = _rows_inputs(case, seed)
    idx = st["idx"][..., None].expand(-1, -1, case["hidden"])
    x = torch.gather(st["hidden"], 1, idx).double()
    return [x, _rms(x, st["weight"].double()), st["cache"].scatter(1, idx, st["values"]).double(),
            st["current"].scatter(1, idx, st["values"]).double()]


def _rope(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos + torch.cat((-x[..., half:], x[..., :half]), dim=-1) * sin


def _exact_projections(case, seed):
    st = {n: t.double() if t.is_floating_point() else t for n, t in _projection_inputs(case, seed).items()}
    b, s = case["batch"], case["seq"]
    cos, sin = st["cos"][:, :, None], st["sin"][:, :, None]
    q, k, v = ((st["x"] @ st["w" + n].t().contiguous() + st["b" + n]).view(b, s, -1, HEAD_DIM) for n in "qkv")
    at = case["cache"] - BLOCK
    st["k_cache"][:, at:at + s] = st["k_block"][:, :s] = _rope(k, cos, sin)
    st["v_cache"][:, at:at + s] = st["v_block"][:, :s] = v
    return [_rope(q, cos, sin), st["k_cache"], st["v_cache"], st["k_block"], st["v_block"]]


def _exact_unmask(case, seed):
    st = _unmask_inputs(case, seed)
    lg = torch.cat([st["logits"][:, :1], st["logits"][:, :-1]], dim=1)
    tok, conf = [], []
    for row in lg:  # one sequence at a time: the vocabulary in 64 bits
        p = torch.softmax(row.double(), dim=-1).to(lg.dtype).float()
        top = p.max(dim=-1, keepdim=True).values
        tok.append((p == top).to(torch.uint8).argmax(dim=-1))
        conf.append(top[:, 0])
    tok, conf = torch.stack(tok), torch.stack(conf)
    masked = st["ids"] == MASK_ID
    c = torch.where(masked, conf, torch.full_like(conf, float("-inf")))
    un = c > 0.9
    un[torch.arange(case["batch"], device="cuda"), c.argmax(dim=-1)] = True
    un &= masked
    ids = torch.where(un, tok, st["ids"])
    left = ids == MASK_ID
    counts = torch.stack([un.sum(), (masked & ~un).sum(), left[:, 0].sum(), st["finished"].sum()])
    return [ids, tok, conf.double(), counts.to(torch.int32)]


def _exact_model(case, seed):
    weights, ids, kc, vc, n = _model_inputs(case, seed)
    cfg = _config(case)
    b, s = ids.shape
    at = n - BLOCK + (0 if s == BLOCK else 8)
    cos, sin = (t.double()[:, :, None] for t in _rotary(at, s, torch.bfloat16))
    length = (n + 255) // 256 * 256
    ck, cv = (torch.zeros(cfg.num_hidden_layers, b, length, *kc.shape[3:], dtype=torch.float64, device="cuda")
              for _ in range(2))
    ck[:, :, :n], cv[:, :, :n] = kc.double(), vc.double()

    def lin(x, name, bias=False):
        y = x @ weights[name + ".weight"].double().t().contiguous()
        return y + weights[name + ".bias"].double() if bias else y

    h = weights["model.embed_tokens.weight"][ids].double()
    for layer in range(cfg.num_hidden_layers):
        p = f"model.layers.{layer}."
        x = _rms(h, weights[p + "input_layernorm.weight"].double())
        q, k, v = (lin(x, p + f"self_attn.{y}_proj", True).view(b, s, -1, HEAD_DIM) for y in "qkv")
        ck[layer][:, at:at + s], cv[layer][:, at:at + s] = _rope(k, cos, sin), v
        a = torch.stack([_attend(r, ck[layer][i, :n], cv[layer][i, :n], HEAD_DIM ** -0.5)
                         for i, r in enumerate(_rope(q, cos, sin))])
        h = h + lin(a.reshape(b, s, -1), p + "self_attn.o_proj")
        x = _rms(h, weights[p + "post_attention_layernorm.weight"].double())
        gate = lin(x, p + "mlp.gate_proj")
        h = h + lin(gate * torch.sigmoid(gate) * lin(x, p + "mlp.up_proj"), p + "mlp.down_proj")
    logits = lin(_rms(h, weights["model.norm.weight"].double()), "lm_head")
    return [logits] + list(ck) + list(cv)


def exact(case, seed):
    return {"attention": _exact_attention, "rows": _exact_rows, "projections": _exact_projections,
            "unmask": _exact_unmask, "model": _exact_model}[case["kind"]](case, seed)
