"""What this framework is timed on: the calls a serving engine makes, through
the library's public entry points, from one user's decode step to a
long-context batch.

Kinds of case (``case["kind"]``) and the ranges draw() takes them from. Head
shapes and layer counts are those of the models the repository's benchmark
and configurations name (Qwen3-0.6B, Qwen3-8B, Qwen2.5-0.5B, Qwen2.5-7B).

decode   one decode step's attention in every layer: the step's plan, then per
         layer q/k norm + RoPE + append + paged GQA decode
         (rlse_decode_step_planned; one unplanned rlse_decode_step where the
         step has one layer and one sequence). Batches of 1 to 128 sequences,
         16 to 32768 cached tokens, bf16, f16 and f32.
fork     the same step for sequences forked from cached prefixes, the shared
         pages attended once (rlse_decode_step_cascade; with several prefixes
         and unforked sequences, rlse_decode_step_groups). 2 to 96 sequences,
         prefixes of 64 to 4096 tokens, bf16 and f16.
prefill  one layer's prefill attention of a prompt, or of a chunk after cached
         tokens: rlse_qk_norm_rope_append, rlse_prefill_attn. Chunks of 1 to
         2048 tokens after 0 to 8192 cached ones, bf16, f16 and f32.
dense    one layer's dense half: embedding rows in, the two RMSNorms, the
         q/k/v, output, gate/up and down projections with their epilogues,
         over packed weights as DecodeModel keeps them. 1 to 2048 rows (a
         decode batch or a prompt), bf16 and f16.
restore  a cached prefix's K/V snapshot written into pages and read back, all
         layers (rlse_kv_scatter, rlse_kv_gather). 1 to 4096 tokens.
step     a whole decode step of DecodeModel, replayed from its captured graph.
         1 to 64 sequences, 16 to 2048 cached tokens, bf16 and f16.
"""
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "mini-serve-rs_amd"))

import rlse_kv as kv  # noqa: E402
from decode_model import DecodeModel, ModelConfig  # noqa: E402

DEV = "cuda:0"
TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
EPS, THETA = 1e-6, 1e6

# name: (query heads, KV heads, head_dim, layers, q/k RMSNorm)
ATTN = {
    "qwen3_0_6b": (16, 8, 128, 28, True),
    "qwen2_5_0_5b": (14, 2, 64, 24, False),
    "qwen2_5_7b": (28, 4, 128, 28, False),
    "qwen3_8b": (32, 8, 128, 36, True),
}
# name: (hidden, query heads, KV heads, head_dim, intermediate, q/k/v bias)
DENSE = {
    "qwen3_0_6b": (1024, 16, 8, 128, 3072, False),
    "qwen2_5_0_5b": (896, 14, 2, 64, 4864, True),
}
VOCAB = 151936


def listed():
    return [
        # One user's decode step in f32, the reference's own dtype, one
        # attention layer: the smallest call, all launch and latency.
        {"name": "decode_one_f32", "kind": "decode", "model": "qwen3_0_6b", "dtype": "f32",
         "layers": 1, "batch": 1, "lo": 512, "hi": 512},
        # A busy server's step: 32 users in the middle of their answers.
        {"name": "decode_b32", "kind": "decode", "model": "qwen3_0_6b", "dtype": "bf16",
         "layers": 28, "batch": 32, "lo": 128, "hi": 2048},
        # Many users with long documents on the small high-GQA model.
        {"name": "decode_b64_gqa7", "kind": "decode", "model": "qwen2_5_0_5b", "dtype": "bf16",
         "layers": 24, "batch": 64, "lo": 4096, "hi": 4096},
        # Long contexts, large batch: the largest call (one layer, 10.7 GB).
        {"name": "decode_long", "kind": "decode", "model": "qwen3_8b", "dtype": "bf16",
         "layers": 1, "batch": 128, "lo": 8192, "hi": 32768},
        # 64 requests behind one system prompt.
        {"name": "fork_64", "kind": "fork", "model": "qwen3_0_6b", "dtype": "bf16",
         "layers": 28, "batch": 64, "groups": 1, "prefix": 1024, "unforked": 0, "lo": 64,
         "hi": 512},
        # A whole prompt of odd length, nothing cached.
        {"name": "prefill_prompt", "kind": "prefill", "model": "qwen3_0_6b", "dtype": "bf16",
         "tokens": 1000, "cached": 0},
        # A chunk of a long document's prefill.
        {"name": "prefill_chunk", "kind": "prefill", "model": "qwen3_8b", "dtype": "bf16",
         "tokens": 512, "cached": 8192},
        # A question after a restored prefix, in f32 (the reference's dtype).
        {"name": "prefill_suffix_f32", "kind": "prefill", "model": "qwen3_0_6b", "dtype": "f32",
         "tokens": 333, "cached": 1030},
        # The dense half of one layer over the same prompt.
        {"name": "dense_prompt", "kind": "dense", "model": "qwen3_0_6b", "dtype": "bf16",
         "rows": 1000},
        # A cached system prompt restored into pages, and exported again.
        {"name": "restore_prefix", "kind": "restore", "model": "qwen3_0_6b", "dtype": "bf16",
         "tokens": 1030, "start": 0},
        # The whole step of the busy server, logits out.
        {"name": "step_b32", "kind": "step", "model": "qwen3_0_6b", "dtype": "bf16",
         "batch": 32, "lo": 128, "hi": 2048},
        # The whole step of one user on the small model.
        {"name": "step_one", "kind": "step", "model": "qwen2_5_0_5b", "dtype": "bf16",
         "batch": 1, "lo": 512, "hi": 512},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "fork", "prefill", "prefill", "prefill", "dense",
                       "dense", "dense", "restore", "step"])
    if kind == "decode":
        model = rng.choice(list(ATTN))
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        batch = _log_int(rng, 1, 128)
        lo = _log_int(rng, 16, 16384)
        hi = min(32768, _log_int(rng, lo, 2 * lo))
        hq, hkv, d, layers, _ = ATTN[model]
        # at most 4 GB of K/V a step: as many of the model's layers as fit
        per = 2 * batch * hi * hkv * d * (4 if dtype == "f32" else 2)
        batch = max(1, min(batch, batch * 4_000_000_000 // per))
        per = 2 * batch * hi * hkv * d * (4 if dtype == "f32" else 2)
        return {"kind": kind, "model": model, "dtype": dtype,
                "layers": max(1, min(layers, 4_000_000_000 // per)), "batch": batch, "lo": lo,
                "hi": hi}
    if kind == "fork":
        groups = rng.choice([1, 1, rng.randint(2, 6)])
        batch = max(2 * groups, _log_int(rng, 2, 96))
        lo = _log_int(rng, 16, 512)
        return {"kind": kind, "model": rng.choice(["qwen3_0_6b", "qwen2_5_0_5b", "qwen2_5_7b"]),
                "dtype": rng.choice(["bf16", "bf16", "f16"]), "layers": rng.randint(4, 24),
                "batch": batch, "groups": groups, "prefix": _log_int(rng, 64, 4096),
                "unforked": 0 if groups == 1 else rng.randint(0, batch - 2 * groups), "lo": lo,
                "hi": _log_int(rng, lo, 8 * lo)}
    if kind == "prefill":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
        cached = rng.choice([0, _log_int(rng, 16, 8192)])
        return {"kind": kind, "model": rng.choice(list(ATTN)), "dtype": dtype,
                "tokens": _log_int(rng, 1, 512 if dtype == "f32" else 2048), "cached": cached}
    if kind == "dense":
        return {"kind": kind, "model": rng.choice(list(DENSE)),
                "dtype": rng.choice(["bf16", "bf16", "f16"]), "rows": _log_int(rng, 1, 2048)}
    if kind == "restore":
        return {"kind": kind, "model": rng.choice(["qwen3_0_6b", "qwen2_5_0_5b", "qwen2_5_7b"]),
                "dtype": rng.choice(["bf16", "f16", "f32"]), "tokens": _log_int(rng, 1, 4096),
                "start": rng.choice([0, rng.randint(1, 500)])}
    lo = _log_int(rng, 16, 1024)
    return {"kind": kind, "model": rng.choice(list(DENSE)),
            "dtype": rng.choice(["bf16", "bf16", "f16"]), "batch": _log_int(rng, 1, 64),
            "lo": lo, "hi": _log_int(rng, lo, 2048)}


# -- shared pieces -----------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _randn(g, dtype, *shape):
    return torch.randn(shape, generator=g, device=DEV, dtype=TORCH[dtype])


def _vec(g, dtype, n, base=1.0, sd=0.1):
    return (base + sd * torch.randn(n, generator=g, device=DEV)).to(TORCH[dtype])


def _rope_tables(d, max_pos, dtype):
    c, s = kv.rope_tables(THETA, d, max_pos, dtype)
    up = lambda b: torch.frombuffer(bytearray(b), dtype=torch.uint8).to(DEV).view(TORCH[dtype])  # noqa: E731,E501
    return up(c).view(max_pos, d // 2), up(s).view(max_pos, d // 2)


def _spread(batch, lo, hi):
    """Keys of a batch: cached lengths evenly over [lo, hi], plus the token of
    this step."""
    return [lo + (2 * i + 1) * (hi - lo + 1) // (2 * batch) + 1 for i in range(batch)]


def _lengths(g, batch, lo, hi):
    """_spread in a drawn order: every seed has the same pages in all, so the
    pools have one shape."""
    order = torch.randperm(batch, generator=g, device=DEV).cpu()
    return torch.tensor(_spread(batch, lo, hi))[order]


def _tables(g, pages, nb):
    """Block tables [batch][max pages] drawing each sequence's pages from one
    shuffled pool of nb."""
    mbps = int(max(pages))
    perm = torch.randperm(nb, generator=g, device=DEV).to(torch.int32).cpu()
    t = torch.zeros((len(pages), mbps), dtype=torch.int32)
    used = 0
    for i, k in enumerate(pages):
        t[i, :k] = perm[used:used + k]
        used += k
    return t, used


def _attn_inputs(case, seed):
    """Pools, queries, new tokens and tables of a decode or fork case."""
    hq, hkv, d, _, qk = ATTN[case["model"]]
    g, dt, b, layers = _gen(seed), case["dtype"], case["batch"], case["layers"]
    s = {"case": case}
    if case["kind"] == "decode":
        lens = _lengths(g, b, case["lo"], case["hi"])
        pages = [(int(n) + 15) // 16 for n in lens]
        nb = sum(pages) + 16
        table, _ = _tables(g, pages, nb)
    else:
        # Sequence i belongs to prefix i % groups; the last `unforked` have
        # none. Prefix j holds prefix >> j tokens (its whole pages shared).
        ng = case["groups"]
        shared = [max(1, (case["prefix"] >> j) // 16) for j in range(ng)]
        order = torch.randperm(b, generator=g, device=DEV).cpu().tolist()
        group = [-1] * b
        for at, i in enumerate(order[:b - case["unforked"]]):
            group[i] = at % ng
        own = _lengths(g, b, case["lo"], case["hi"])
        own_pages = [(int(n) + 15) // 16 for n in own]
        nb = sum(own_pages) + sum(shared) + 16
        flat, used = _tables(g, own_pages + shared, nb)
        total = [own_pages[i] + (shared[group[i]] if group[i] >= 0 else 0) for i in range(b)]
        table = torch.zeros((b, max(total)), dtype=torch.int32)
        lens = own.clone()
        for i in range(b):
            p = shared[group[i]] if group[i] >= 0 else 0
            if p:
                table[i, :p] = flat[b + group[i], :p]
            table[i, p:p + own_pages[i]] = flat[i, :own_pages[i]]
            lens[i] += 16 * p
        s["shared"], s["group"] = shared, group
        s["seq_group"] = torch.tensor(group, dtype=torch.int32, device=DEV)
        s["group_pages"] = torch.tensor(shared, dtype=torch.int32, device=DEV)
    mbps = table.shape[1]
    s.update(lens=lens, host_table=table, nb=nb, mbps=mbps, max_pos=mbps * 16,
             table=table.to(DEV), lens_dev=lens.to(torch.int32).to(DEV),
             k=_randn(g, dt, layers, nb, hkv, 16, d), v=_randn(g, dt, layers, nb, hkv, 16, d),
             q=_randn(g, dt, layers, b, hq, d), k_new=_randn(g, dt, layers, b, hkv, d),
             v_new=_randn(g, dt, layers, b, hkv, d),
             qw=_vec(g, dt, d) if qk else None, kw=_vec(g, dt, d) if qk else None)
    s["cos"], s["sin"] = _rope_tables(d, s["max_pos"], dt)
    return s


def _prefill_inputs(case, seed):
    hq, hkv, d, _, qk = ATTN[case["model"]]
    g, dt, t = _gen(seed), case["dtype"], case["tokens"]
    ctx = case["cached"] + t
    pages = (ctx + 15) // 16
    nb = pages + 16
    table, _ = _tables(g, [pages], nb)
    s = {"case": case, "ctx": ctx, "nb": nb, "mbps": pages, "max_pos": pages * 16,
         "table": table.to(DEV), "host_table": table,
         "k": _randn(g, dt, nb, hkv, 16, d), "v": _randn(g, dt, nb, hkv, 16, d),
         "q": _randn(g, dt, t, hq, d), "k_new": _randn(g, dt, t, hkv, d),
         "v_new": _randn(g, dt, t, hkv, d),
         "qw": _vec(g, dt, d) if qk else None, "kw": _vec(g, dt, d) if qk else None,
         "positions": torch.arange(case["cached"], ctx, dtype=torch.int32, device=DEV),
         "seq_index": torch.zeros(t, dtype=torch.int32, device=DEV)}
    s["cos"], s["sin"] = _rope_tables(d, s["max_pos"], dt)
    return s


def _dense_inputs(case, seed):
    """Weights 0.02 N(0,1) (the models' initialiser), norm weights near 1."""
    h, hq, hkv, d, inter, bias = DENSE[case["model"]]
    g, dt, rows = _gen(seed), case["dtype"], case["rows"]
    nq, nkv = hq * d, hkv * d
    mat = lambda o, i: _randn(g, dt, o, i) * 0.02  # noqa: E731
    return {"ids": torch.randint(0, VOCAB, (rows,), generator=g, device=DEV).to(torch.int32),
            "embed": _randn(g, dt, VOCAB, h), "in_norm": _vec(g, dt, h),
            "post_norm": _vec(g, dt, h), "qkv_w": mat(nq + 2 * nkv, h),
            "qkv_b": _vec(g, dt, nq + 2 * nkv, 0.0) if bias else None, "o_w": mat(h, nq),
            "gate_up_w": mat(2 * inter, h), "down_w": mat(h, inter),
            "attn": _randn(g, dt, rows, nq) * 0.3}


def _step_inputs(case, seed):
    """A model's weights (0.02 N(0,1), norm weights near 1), the cached K/V of
    its pool and one batch."""
    cfg = getattr(ModelConfig, case["model"])()
    g, dt, b = _gen(seed), case["dtype"], case["batch"]
    h, d = cfg.hidden, cfg.head_dim
    nq, nkv = cfg.heads * d, cfg.kv_heads * d
    mat = lambda o, i: _randn(g, dt, o, i) * 0.02  # noqa: E731
    w = {"embed": _randn(g, dt, cfg.vocab, h), "norm": _vec(g, dt, h)}
    for l in range(cfg.layers):
        p = f"l{l}."
        w.update({p + "in_norm": _vec(g, dt, h), p + "post_norm": _vec(g, dt, h),
                  p + "q_w": mat(nq, h), p + "k_w": mat(nkv, h), p + "v_w": mat(nkv, h),
                  p + "o_w": mat(h, nq), p + "gate_w": mat(cfg.inter, h),
                  p + "up_w": mat(cfg.inter, h), p + "down_w": mat(h, cfg.inter)})
        if cfg.qkv_bias:
            w.update({p + "q_b": _vec(g, dt, nq, 0.0), p + "k_b": _vec(g, dt, nkv, 0.0),
                      p + "v_b": _vec(g, dt, nkv, 0.0)})
        if cfg.qk_norm:
            w.update({p + "q_norm": _vec(g, dt, d), p + "k_norm": _vec(g, dt, d)})
    lens = _lengths(g, b, case["lo"], case["hi"])
    pages = [(int(n) + 15) // 16 for n in lens]
    nb = sum(pages) + 16
    table, _ = _tables(g, pages, nb)
    ids = torch.randint(0, cfg.vocab, (b,), generator=g, device=DEV).to(torch.int32)
    # K/V of pages 0 .. nb-1, as one contiguous snapshot of nb * 16 tokens
    shape = (cfg.layers, cfg.kv_heads, nb * 16, d)
    return cfg, w, lens, table, nb, ids, _randn(g, dt, *shape), _randn(g, dt, *shape)


# -- prepare -----------------------------------------------------------------
def prepare(case, seed):
    kind, dt = case["kind"], case["dtype"]
    if kind in ("decode", "fork"):
        hq, hkv, d, _, _ = ATTN[case["model"]]
        s = _attn_inputs(case, seed)
        b, layers = case["batch"], case["layers"]
        s["out"] = torch.empty((layers, b, hq, d), dtype=TORCH[dt], device=DEV)
        s["views"] = [tuple(s[n][l] for n in ("q", "k_new", "v_new", "k", "v", "out"))
                      for l in range(layers)]
        s["ws"] = torch.zeros(kv.decode_workspace_size(b, hq, hkv, d), dtype=torch.uint8,
                              device=DEV)
        s["plan"] = torch.zeros(kv.decode_plan_size(), dtype=torch.uint8, device=DEV)
        if kind == "fork":
            n = kv.decode_prefix_size(b, hq, d, max(s["shared"]))
            s["prefix"] = torch.zeros(n, dtype=torch.uint8, device=DEV)
        return s
    if kind == "prefill":
        hq, hkv, d, _, _ = ATTN[case["model"]]
        s = _prefill_inputs(case, seed)
        s["q_rot"], s["out"] = torch.empty_like(s["q"]), torch.empty_like(s["q"])
        n = kv.prefill_workspace_size(case["tokens"], s["ctx"], hq, hkv, d)
        s["ws"] = torch.zeros(max(n, 16), dtype=torch.uint8, device=DEV)
        return s
    if kind == "dense":
        h, hq, hkv, d, inter, _ = DENSE[case["model"]]
        rows, nq, nkv = case["rows"], hq * d, hkv * d
        s = _dense_inputs(case, seed)
        s["case"] = case
        shapes = {"qkv_w": (nq + 2 * nkv, h, 0), "o_w": (h, nq, 0),
                  "gate_up_w": (2 * inter, h, inter), "down_w": (h, inter, 0)}
        ws = 4
        for n, (o, i, pair) in shapes.items():
            w = torch.empty_like(s[n])
            kv.dense_pack(s[n], w, o, i, pair, dt, torch.cuda.current_stream())
            s[n] = w
            ws = max(ws, kv.dense_workspace_size(rows, o, i))
        s["ws"] = torch.zeros(ws, dtype=torch.uint8, device=DEV)
        z = lambda r, n: torch.zeros((r, n), dtype=TORCH[dt], device=DEV)  # noqa: E731
        tiles = (rows + 15) // 16 * 16  # packed rows come in whole 16-row tiles
        s.update(x=z(rows, h), h=z(tiles, h), act=z(tiles, inter), q=z(rows, nq),
                 k=z(rows, nkv), v=z(rows, nkv))
        return s
    if kind == "restore":
        hq, hkv, d, layers, _ = ATTN[case["model"]]
        g, n, start = _gen(seed), case["tokens"], case["start"]
        pages = (start + n + 15) // 16
        nb = pages + 16
        table, _ = _tables(g, [pages], nb)
        end = start + n
        return {"case": case, "nb": nb, "table": table.to(DEV),
                "k_in": _randn(g, dt, layers, hkv, n, d),
                "v_in": _randn(g, dt, layers, hkv, n, d),
                "pool": _randn(g, dt, layers, 2, nb, hkv, 16, d),
                "k_out": torch.empty((layers, hkv, end, d), dtype=TORCH[dt], device=DEV),
                "v_out": torch.empty((layers, hkv, end, d), dtype=TORCH[dt], device=DEV)}
    cfg, w, lens, table, nb, ids, kc, vc = _step_inputs(case, seed)
    b = case["batch"]
    model = DecodeModel(cfg, w, dt, nb, b, table.shape[1], DEV, stream_pages=True)
    every = torch.arange(nb, dtype=torch.int32, device=DEV)
    model.set_kv(every, kc, vc, stream=torch.cuda.current_stream())
    model.ids_in[:b].copy_(ids)
    model.tables_in[:b].copy_(table)
    model.lens_in[:b].copy_(lens.to(torch.int32))
    model.capture(b, feed_back=False)
    return {"case": case, "model": model, "batch": b}


# -- run ---------------------------------------------------------------------
def run(s):
    case = s["case"]
    kind, dt = case["kind"], case["dtype"]
    st = torch.cuda.current_stream()
    if kind == "step":
        logits, _ = s["model"].replay(s["batch"])
        return {"logits": logits}
    if kind in ("decode", "fork"):
        hq, hkv, d, _, _ = ATTN[case["model"]]
        b, mbps, nb, scale = case["batch"], s["mbps"], s["nb"], 1.0 / math.sqrt(d)
        t, lens, ws, plan = s["table"], s["lens_dev"], s["ws"], s["plan"]
        if kind == "decode" and b == 1 and case["layers"] == 1:
            for q, kn, vn, k, v, out in s["views"]:
                kv.decode_step(q, kn, vn, s["qw"], s["kw"], EPS, s["cos"], s["sin"],
                               s["max_pos"], k, v, t, lens, out, b, hq, hkv, d, mbps, nb, scale,
                               dt, ws, ws.numel(), st)
        elif kind == "decode":
            kv.decode_plan(t, lens, b, hkv, mbps, nb, plan, plan.numel(), st)
            for q, kn, vn, k, v, out in s["views"]:
                kv.decode_step_planned(q, kn, vn, s["qw"], s["kw"], EPS, s["cos"], s["sin"],
                                       s["max_pos"], k, v, t, lens, out, b, hq, hkv, d, mbps,
                                       nb, scale, dt, plan, ws, ws.numel(), st,
                                       stream_pages=True)
        elif case["groups"] == 1:
            pages, pre = s["shared"][0], s["prefix"]
            kv.decode_plan_cascade(t, lens, b, hkv, mbps, nb, pages, plan, plan.numel(), st)
            for q, kn, vn, k, v, out in s["views"]:
                kv.decode_step_cascade(q, kn, vn, s["qw"], s["kw"], EPS, s["cos"], s["sin"],
                                       s["max_pos"], k, v, t, lens, out, b, hq, hkv, d, mbps,
                                       nb, scale, dt, plan, pages, pre, pre.numel(), ws,
                                       ws.numel(), st, stream_pages=True)
        else:
            most, pre = max(s["shared"]), s["prefix"]
            kv.decode_plan_groups(t, lens, s["seq_group"], s["group_pages"], case["groups"], b,
                                  hq, hkv, mbps, nb, plan, plan.numel(), st)
            for q, kn, vn, k, v, out in s["views"]:
                kv.decode_step_groups(q, kn, vn, s["qw"], s["kw"], EPS, s["cos"], s["sin"],
                                      s["max_pos"], k, v, t, lens, out, b, hq, hkv, d, mbps,
                                      nb, scale, dt, plan, case["groups"], most, pre,
                                      pre.numel(), ws, ws.numel(), st, stream_pages=True)
        return {"out": s["out"], "k": s["k"], "v": s["v"]}
    if kind == "prefill":
        hq, hkv, d, _, _ = ATTN[case["model"]]
        n, ws = case["tokens"], s["ws"]
        kv.qk_norm_rope_append(s["q"], s["k_new"], s["v_new"], s["qw"], s["kw"], EPS, s["cos"],
                               s["sin"], s["max_pos"], s["positions"], s["table"], 1,
                               s["seq_index"], n, hq, hkv, d, s["mbps"], s["nb"], s["q_rot"],
                               s["k"], s["v"], dt, st)
        kv.prefill_attn(s["q_rot"], s["k"], s["v"], s["table"], s["ctx"], n, s["out"], hq, hkv,
                        d, s["mbps"], s["nb"], 1.0 / math.sqrt(d), dt, ws, ws.numel(), st)
        return {"out": s["out"], "k": s["k"], "v": s["v"]}
    if kind == "dense":
        h, hq, hkv, d, inter, _ = DENSE[case["model"]]
        rows, nq, nkv, ws = case["rows"], hq * d, hkv * d, s["ws"]
        kv.embedding(s["ids"], s["embed"], s["x"], rows, h, VOCAB, dt, st)
        kv.add_rmsnorm(None, s["x"], s["in_norm"], s["h"], rows, h, EPS, dt, st, packed_out=True)
        kv.qkv_proj(s["h"], s["qkv_w"], s["qkv_b"], s["q"], s["k"], s["v"], rows, h, nq, nkv, dt,
                    ws, st, packed=True, packed_x=True)
        kv.linear_residual(s["attn"], s["o_w"], s["x"], rows, h, nq, dt, ws, st, packed=True)
        kv.add_rmsnorm(None, s["x"], s["post_norm"], s["h"], rows, h, EPS, dt, st,
                       packed_out=True)
        kv.gate_up_silu(s["h"], s["gate_up_w"], s["act"], rows, h, inter, dt, ws, st,
                        packed=True, packed_x=True, packed_out=True)
        kv.linear_residual(s["act"], s["down_w"], s["x"], rows, h, inter, dt, ws, st,
                           packed=True, packed_x=True)
        return {"q": s["q"], "k": s["k"], "v": s["v"], "x": s["x"]}
    hq, hkv, d, layers, _ = ATTN[case["model"]]
    n, start, pool = case["tokens"], case["start"], s["pool"]
    stride, end = pool[0].numel(), case["start"] + case["tokens"]
    kv.kv_scatter(s["k_in"], s["v_in"], pool[:, 0], pool[:, 1], stride, layers, s["table"],
                  start, n, hkv, d, s["nb"], dt, st)
    kv.kv_gather(pool[:, 0], pool[:, 1], stride, layers, s["table"], end, s["k_out"],
                 s["v_out"], hkv, d, s["nb"], dt, st)
    return {"k": s["k_out"], "v": s["v_out"], "pool": pool}


# -- work --------------------------------------------------------------------
def work(case):
    """Bytes: every input and output once."""
    kind = case["kind"]
    es = 4 if case["dtype"] == "f32" else 2
    if kind in ("decode", "fork"):
        hq, hkv, d, _, _ = ATTN[case["model"]]
        b = case["batch"]
        own = sum(_spread(b, case["lo"], case["hi"]))
        attended = own
        if kind == "fork":
            ng = case["groups"]
            shared = [max(1, (case["prefix"] >> j) // 16) * 16 for j in range(ng)]
            members = b - case["unforked"]
            own += sum(shared)  # each prefix once
            attended += sum(shared[i % ng] for i in range(members))
        # K/V of every page, the queries and outputs, the new token in and out
        per = 2 * own * hkv * d * es + 2 * b * hq * d * es + 4 * b * hkv * d * es
        return {"bytes": case["layers"] * per,
                "flops": case["layers"] * 4.0 * attended * hq * d}
    if kind == "prefill":
        hq, hkv, d, _, _ = ATTN[case["model"]]
        n, cached = case["tokens"], case["cached"]
        pairs = n * cached + n * (n + 1) / 2
        return {"bytes": 2 * (cached + n) * hkv * d * es + 2 * n * hq * d * es
                + 2 * n * hkv * d * es, "flops": 4.0 * d * hq * pairs}
    if kind == "dense":
        h, hq, hkv, d, inter, _ = DENSE[case["model"]]
        rows, nq, nkv = case["rows"], hq * d, hkv * d
        weights = h * (nq + 2 * nkv) + h * nq + 3 * h * inter
        return {"bytes": es * (weights + rows * (2 * h + 2 * nq + 2 * nkv)),
                "flops": 2.0 * rows * weights}
    if kind == "restore":
        hq, hkv, d, layers, _ = ATTN[case["model"]]
        n, end = case["tokens"], case["start"] + case["tokens"]
        row = 2 * layers * hkv * d * es
        return {"bytes": 2.0 * row * (n + end), "flops": 0}
    cfg = getattr(ModelConfig, case["model"])()
    b = case["batch"]
    keys = sum(_spread(b, case["lo"], case["hi"]))
    nq, nkv = cfg.heads * cfg.head_dim, cfg.kv_heads * cfg.head_dim
    weights = cfg.layers * (cfg.hidden * (2 * nq + 2 * nkv) + 3 * cfg.hidden * cfg.inter)
    weights += cfg.vocab * cfg.hidden
    attn = cfg.layers * keys * nkv
    return {"bytes": es * (weights + 2 * attn + b * cfg.vocab),
            "flops": 2.0 * b * weights + 4.0 * cfg.layers * keys * nq}


# -- tolerance and exact -----------------------------------------------------
def tolerance(case):
    """About four times what each path shows against 64 bits. 16-bit
    attention: one layer's rotated queries, probabilities and outputs rounded
    to 16 bits (0.004 in bf16, 0.0005 in f16). Dense: a chain of four products
    with 16-bit activations between them (0.003, 0.0004). A whole step: the
    same through every layer (0.018 in bf16)."""
    kind = case["kind"]
    if kind == "restore":
        return "exact"
    if case["dtype"] == "f32":
        return {"rel": 1e-5}
    half = case["dtype"] == "f16"
    if kind == "step":
        return {"rel": 0.008 if half else 0.03}
    return {"rel": 0.002 if half else 0.015}


def _norm_rope64(x, w, cos, sin, pos):
    """q/k RMSNorm (where the model has it) and NeoX RoPE of [n][heads][d]."""
    x = x.double()
    if w is not None:
        x = x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()
    c, s = cos[pos].double()[:, None, :], sin[pos].double()[:, None, :]
    a, b = x.chunk(2, -1)
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _rows64(pool, table, n):
    """The first n tokens of one sequence's pages: [heads][n][d] in 64 bits."""
    p = pool[table[:(n + 15) // 16].long()]
    return p.permute(1, 0, 2, 3).reshape(p.shape[1], -1, p.shape[3])[:, :n].double()


def _attend64(q, k, v, first):
    """q [t][Hq][d] over k/v [Hkv][n][d]; query i sees keys 0 .. first + i."""
    t, hq, d = q.shape
    hkv, n, _ = k.shape
    q = q.view(t, hkv, hq // hkv, d).permute(1, 2, 0, 3).reshape(hkv, -1, d)
    out = torch.empty_like(q)
    for h in range(hkv):
        sc = q[h] @ k[h].t().contiguous() / math.sqrt(d)
        if t > 1:
            see = torch.arange(n, device=DEV)[None, :] <= (
                first + torch.arange(t, device=DEV))[:, None]
            sc = sc.masked_fill(~see.repeat(hq // hkv, 1), -math.inf)
        out[h] = torch.softmax(sc, -1) @ v[h]
    return out.view(hkv, hq // hkv, t, d).permute(2, 0, 1, 3).reshape(t, hq, d)


def _decode64(q, kn, vn, k, v, table, lens):
    """Rotated q [b][Hq][d] over each sequence's cached rows and its new one."""
    out = torch.empty_like(q)
    for i in range(q.shape[0]):
        n = int(lens[i])
        ki, vi = _rows64(k, table[i], n), _rows64(v, table[i], n)
        ki[:, n - 1], vi[:, n - 1] = kn[i], vn[i].double()
        out[i] = _attend64(q[i:i + 1], ki, vi, n - 1)[0]
    return out


def _rms64(x, w):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()


def exact(case, seed):
    kind = case["kind"]
    if kind == "restore":
        return None
    if kind in ("decode", "fork"):
        s = _attn_inputs(case, seed)
        pos = s["lens_dev"].long() - 1
        out = []
        for l in range(case["layers"]):
            q = _norm_rope64(s["q"][l], s["qw"], s["cos"], s["sin"], pos)
            kn = _norm_rope64(s["k_new"][l], s["kw"], s["cos"], s["sin"], pos)
            out.append(_decode64(q, kn, s["v_new"][l], s["k"][l], s["v"][l], s["table"],
                                 s["lens"]))
        return {"out": torch.stack(out), "k": None, "v": None}
    if kind == "prefill":
        s = _prefill_inputs(case, seed)
        pos, n, ctx = s["positions"].long(), case["tokens"], s["ctx"]
        q = _norm_rope64(s["q"], s["qw"], s["cos"], s["sin"], pos)
        kn = _norm_rope64(s["k_new"], s["kw"], s["cos"], s["sin"], pos)
        k, v = _rows64(s["k"], s["table"][0], ctx), _rows64(s["v"], s["table"][0], ctx)
        k[:, ctx - n:], v[:, ctx - n:] = kn.transpose(0, 1), s["v_new"].double().transpose(0, 1)
        return {"out": _attend64(q, k, v, ctx - n), "k": None, "v": None}
    if kind == "dense":
        h, hq, hkv, d, inter, _ = DENSE[case["model"]]
        s = _dense_inputs(case, seed)
        nq, nkv = hq * d, hkv * d
        lin = lambda x, w: x @ w.double().t().contiguous()  # noqa: E731
        x = s["embed"][s["ids"].long()].double()
        qkv = lin(_rms64(x, s["in_norm"]), s["qkv_w"])
        if s["qkv_b"] is not None:
            qkv = qkv + s["qkv_b"].double()
        x = x + lin(s["attn"].double(), s["o_w"])
        gu = lin(_rms64(x, s["post_norm"]), s["gate_up_w"])
        x = x + lin(torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:], s["down_w"])
        return {"q": qkv[:, :nq], "k": qkv[:, nq:nq + nkv], "v": qkv[:, nq + nkv:], "x": x}
    cfg, w, lens, table, nb, ids, kc, vc = _step_inputs(case, seed)
    b, d = case["batch"], cfg.head_dim
    nq, nkv = cfg.heads * d, cfg.kv_heads * d
    cos, sin = _rope_tables(d, table.shape[1] * 16, case["dtype"])
    pos = lens.to(DEV).long() - 1
    table = table.to(DEV)
    paged = lambda c: c.view(cfg.kv_heads, nb, 16, d).permute(1, 0, 2, 3)  # noqa: E731
    x = w["embed"][ids.long()].double()
    for l in range(cfg.layers):
        p = f"l{l}."
        lin = lambda a, n: (a @ w[p + n + "_w"].double().t().contiguous() + (  # noqa: E731
            w[p + n + "_b"].double() if p + n + "_b" in w else 0.0))
        hid = _rms64(x, w[p + "in_norm"])
        q = _norm_rope64(lin(hid, "q").view(b, cfg.heads, d), w.get(p + "q_norm"), cos, sin, pos)
        kn = _norm_rope64(lin(hid, "k").view(b, cfg.kv_heads, d), w.get(p + "k_norm"), cos, sin,
                          pos)
        vn = lin(hid, "v").view(b, cfg.kv_heads, d)
        att = _decode64(q, kn, vn, paged(kc[l]), paged(vc[l]), table, lens)
        x = x + lin(att.view(b, nq), "o")
        hid = _rms64(x, w[p + "post_norm"])
        x = x + lin(torch.nn.functional.silu(lin(hid, "gate")) * lin(hid, "up"), "down")
    emb = w["embed"] if cfg.tied else w["lm_head"]
    return {"logits": _rms64(x, w["norm"]) @ emb.double().t().contiguous()}
