"""Chunked-prefill attention (MFMA tiles) on the GPU against the oracle.

Reference: the prefill branch of Attention::forward (src/backends/qwen2.rs:
329-345) with prepare_causal_attention_mask (:476-503): the chunk's queries
at positions offset .. offset+Tq-1 see keys 0 .. offset+t, query head hq
reading KV head hq // G. The oracle is orc_prefill_f32 (the C restatement of
that Candle CPU path, pinned against float64 in tests/test_oracle.py), run on
the same bf16/f16-rounded inputs laid out contiguously as KvCache holds them.
Bars: max-abs 2e-2 for bf16 and f16 (the probabilities enter the P.V product
rounded to the pool dtype), 2e-3 for f32 (the reference CPU path's dtype: f32
products on f32 MFMAs); the relative error is printed beside it.
"""
import importlib.util
import math
import shutil
import sys

import numpy as np
import pytest
import torch

import oracle as O
from gpu_helpers import DEV, TOL, as_f32, err_report, random_values, to_dev, to_host

pytestmark = pytest.mark.gpu


def make_case(rng, hq, hkv, d, tq, offset, dtype, spare_blocks=9):
    """Random pool + one sequence of ctx_len = offset + tq keys on shuffled pages."""
    L = offset + tq
    npages = (L + 15) // 16
    nb = npages + spare_blocks
    table = rng.permutation(nb)[:npages].astype(np.int32)
    kp = random_values(rng, (nb, hkv, 16, d), dtype)
    vp = random_values(rng, (nb, hkv, 16, d), dtype)
    q = random_values(rng, (tq, hq, d), dtype)
    return q, kp, vp, table, L


def run_prefill(kv, q, kp, vp, table, L, hq, hkv, d, dtype, scale, max_blocks=None):
    tq = q.shape[0]
    qd, kd, vd = to_dev(q, dtype), to_dev(kp, dtype), to_dev(vp, dtype)
    out = torch.empty_like(qd)
    td = to_dev(table)
    mb = max_blocks if max_blocks is not None else table.shape[0]
    kv.prefill_attn(qd, kd, vd, td, L, tq, out, hq, hkv, d, mb, kp.shape[0], scale, dtype)
    return to_host(out)


def oracle_prefill(q, kp, vp, table, L, hq, hkv, d, dtype, scale, heads=None):
    """orc_prefill_f32 on the contiguous [Hkv, L, d] buffers; q token-major
    [Tq, Hq, d] is transposed to the oracle's [Hq, Tq, d]. heads = a KV-head
    subset to evaluate (returns [Tq, len(heads)*G, d])."""
    tq = q.shape[0]
    g = hq // hkv
    kc = as_f32(O.paged_to_contiguous(kp, table, L), dtype)
    vc = as_f32(O.paged_to_contiguous(vp, table, L), dtype)
    qf = as_f32(q, dtype)
    heads = list(range(hkv)) if heads is None else heads
    outs = []
    for h in heads:
        qh = np.ascontiguousarray(qf[:, h * g:(h + 1) * g, :].transpose(1, 0, 2))
        o = O.prefill_f32(qh, kc[h:h + 1], vc[h:h + 1], L - tq, scale)
        outs.append(o.transpose(1, 0, 2))
    return np.concatenate(outs, axis=1)


def check(name, got, want, dtype):
    mx, rel = err_report(got, want)
    print(f"[{name}] dtype={dtype} max_abs={mx:.3e} rel={rel:.3e}")
    assert np.isfinite(got).all()
    assert mx <= TOL[dtype], (name, mx)


SHAPES = [(32, 8, 128), (14, 2, 64), (8, 8, 128), (16, 2, 128)]
CHUNKS = [(1, 0), (1, 37), (7, 0), (64, 100), (130, 5), (300, 1000)]


@pytest.mark.parametrize("dtype", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"Hq{s[0]}-Hkv{s[1]}-d{s[2]}")
def test_prefill_matches_oracle(kv, dtype, shape):
    hq, hkv, d = shape
    rng = np.random.default_rng(hq * 1000 + d)
    scale = 1.0 / math.sqrt(d)
    for tq, offset in CHUNKS:
        q, kp, vp, table, L = make_case(rng, hq, hkv, d, tq, offset, dtype)
        print(f"case Hq={hq} Hkv={hkv} d={d} Tq={tq} offset={offset} {dtype}", flush=True)
        got = as_f32(run_prefill(kv, q, kp, vp, table, L, hq, hkv, d, dtype, scale), dtype)
        want = oracle_prefill(q, kp, vp, table, L, hq, hkv, d, dtype, scale)
        check(f"prefill Tq={tq} off={offset}", got, want, dtype)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_prefill_split_keys_path(kv, dtype):
    """Few row tiles over a long context: the keys are split across
    workgroups and merged; the result must not depend on the split."""
    hq, hkv, d = 8, 8, 128
    rng = np.random.default_rng(11)
    for tq, offset in [(16, 3000), (64, 5000), (3, 9000)]:
        q, kp, vp, table, L = make_case(rng, hq, hkv, d, tq, offset, dtype)
        ws = kv.prefill_workspace_size(tq, L, hq, hkv, d)
        print(f"split case Tq={tq} offset={offset} workspace={ws}", flush=True)
        assert ws > 0  # this shape must take the split path
        got = as_f32(run_prefill(kv, q, kp, vp, table, L, hq, hkv, d, dtype, 1 / math.sqrt(d)),
                     dtype)
        want = oracle_prefill(q, kp, vp, table, L, hq, hkv, d, dtype, 1 / math.sqrt(d))
        check(f"split Tq={tq} off={offset}", got, want, dtype)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_prefill_skips_invalid_pages(kv, dtype):
    """Keys on pages whose id is outside the pool are skipped, as the decode
    kernel does; checked against a float64 evaluation with those keys masked."""
    hq, hkv, d = 4, 2, 64
    rng = np.random.default_rng(5)
    tq, offset = 20, 80
    q, kp, vp, table, L = make_case(rng, hq, hkv, d, tq, offset, dtype)
    nb = kp.shape[0]
    bad = table.copy()
    bad[1] = nb + 3      # out of range
    bad[3] = -1          # negative
    scale = 1 / math.sqrt(d)
    print("invalid-page case", flush=True)
    got = as_f32(run_prefill(kv, q, kp, vp, bad, L, hq, hkv, d, dtype, scale), dtype)
    kc = as_f32(O.paged_to_contiguous(kp, table, L), dtype).astype(np.float64)
    vc = as_f32(O.paged_to_contiguous(vp, table, L), dtype).astype(np.float64)
    qf = as_f32(q, dtype).astype(np.float64)
    g = hq // hkv
    keep = np.ones(L, bool)
    keep[16:32] = False
    keep[48:64] = False
    want = np.zeros_like(qf)
    for t in range(tq):
        for hh in range(hq):
            s = kc[hh // g] @ qf[t, hh] * scale
            vis = keep & (np.arange(L) <= offset + t)
            s = np.where(vis, s, -np.inf)
            p = np.exp(s - s.max())
            want[t, hh] = (p / p.sum()) @ vc[hh // g]
    check("invalid pages skipped", got, want, dtype)


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("hq,hkv,tq,offset", [
    (16, 8, 32, 200),    # two key groups, one split; spare waves only stage
    (16, 8, 200, 200),   # the full kernel
    (4, 1, 3, 2000),     # eight splits
    (4, 1, 150, 4100)])  # twelve, of three steps each
@pytest.mark.parametrize("bad", ["even", "odd", "all even", "all odd", "each in turn"])
def test_prefill_key_groups_skip_invalid_pages(kv, dtype, hq, hkv, tq, offset, bad):
    """Two key groups take the even and the odd 64-key tiles of a step: page
    ids outside the pool in the tiles of one group only, on every page of that
    group (its keys are all masked) or at another place in each tile hide the
    same keys as a float64 evaluation without them."""
    d = 128
    rng = np.random.default_rng(tq + offset)
    q, kp, vp, table, L = make_case(rng, hq, hkv, d, tq, offset, dtype)
    scale = 1 / math.sqrt(d)
    page = np.arange(len(table))
    odd, at = page // 4 % 2 == 1, page % 4
    hit = {"even": ~odd & (at == 1), "odd": odd & (at == 2), "all even": ~odd, "all odd": odd,
           "each in turn": page % 8 == page // 8 % 8}[bad]
    table_bad = table.copy()
    table_bad[hit] = np.where(page[hit] % 3 == 0, -1, kp.shape[0] + page[hit]).astype(np.int32)
    got = as_f32(run_prefill(kv, q, kp, vp, table_bad, L, hq, hkv, d, dtype, scale), dtype)
    kc = as_f32(O.paged_to_contiguous(kp, table, L), dtype).astype(np.float64)
    vc = as_f32(O.paged_to_contiguous(vp, table, L), dtype).astype(np.float64)
    qf = as_f32(q, dtype).astype(np.float64)
    visible = ~np.repeat(hit, 16)[:L] & (np.arange(L) <= offset + np.arange(tq)[:, None])
    want = np.zeros_like(qf)
    for hh in range(hq):
        x = np.where(visible, qf[:, hh] @ kc[hh // (hq // hkv)].T * scale, -np.inf)
        p = np.exp(x - x.max(1, keepdims=True))
        want[:, hh] = p / p.sum(1, keepdims=True) @ vc[hh // (hq // hkv)]
    check(f"invalid pages, {bad}", got, want, dtype)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_prefill_qwen3_8b_chunk(kv, dtype):
    """The Qwen3-8B chunk: 512 queries after 8192 cached tokens, 32 q / 8 kv
    heads, d=128, bf16 and f32; KV heads 0 and 7 checked against the oracle."""
    hq, hkv, d = 32, 8, 128
    rng = np.random.default_rng(8)
    q, kp, vp, table, L = make_case(rng, hq, hkv, d, 512, 8192, dtype)
    print(f"qwen3-8b chunk Tq=512 offset=8192 {dtype}", flush=True)
    got = as_f32(run_prefill(kv, q, kp, vp, table, L, hq, hkv, d, dtype, 1 / math.sqrt(d)),
                 dtype)
    assert np.isfinite(got).all()
    g = hq // hkv
    want = oracle_prefill(q, kp, vp, table, L, hq, hkv, d, dtype, 1 / math.sqrt(d), heads=[0, 7])
    sub = np.concatenate([got[:, 0:g], got[:, 7 * g:8 * g]], axis=1)
    check("qwen3-8b chunk heads 0,7", sub, want, dtype)
    # Every KV head (each one's row tiles on their own XCD and key splits) on
    # the tokens at the edges of the 64-token row tiles and at the chunk ends.
    tq = q.shape[0]
    kc = as_f32(O.paged_to_contiguous(kp, table, L), dtype)
    vc = as_f32(O.paged_to_contiguous(vp, table, L), dtype)
    qf = as_f32(q, dtype)
    toks = [0, 1, 63, 64, 127, 128, 191, 255, 256, 319, 383, 384, 447, 448, 510, 511]
    worst = 0.0
    for h in range(hkv):
        for t in toks:
            qh = np.ascontiguousarray(qf[t:t + 1, h * g:(h + 1) * g, :].transpose(1, 0, 2))
            o = O.prefill_f32(qh, kc[h:h + 1], vc[h:h + 1], L - tq + t, 1 / math.sqrt(d))
            mx, _ = err_report(got[t, h * g:(h + 1) * g], o[:, 0, :])
            worst = max(worst, mx)
            assert mx <= TOL[dtype], (h, t, mx)
    print(f"qwen3-8b chunk: all {hkv} KV heads x {len(toks)} tokens within {worst:.3e}")


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_prefill_single_token_equals_decode(kv, dtype):
    """A one-token chunk is the decode of that token over its prefix."""
    hq, hkv, d = 16, 8, 128
    rng = np.random.default_rng(3)
    q, kp, vp, table, L = make_case(rng, hq, hkv, d, 1, 200, dtype)
    scale = 1 / math.sqrt(d)
    print("single-token chunk vs decode", flush=True)
    got = run_prefill(kv, q, kp, vp, table, L, hq, hkv, d, dtype, scale)
    out = torch.empty_like(to_dev(q, dtype))
    qd, kd, vd = to_dev(q, dtype), to_dev(kp, dtype), to_dev(vp, dtype)
    td, ld = to_dev(table.reshape(1, -1)), to_dev(np.array([L], np.int32))
    kv.paged_gqa_decode(qd, kd, vd, td, ld, out, 1, hq, hkv, d, table.shape[0], kp.shape[0],
                        scale, dtype)
    dec = to_host(out)
    mx, rel = err_report(as_f32(got, dtype), as_f32(dec, dtype))
    print(f"[prefill(1) vs decode] max_abs={mx:.3e} rel={rel:.3e}")
    assert mx <= TOL[dtype]


@pytest.mark.parametrize("dtype", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("hq,hkv,d,tq,offset", [
    (16, 8, 128, 32, 200),   # 64 rows: the last chunk whose spare waves only stage (2 key groups)
    (16, 8, 128, 33, 200),   # 66 rows
    (16, 8, 128, 65, 130),   # 130 rows: two half tiles, four tiles of keys
    (4, 1, 128, 3, 2000),    # many splits, an odd number of tiles in some
    (4, 1, 128, 150, 4100),  # 600 rows after a long context: splits and two key groups
    (14, 2, 64, 27, 300),    # 189 rows of 256: spare waves, one key group
    (14, 2, 64, 28, 301)])   # 196 rows
def test_prefill_row_and_key_groups_match_oracle(kv, dtype, hq, hkv, d, tq, offset):
    """Chunks around the edges of the row tiles, the key groups and the
    splits, one page id outside the pool never read (its keys invisible to no
    query: past the context)."""
    rng = np.random.default_rng(tq * 7 + offset)
    q, kp, vp, table, L = make_case(rng, hq, hkv, d, tq, offset, dtype)
    scale = 1.0 / np.sqrt(d)
    table = np.concatenate([table, np.array([kp.shape[0] + 5], np.int32)])
    got = as_f32(run_prefill(kv, q, kp, vp, table, L, hq, hkv, d, dtype, scale), dtype)
    want = oracle_prefill(q, kp, vp, table, L, hq, hkv, d, dtype, scale)
    mx, rel = err_report(got, want)
    print(f"[prefill groups {hq}/{hkv}/{d} {tq}+{offset}] {dtype} max_abs={mx:.3e} rel={rel:.3e}")
    assert np.isfinite(got).all() and mx <= TOL[dtype]


@pytest.mark.parametrize("dtype,hq,hkv,d,large,small", [
    ("f32", 16, 8, 128, (256, 1280), (200, 1000)),
    ("bf16", 28, 4, 128, (2048, 2048), (200, 1000)),
    ("bf16", 14, 2, 64, (2048, 2100), (64, 1500)),
    ("f16", 32, 8, 128, (512, 17000), (5, 9000))])
def test_prefill_workspace_holds_for_smaller_calls(kv, dtype, hq, hkv, d, large, small):
    """A workspace sized once for the longest chunk and context is enough for
    every smaller call, and the size never falls with either length."""
    size = kv.prefill_workspace_size(*large, hq, hkv, d)
    for tq in (1, 7, 64, 200, 500, 1000, 1667, 2048):
        for ctx in (2048, 2100, 9743, 17000, 40000):
            n = kv.prefill_workspace_size(tq, ctx, hq, hkv, d)
            assert n >= kv.prefill_workspace_size(tq, max(tq, ctx - 900), hq, hkv, d)
            assert n >= kv.prefill_workspace_size(max(1, tq // 2), ctx, hq, hkv, d)
            # two blocks of 256 rows (f32 sums and a max and a sum) per compute unit, or
            # the splits that page ids in LDS ask for
            tiles = -(-tq * (hq // hkv) // 256) * hkv
            assert n <= max(512, -(-ctx // 16384) * tiles) * 256 * (d + 8) * 4
    rng = np.random.default_rng(hq + d)
    tq, L = small
    q, kp, vp, table, L = make_case(rng, hq, hkv, d, tq, L - tq, dtype)
    scale = 1.0 / math.sqrt(d)
    want = oracle_prefill(q, kp, vp, table, L, hq, hkv, d, dtype, scale)
    qd, kd, vd, td = to_dev(q, dtype), to_dev(kp, dtype), to_dev(vp, dtype), to_dev(table)
    for n in (size, size // 8, 0):
        ws = torch.empty(max(n, 16), dtype=torch.uint8, device=DEV)
        out = torch.empty_like(qd)
        kv.prefill_attn(qd, kd, vd, td, L, tq, out, hq, hkv, d, len(table), kp.shape[0], scale,
                        dtype, ws, n)
        torch.cuda.synchronize()
        check(f"prefill workspace {n}", as_f32(to_host(out), dtype), want, dtype)


def test_prefill_long_context_needs_its_workspace(kv):
    """Over 16384 keys must be split: a workspace too small for that is refused."""
    d = torch.zeros(64, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(kv.RlseError) as e:
        kv.prefill_attn(d, d, d, torch.zeros(1025, dtype=torch.int32, device=DEV), 16390, 1, d, 4,
                        1, 128, 1025, 1, 0.1, "bf16", d, d.numel() * 2)
    assert e.value.status == kv.ERR_BUFFER_TOO_SMALL


def test_prefill_captured_before_any_workspace_exists(kv, tmp_path, monkeypatch):
    """A chunk short enough to run unsplit can be captured with the
    library-owned workspace although nothing has allocated one yet (a copy of
    the library has its own); every replay gives the eager result's values."""
    lib = tmp_path / "librlse_kv_copy.so"
    shutil.copy(kv.LIB_PATH, lib)
    monkeypatch.setenv("RLSE_KV_LIB", str(lib))
    spec = importlib.util.spec_from_file_location("rlse_kv_copy", kv.__file__)
    fresh = importlib.util.module_from_spec(spec)
    monkeypatch.setitem(sys.modules, "rlse_kv_copy", fresh)
    spec.loader.exec_module(fresh)
    rng = np.random.default_rng(3)
    hq, hkv, d, tq, dtype = 16, 8, 128, 20, "f32"
    q, kp, vp, table, L = make_case(rng, hq, hkv, d, tq, 400, dtype)
    scale = 1.0 / math.sqrt(d)
    qd, kd, vd, td = to_dev(q), to_dev(kp), to_dev(vp), to_dev(table)
    out = torch.empty_like(qd)

    def call():
        fresh.prefill_attn(qd, kd, vd, td, L, tq, out, hq, hkv, d, len(table), kp.shape[0], scale,
                           dtype, stream=torch.cuda.current_stream())

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    want = oracle_prefill(q, kp, vp, table, L, hq, hkv, d, dtype, scale)
    for _ in range(3):
        out.fill_(7)
        graph.replay()
        torch.cuda.synchronize()
        check("captured", to_host(out), want, dtype)
        call()  # eager: allocates
        torch.cuda.synchronize()
        check("eager", to_host(out), want, dtype)
