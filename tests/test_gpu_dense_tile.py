"""The fused projections over more rows than a decode batch (prompts), and the
norm + projection calls.

Reference: the q/k/v, o, gate/up and down projections of the prefill branch
(src/backends/qwen2.rs:153-175, 233-252). Shapes put the output on each tile
size and on its edges: one row past a 16-row tile, features that end inside a
tile, one, an odd number and an even number of 32-element k steps. The bar is
one rounding of the dtype at the result's magnitude: the products are
accumulated in f32, so a sum in another order moves a result by at most a
neighbouring value, and each further rounding (the residual sum, silu's) by
one more.
"""
import numpy as np
import pytest
import torch

import oracle as O
from gpu_helpers import DEV

pytestmark = pytest.mark.gpu

_T = {"bf16": torch.bfloat16, "f16": torch.float16}
ULP = {"bf16": 2.0 ** -7, "f16": 2.0 ** -10}
# rows, hidden (K of q/k/v and gate/up), q features, kv features, inter
SHAPES = [(65, 32, 32, 16, 32),        # 32 x 32 tiles, one k step
          (81, 96, 64, 16, 32),        # three k steps
          (129, 896, 896, 128, 1024),  # 64 x 64 tiles, q/k/v ends inside one
          (337, 1024, 2048, 1024, 3104),  # 128 x 64 tiles, K 3104: 97 k steps
          (97, 3072, 512, 256, 64)]    # a long K: row tiles per workgroup row


def _dev(a, dt):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(DEV).to(_T[dt])


def _pack_rows(x):
    """[rows][K] -> packed rows, whole 16-row tiles."""
    n, k = x.shape
    full = np.zeros(((n + 15) // 16 * 16, k), np.float32)
    full[:n] = x
    return full.reshape(-1, 16, k // 32, 4, 8).transpose(0, 2, 3, 1, 4).reshape(full.shape)


def _unpack_rows(x, n):
    t, k = x.shape
    return x.reshape(t // 16, k // 32, 4, 16, 8).transpose(0, 3, 1, 2, 4).reshape(t, k)[:n]


def _close(name, got, want, dt, roundings):
    torch.cuda.synchronize()
    got = got.float().cpu().numpy() if isinstance(got, torch.Tensor) else got
    scale = np.maximum(np.abs(want), np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    worst = float((np.abs(got - want) / (ULP[dt] * scale)).max())
    print(f"[{name}] dtype={dt} worst {worst:.2f} of {roundings} ulps")
    assert np.isfinite(got).all() and worst <= roundings, (name, worst)


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("rows,hidden,nq,nkv,inter", SHAPES)
def test_prompt_projections_match_oracle(kv, dt, packed, rows, hidden, nq, nkv, inter):
    rng = np.random.default_rng(rows + hidden)
    r = lambda *s: O.round_to(rng.standard_normal(s) / np.sqrt(s[-1]), dt)  # noqa: E731
    tiles = (rows + 15) // 16 * 16
    x = O.round_to(rng.standard_normal((rows, hidden)), dt)

    def weight(w, pair=0):
        w = _dev(w, dt)
        if not packed:
            return w
        out = torch.empty_like(w)
        kv.dense_pack(w, out, w.shape[0], w.shape[1], pair, dt)
        return out

    def ws(n_out, n_in):
        n = kv.dense_workspace_size(rows, n_out, n_in)
        return torch.zeros(max(n, 4), dtype=torch.uint8, device=DEV)

    xd = _dev(_pack_rows(x) if packed else x, dt)
    # guard rows past the outputs stay untouched
    z = lambda n, extra=3: torch.full((rows + extra, n), 7.0, dtype=_T[dt], device=DEV)  # noqa: E731

    wq = [r(n, hidden) for n in (nq, nkv, nkv)]
    bq = [O.round_to(rng.standard_normal(n), dt) for n in (nq, nkv, nkv)]
    outs = [z(n) for n in (nq, nkv, nkv)]
    kv.qkv_proj(xd, weight(np.concatenate(wq)), _dev(np.concatenate(bq), dt), *outs, rows, hidden,
                nq, nkv, dt, ws(nq + 2 * nkv, hidden), packed=packed, packed_x=packed)
    for name, o, w, b in zip("qkv", outs, wq, bq):
        _close(f"qkv_proj {name}", o[:rows], O.linear_ref(x, w, b, dt), dt, 2)
        assert bool((o[rows:] == 7).all())

    wg, wu = r(inter, hidden), r(inter, hidden)
    act = torch.zeros((tiles, inter), dtype=_T[dt], device=DEV)
    kv.gate_up_silu(xd, weight(np.concatenate([wg, wu]), inter), act, rows, hidden, inter, dt,
                    ws(2 * inter, hidden), packed=packed, packed_x=packed, packed_out=packed)
    want = O.silu_mul_ref(O.linear_ref(x, wg, None, dt), O.linear_ref(x, wu, None, dt), dt)
    got = act.float().cpu().numpy()
    # gate, up, exp, sum, quotient and product each round once
    _close("gate_up_silu", _unpack_rows(got, rows) if packed else got[:rows], want, dt, 6)

    if hidden % 16 == 0:
        a = O.round_to(rng.standard_normal((rows, inter)), dt)
        wd, res = r(hidden, inter), O.round_to(rng.standard_normal((rows, hidden)), dt)
        y = z(hidden)
        y[:rows] = _dev(res, dt)
        kv.linear_residual(_dev(_pack_rows(a) if packed else a, dt), weight(wd), y, rows, hidden,
                           inter, dt, ws(hidden, inter), packed=packed, packed_x=packed)
        want = O.round_to(res + O.linear_ref(a, wd, None, dt), dt)
        _close("linear_residual", y[:rows], want, dt, 2)
        assert bool((y[rows:] == 7).all())


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("rows,hidden,nq,nkv,inter", [
    (1, 896, 896, 128, 4864),    # the norm in both launches (q/k/v: 16 waves, 2 k steps each)
    (16, 1024, 2048, 1024, 3072),  # 8 k steps a wave
    (7, 992, 4096, 32, 4096),    # 31 k steps; gate/up two tiles a workgroup
    (9, 32, 4096, 16, 2048),     # one k step: waves without any
    (5, 1056, 4096, 16, 2048),   # 33 k steps: the norm as a launch of its own
    (17, 1024, 2048, 1024, 3072),  # past its row count
    (70, 96, 64, 16, 64),        # a prompt
    (2, 8224, 64, 16, 32)])      # rows longer than the register-held norm's
def test_norm_projections_match_two_calls(kv, dt, packed, rows, hidden, nq, nkv, inter):
    """norm_qkv_proj and norm_gate_up_silu against add_rmsnorm and the
    projection: the sum of squares may run in another order (one unit in the
    last place of a few h elements, far below the result's rounding); an
    infinite row gives NaN either way, a huge one (its sum overflows) the
    projection of zeros, and the residual is left alone."""
    rng = np.random.default_rng(rows + hidden)
    r = lambda *s: O.round_to(rng.standard_normal(s) / np.sqrt(s[-1]), dt)  # noqa: E731
    tiles = (rows + 15) // 16 * 16
    x = _dev(O.round_to(3 * rng.standard_normal((rows, hidden)), dt), dt)
    if rows > 4:
        x[2] = 0
        x[3, 5] = float("inf")
        x[4] = 3.0e38 if dt == "bf16" else 6.0e4
    nw = _dev(O.round_to(1 + 0.1 * rng.standard_normal(hidden), dt), dt)
    z = lambda n: torch.zeros((tiles, n), dtype=_T[dt], device=DEV)  # noqa: E731

    def weight(w, pair=0):
        w = _dev(w, dt)
        if not packed:
            return w
        out = torch.empty_like(w)
        kv.dense_pack(w, out, w.shape[0], w.shape[1], pair, dt)
        return out

    def ws(n_out):
        n = kv.dense_workspace_size(rows, n_out, hidden)
        return torch.zeros(max(n, 4), dtype=torch.uint8, device=DEV)

    w, wg = weight(r(nq + 2 * nkv, hidden)), weight(r(2 * inter, hidden), inter)
    b = _dev(O.round_to(rng.standard_normal(nq + 2 * nkv), dt), dt)
    keep, h = x.clone(), z(hidden)
    kv.add_rmsnorm(None, x, nw, h, rows, hidden, 1e-6, dt)
    want = [z(n)[:rows] for n in (nq, nkv, nkv)] + [z(inter)]
    kv.qkv_proj(h, w, b, *want[:3], rows, hidden, nq, nkv, dt, ws(nq + 2 * nkv), packed=packed)
    kv.gate_up_silu(h, wg, want[3], rows, hidden, inter, dt, ws(2 * inter), packed=packed)
    got = [z(n)[:rows] for n in (nq, nkv, nkv)] + [z(inter)]
    kv.norm_qkv_proj(x, nw, 1e-6, z(hidden), w, b, *got[:3], rows, hidden, nq, nkv, dt,
                     ws(nq + 2 * nkv), packed=packed)
    kv.norm_gate_up_silu(x, nw, 1e-6, z(hidden), wg, got[3], rows, hidden, inter, dt,
                         ws(2 * inter), packed=packed)
    torch.cuda.synchronize()
    assert torch.equal(x, keep)
    for name, a, c, n in zip(("q", "k", "v", "act"), got, want, (2, 2, 2, 6)):
        a, c = a[:rows].float().cpu().numpy(), c[:rows].float().cpu().numpy()
        np.testing.assert_array_equal(np.isnan(a), np.isnan(c))
        ok = ~np.isnan(c).any(1)
        _close(name, a[ok], c[ok], dt, n)


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("kind,rows,n,k", [
    ("qkv", 333, 4096, 1024),       # one slice of K: 64 x 64 tiles
    ("qkv", 700, 4096, 992),        # 128 x 64 tiles, segments of 8, 8, 8 and 7 k steps
    ("gate_up", 70, 8192, 32),      # one k step: the second half of K is empty
    ("gate_up", 129, 8192, 160),    # 5 k steps in segments of 2
    ("residual", 200, 2048, 1056),  # two slices
    ("qkv", 97, 1536, 1056),        # three, of 11 k steps
    ("residual", 300, 1024, 2048),  # four
    ("residual", 800, 3584, 544),   # two, 128 x 64 tiles
    ("residual", 90, 1024, 3072),   # four, few tiles
    ("gate_up", 130, 640, 1024),    # seven, 32 x 32 tiles
    ("gate_up", 150, 512, 1056)])   # eight
@pytest.mark.parametrize("workspace", [True, False])
def test_prompt_rows_have_the_bits_of_smaller_calls(kv, dt, kind, rows, n, k, workspace):
    """Every row of a prompt's projections is, bit for bit, what a call of at
    most 64 rows gives it (one token's K and V do not depend on the length of
    the chunk it came in), with and without a K split, packed or not."""
    g = torch.Generator(device=DEV).manual_seed(rows + n)
    rnd = lambda *s: torch.randn(s, generator=g, device=DEV).to(_T[dt])  # noqa: E731
    w, bias, res = rnd(n, k), rnd(n), rnd(rows, n)
    x = rnd(rows, k)
    n2 = 128 if n <= 1536 else 1024
    packed = torch.empty_like(w)
    kv.dense_pack(w, packed, n, k, n // 2 if kind == "gate_up" else 0, dt)
    tiles = (rows + 15) // 16 * 16
    px = torch.zeros((tiles, k), dtype=_T[dt], device=DEV)
    px[:rows] = x
    px = px.reshape(-1, 16, k // 32, 4, 8).permute(0, 2, 3, 1, 4).contiguous().reshape(tiles, k)

    def call(x, res, r, w, packed, packed_x):
        ws = torch.zeros(max(kv.dense_workspace_size(r, n, k), 8), dtype=torch.uint8, device=DEV)
        ws = ws if workspace else None
        flags = {"packed": packed, "packed_x": packed_x}
        if kind == "qkv":
            outs = [torch.empty((r, c), dtype=_T[dt], device=DEV) for c in (n - 2 * n2, n2, n2)]
            kv.qkv_proj(x, w, bias, *outs, r, k, n - 2 * n2, n2, dt, ws, **flags)
        elif kind == "residual":
            outs = [res.clone()]
            kv.linear_residual(x, w, outs[0], r, n, k, dt, ws, **flags)
        else:
            outs = [torch.empty((r, n // 2), dtype=_T[dt], device=DEV)]
            kv.gate_up_silu(x, w, outs[0], r, k, n // 2, dt, ws, **flags)
        return outs

    chunks = [call(x[i:i + 64], res[i:i + 64], min(64, rows - i), w, False, False)
              for i in range(0, rows, 64)]
    want = [torch.cat(c) for c in zip(*chunks)]
    for got in (call(x, res, rows, w, False, False), call(px, res, rows, packed, True, True)):
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("eps", [1e-6, 0.0])
@pytest.mark.parametrize("hidden,nq,nkv,inter", [
    (896, 896, 128, 4864),     # q/k/v: 16 waves, 2 k steps each; gate/up: two tiles a workgroup
    (1024, 2048, 1024, 3072),  # 8 k steps a wave
    (544, 4096, 32, 2048),     # 17 k steps: one past the first tree of 16
    (32, 4096, 16, 2048),      # one
    (1056, 4096, 16, 2048)])   # 33: the norm as a launch of its own at any row count
def test_norm_projections_have_the_two_calls_bits(kv, dt, eps, hidden, nq, nkv, inter):
    """norm_qkv_proj and norm_gate_up_silu give add_rmsnorm's and the
    projection's bits, so a row's do not depend on whether its call norms in the
    projection's launch (up to 16 rows) or before it: ordinary rows, rows with
    elements far below the rest, rows whose squares underflow (with eps 0 the
    division is by zero: infinities and NaN, not one for the other) or
    overflow, and zeros."""
    g = torch.Generator(device=DEV).manual_seed(hidden + nq)
    rnd = lambda *s: torch.randn(s, generator=g, device=DEV)  # noqa: E731
    x = 3 * rnd(33, hidden)
    small = 1e-30 if dt == "bf16" else 6e-8
    x[1] *= small
    x[2, ::3] = small
    x[3] = 0
    x[4, 5 % hidden] = float("inf")
    x[5] = 3.0e38 if dt == "bf16" else 6.0e4
    x[6, ::2] *= 1e-38
    x[7] *= 1e-20
    x[8, 7] = float("nan")
    x[9] = x[9].abs() * small  # with w[0] positive: an infinite product, not NaN
    x = x.to(_T[dt])
    nw = (1 + 0.1 * rnd(hidden)).to(_T[dt])
    w, b = rnd(nq + 2 * nkv, hidden).to(_T[dt]), rnd(nq + 2 * nkv).to(_T[dt])
    w[0] = w[0].abs() + 0.01
    wg = rnd(2 * inter, hidden).to(_T[dt])

    def call(lo, rows, fused):
        xr, pad = x[lo:lo + rows].contiguous(), (rows + 15) // 16 * 16
        h = torch.zeros((pad, hidden), dtype=_T[dt], device=DEV)
        outs = [torch.zeros((rows, n), dtype=_T[dt], device=DEV) for n in (nq, nkv, nkv, inter)]
        ws = [torch.zeros(max(kv.dense_workspace_size(rows, n, hidden), 8), dtype=torch.uint8,
                          device=DEV) for n in (nq + 2 * nkv, 2 * inter)]
        if fused:
            kv.norm_qkv_proj(xr, nw, eps, h, w, b, *outs[:3], rows, hidden, nq, nkv, dt, ws[0])
            kv.norm_gate_up_silu(xr, nw, eps, h, wg, outs[3], rows, hidden, inter, dt, ws[1])
        else:
            kv.add_rmsnorm(None, xr, nw, h, rows, hidden, eps, dt)
            kv.qkv_proj(h, w, b, *outs[:3], rows, hidden, nq, nkv, dt, ws[0])
            kv.gate_up_silu(h, wg, outs[3], rows, hidden, inter, dt, ws[1])
        torch.cuda.synchronize()
        return outs

    want = call(0, 33, False)
    for lo, rows in ((0, 1), (0, 7), (0, 16), (1, 16), (5, 1), (20, 13), (0, 17), (0, 33)):
        for a, c in zip(call(lo, rows, True), want):
            c = c[lo:lo + rows]
            ok = ~c.isnan()
            assert torch.equal(~a.isnan(), ok), (lo, rows)
            assert torch.equal(a.view(torch.int16)[ok], c.view(torch.int16)[ok]), (lo, rows)


def test_more_rows_than_a_grid_holds(kv):
    """2^23 row tiles of 512 threads pass the 2^32 threads of a grid: the rows
    before, at and after that point, and the last, are those of small calls."""
    rows, n, k, dt = (1 << 29) + 1000, 16, 32, "bf16"
    g = torch.Generator(device=DEV).manual_seed(1)
    w = torch.randn((n, k), generator=g, device=DEV).to(_T[dt])
    x = torch.zeros((rows, k), dtype=_T[dt], device=DEV)
    y = torch.zeros((rows, n), dtype=_T[dt], device=DEV)
    spans = [(0, 300), ((1 << 29) - 1024, (1 << 29) + 300), (rows - 100, rows)]
    for a, b in spans:
        x[a:b] = torch.randn((b - a, k), generator=g, device=DEV).to(_T[dt])
    kv.linear_residual(x, w, y, rows, n, k, dt)
    for a, b in spans:
        want = torch.zeros((b - a, n), dtype=_T[dt], device=DEV)
        kv.linear_residual(x[a:b], w, want, b - a, n, k, dt)
        torch.cuda.synchronize()
        assert torch.equal(y[a:b], want) and bool(want.any(1).all())
    del x, y
    torch.cuda.empty_cache()
