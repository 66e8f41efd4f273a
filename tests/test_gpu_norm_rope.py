"""RMSNorm, RoPE and the fused q/k-norm + RoPE + append on the GPU.

Reference: RmsNorm::forward (src/backends/qwen2.rs:68-75), RotaryEmbedding and
apply_rope (:84-142), Attention::forward's norm -> transpose -> RoPE -> append
order (:291-313). RoPE uses the same host-built tables as the oracle, and the
kernels round at the same points as Candle; the sum of squares of RMSNorm
follows the oracle's fixed order (orc_sumsq_tree), so RMSNorm, RoPE and the
fused q/k-norm + RoPE + append are all checked bit for bit. The case matrix
rows {1, 4, 17, 64} x n {128, 1024} is the reference harness's
(scripts/validate_cuda_kernels.py:132-160).
"""
import numpy as np
import pytest
import torch

import oracle as O
from gpu_helpers import DEV, as_f32, build_tables, random_values, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("rows", [1, 4, 17, 64])
@pytest.mark.parametrize("n", [128, 1024, 100, 896, 8192])
def test_rmsnorm_matrix(kv, dtype, rows, n):
    rng = np.random.default_rng(rows * 7 + n)
    x = random_values(rng, (rows, n), dtype)
    w = random_values(rng, (n,), dtype)
    out = torch.empty((rows, n), dtype=to_dev(x, dtype).dtype, device=DEV)
    kv.rmsnorm(to_dev(x, dtype), to_dev(w, dtype), out, rows, n, 1e-6, dtype)
    got = to_host(out)
    if dtype == "bf16":
        want = O.rmsnorm_bf16(x, w, 1e-6)
    elif dtype == "f16":
        want = O.rmsnorm_f16(x, w, 1e-6)
    else:
        want = O.rmsnorm_f32(x, w, 1e-6)
    np.testing.assert_array_equal(got, want)
    # the reference harness's bar (validate_cuda_kernels.py:126-129)
    atol, rtol = (1e-5, 1e-4) if dtype == "f32" else (5e-3, 5e-3)
    ref = O.rmsnorm_f64(as_f32(x, dtype), as_f32(w, dtype), 1e-6)
    assert np.all(np.abs(as_f32(got, dtype) - ref) <= atol + rtol * np.abs(ref) +
                  (0 if dtype == "f32" else 2.0 ** -7 * np.abs(ref)))


def test_prototype_rmsnorm_launchers(kv):
    rng = np.random.default_rng(5)
    x = rng.standard_normal((4, 1024)).astype(np.float32)
    w = rng.standard_normal(1024).astype(np.float32)
    a = torch.empty((4, 1024), dtype=torch.float32, device=DEV)
    xd, wd = to_dev(x), to_dev(w)  # keep the buffers alive until the kernel ran
    assert kv.load().launch_rmsnorm_f32(xd.data_ptr(), wd.data_ptr(), a.data_ptr(), 4, 1024,
                                        1e-6) == 0
    np.testing.assert_array_equal(to_host(a), O.rmsnorm_f32(x, w, 1e-6))
    xb, wb = O.f32_to_bf16_bits(x), O.f32_to_bf16_bits(w)
    b = torch.empty((4, 1024), dtype=torch.bfloat16, device=DEV)
    xbd, wbd = to_dev(xb, "bf16"), to_dev(wb, "bf16")
    assert kv.load().launch_rmsnorm_bf16(xbd.data_ptr(), wbd.data_ptr(), b.data_ptr(), 4, 1024,
                                         1e-6) == 0
    np.testing.assert_array_equal(to_host(b), O.rmsnorm_bf16(xb, wb, 1e-6))


def _tables(kv, theta, d, max_pos, dtype):
    np_dt = {"f32": np.float32, "bf16": np.uint16, "f16": np.float16}[dtype]
    cb, sb = kv.rope_tables(theta, d, max_pos, dtype)
    c = np.frombuffer(cb, np_dt).reshape(max_pos, d // 2).copy()
    s = np.frombuffer(sb, np_dt).reshape(max_pos, d // 2).copy()
    return c, s


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("d", [64, 128])
def test_rope_bit_exact(kv, dtype, d):
    rng = np.random.default_rng(d)
    ntok, hq, hkv, theta, max_pos = 6, 16, 8, 1e6, 4096
    c, s = _tables(kv, theta, d, max_pos, dtype)
    q = random_values(rng, (ntok, hq, d), dtype)
    k = random_values(rng, (ntok, hkv, d), dtype)
    pos = np.array([0, 1, 17, 512, 2047, 4095], np.int32)
    qd, kd = to_dev(q, dtype), to_dev(k, dtype)
    kv.rope(qd, kd, to_dev(c, dtype), to_dev(s, dtype), to_dev(pos), ntok, hq, hkv, d, max_pos,
            dtype)
    for x, dev, h in ((q, qd, hq), (k, kd, hkv)):
        rows = x.reshape(ntok * h, d)
        rpos = np.repeat(pos, h)
        if dtype == "bf16":
            want = O.apply_rope_bf16(rows, rpos, c, s)
        else:
            want = O.apply_rope_f32(rows, rpos, c, s)
        np.testing.assert_array_equal(to_host(dev).reshape(ntok * h, d), want)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_qk_norm_rope_append_matches_reference_order(kv, dtype):
    rng = np.random.default_rng(21)
    b, hq, hkv, d, eps, theta = 5, 16, 8, 128, 1e-6, 1e6
    pos = np.array([0, 15, 16, 200, 511], np.int32)
    nb, mbps = 64, 32
    tables = build_tables(rng, pos + 1, nb, mbps)
    q = random_values(rng, (b, hq, d), dtype)
    k = random_values(rng, (b, hkv, d), dtype)
    v = random_values(rng, (b, hkv, d), dtype)
    qw = O.f32_to_bf16_bits(1 + 0.1 * rng.standard_normal(d)) if dtype == "bf16" else \
        (1 + 0.1 * rng.standard_normal(d)).astype(np.float32)
    kw = O.f32_to_bf16_bits(1 + 0.1 * rng.standard_normal(d)) if dtype == "bf16" else \
        (1 + 0.1 * rng.standard_normal(d)).astype(np.float32)
    c, s = _tables(kv, theta, d, 600, dtype)
    tdt = {"bf16": torch.bfloat16, "f32": torch.float32}[dtype]
    kp = torch.zeros((nb, hkv, 16, d), dtype=tdt, device=DEV)
    vp = torch.zeros_like(kp)
    q_out = torch.empty((b, hq, d), dtype=tdt, device=DEV)
    kv.qk_norm_rope_append(to_dev(q, dtype), to_dev(k, dtype), to_dev(v, dtype), to_dev(qw, dtype),
                           to_dev(kw, dtype), eps, to_dev(c, dtype), to_dev(s, dtype), 600,
                           to_dev(pos), to_dev(tables), b, None, b, hq, hkv, d, mbps, nb, q_out,
                           kp, vp, dtype)
    norm = O.rmsnorm_bf16 if dtype == "bf16" else O.rmsnorm_f32
    rope = O.apply_rope_bf16 if dtype == "bf16" else O.apply_rope_f32
    q_ref = rope(norm(q.reshape(-1, d), qw, eps), np.repeat(pos, hq), c, s).reshape(b, hq, d)
    k_ref = rope(norm(k.reshape(-1, d), kw, eps), np.repeat(pos, hkv), c, s).reshape(b, hkv, d)
    np.testing.assert_array_equal(to_host(q_out), q_ref)
    pool_k, pool_v = to_host(kp), to_host(vp)
    for i in range(b):
        blk, slot = tables[i, pos[i] // 16], pos[i] % 16
        np.testing.assert_array_equal(pool_k[blk, :, slot], k_ref[i])
        np.testing.assert_array_equal(pool_v[blk, :, slot], v[i])  # V is appended raw


def test_qwen2_path_without_qk_norm(kv):
    """Qwen2 has no q_norm/k_norm (qwen2.rs:251-260): null weights skip the norm,
    and the result equals plain RoPE + append."""
    rng = np.random.default_rng(22)
    b, hq, hkv, d, dtype = 3, 14, 2, 64, "bf16"
    pos = np.array([3, 40, 100], np.int32)
    nb, mbps = 16, 8
    tables = build_tables(rng, pos + 1, nb, mbps)
    q, k, v = (random_values(rng, (b, h, d), dtype) for h in (hq, hkv, hkv))
    c, s = _tables(kv, 1e6, d, 128, dtype)
    kp = torch.zeros((nb, hkv, 16, d), dtype=torch.bfloat16, device=DEV)
    vp = torch.zeros_like(kp)
    q_out = torch.empty((b, hq, d), dtype=torch.bfloat16, device=DEV)
    kv.qk_norm_rope_append(to_dev(q, dtype), to_dev(k, dtype), to_dev(v, dtype), None, None, 1e-6,
                           to_dev(c, dtype), to_dev(s, dtype), 128, to_dev(pos), to_dev(tables), b,
                           None, b, hq, hkv, d, mbps, nb, q_out, kp, vp, dtype)
    np.testing.assert_array_equal(
        to_host(q_out), O.apply_rope_bf16(q.reshape(-1, d), np.repeat(pos, hq), c, s)
        .reshape(b, hq, d))
    k_ref = O.apply_rope_bf16(k.reshape(-1, d), np.repeat(pos, hkv), c, s).reshape(b, hkv, d)
    pool_k = to_host(kp)
    for i in range(b):
        np.testing.assert_array_equal(pool_k[tables[i, pos[i] // 16], :, pos[i] % 16], k_ref[i])


@pytest.mark.parametrize("dtype", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("hq,hkv,d", [(7, 1, 64), (4, 2, 128), (3, 3, 32), (2, 1, 256)])
@pytest.mark.parametrize("norm", [True, False])
def test_qk_norm_rope_append_packet_rows_give_the_element_bits(kv, dtype, hq, hkv, d, norm):
    """Aligned rows of whole packets (several rows a wave) and the same rows
    one element into their buffers (a wave a row, element accesses) leave the
    same bits: q, the appended K and V, and nothing where a position, page id
    or sequence is invalid. NaN, infinities, zeros and subnormals included."""
    g = torch.Generator(device=DEV).manual_seed(d + hq)
    tdt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[dtype]
    n, nb, mbps, max_pos = 37, 15, 5, 70
    rnd = lambda *s: torch.randn(s, generator=g, device=DEV).to(tdt)  # noqa: E731
    q, k, v = rnd(n, hq, d), rnd(n, hkv, d), rnd(n, hkv, d)
    q[1, 0, 3], q[2, 0, d - 1], k[3, 0, 0], k[4, 0, 1] = float("inf"), float("nan"), -0.0, 1e-7
    q[5], k[6] = 0.0, 3.0e4
    w = [1 + 0.1 * rnd(d), 1 + 0.1 * rnd(d)] if norm else [None, None]
    cos, sin = rnd(max_pos, d // 2), rnd(max_pos, d // 2)
    pos = torch.arange(n, dtype=torch.int32, device=DEV)
    pos[7], pos[8] = -1, max_pos
    seq = (pos % 3).to(torch.int32)
    seq[10], seq[11] = 3, -1
    tables = torch.randperm(nb, generator=g, device=DEV).to(torch.int32).view(3, 5)
    tables[0, 1], tables[1, 0] = nb, -1

    def shifted(t, by):
        buf = torch.full((t.numel() + 8,), 5.0, dtype=tdt, device=DEV)
        out = buf[by:by + t.numel()].view(t.shape)
        out.copy_(t)
        return out

    got = []
    for by in (0, 1):
        a = [None if t is None else shifted(t, by) for t in (q, k, v, *w, cos, sin)]
        q_out, kp, vp = (shifted(torch.full(s, 9.0, dtype=tdt, device=DEV), by)
                         for s in ((n, hq, d), (nb, hkv, 16, d), (nb, hkv, 16, d)))
        kv.qk_norm_rope_append(*a[:5], 1e-6, *a[5:], max_pos, pos, tables, 3, seq, n, hq, hkv, d,
                               mbps, nb, q_out, kp, vp, dtype)
        torch.cuda.synchronize()
        got.append([t.contiguous().view(torch.int32 if dtype == "f32" else torch.int16).cpu()
                    for t in (q_out, kp, vp)])
    for x, y in zip(*got):
        assert torch.equal(x, y)


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_conversion_instruction_rounds_to_nearest_even(kv, dtype):
    """Roundings through the conversion instruction (the projections'
    epilogues, the norms, the q/k norm + RoPE) against the integer sequence: a
    product whose f32 results are a 16-bit value plus each of the 2^16 lower
    significands. Signs, exponents to the overflow and (f16) subnormal edges."""
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float16
    # x = [hi, 2^e, 2^e'] against w = [1, low / 256, low % 256]: sums of at most 24 significant
    # bits, exact in f32 in any order.
    low = torch.arange(1 << 16, device=DEV)
    w = torch.zeros((1 << 16, 32), device=DEV)
    w[:, 0], w[:, 1], w[:, 2] = 1, low // 256, low % 256
    exps = (range(-100, 128, 9) if dtype == "bf16" else range(-18, 16))
    rows = [(s * (1 + m / 128), e) for e in list(exps) + ([127] if dtype == "bf16" else [])
            for m in (0, 1, 2, 63, 64, 127) for s in (1.0, -1.0)]
    x = torch.zeros((len(rows), 32), dtype=torch.float64, device=DEV)
    for i, (m, e) in enumerate(rows):
        sign = 1 if m > 0 else -1
        x[i, 0] = m * 2.0 ** e
        x[i, 1], x[i, 2] = sign * 2.0 ** (e - 15), sign * 2.0 ** (e - 23)
    keep = (x.to(tdt).double() == x).all(1)  # (f16 has no 2^(e - 23) for the smallest)
    assert int(keep.sum()) >= 60
    x = x[keep]
    exact = (x @ w.double().T).float()  # one f32 each
    bits = exact.view(torch.int32)
    if dtype == "bf16":
        want = ((bits + 0x7FFF + ((bits >> 16) & 1)) >> 16).to(torch.int16)
    else:
        want = exact.cpu().half().view(torch.int16).to(DEV)
    out = torch.zeros((x.shape[0], 1 << 16), dtype=tdt, device=DEV)
    kv.linear(x.to(tdt).contiguous(), w.to(tdt), None, out, x.shape[0], 1 << 16, 32, dtype)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), want)
