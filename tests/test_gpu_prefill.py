"""GPU parity of the prefill path: the batched projection (split fp16 operands),
the q/k norm + RoPE + KV-write rows, causal prefill attention, and the chunked
model prefill against token-by-token decode.

Floating-point bound: max |gpu - ref| / max |ref| <= 2e-3 (the north-star
bound), with tighter checks where the arithmetic allows (the GEMM against an
fp64 product: 1e-5).  Token ids are compared exactly.
"""
from __future__ import annotations

import numpy as np
import pytest

from conftest import load_golden, rel_err

pytestmark = pytest.mark.gpu
TOL = 2e-3


def f16_weights(rng, rows, cols, std=0.02):
    w = (rng.standard_normal((rows, cols)) * std).astype(np.float16)
    return w, w.astype(np.float32)


# (batch, rows, cols): MiniMind2 prefill projections at several prompt lengths,
# the lm_head shape, and ragged batches / small shapes (tile edges)
MATMUL_SHAPES = [(1, 1152, 768), (7, 768, 768), (64, 4096, 768), (100, 768, 2048), (512, 1152, 768),
                 (512, 4096, 768), (512, 768, 768), (512, 768, 2048), (33, 100, 64), (65, 6400, 768), (3, 13, 32),
                 (40, 96, 1408), (9, 24, 200)]


@pytest.mark.parametrize("batch,rows,cols", MATMUL_SHAPES)
def test_matmul_matches_fp64_and_oracle(gpu, oracle, batch, rows, cols):
    mmr = gpu
    print(f"[case] matmul {batch}x{rows}x{cols}", flush=True)
    rng = np.random.default_rng(batch * 31 + rows + cols)
    w16, w32 = f16_weights(rng, rows, cols)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    dw, dx = mmr.DeviceArray.from_numpy(w16.view(np.uint16)), mmr.DeviceArray.from_numpy(x)
    dy = mmr.DeviceArray((batch, rows), np.float32)
    mmr.matmul_f16(dw, rows, cols, dx, batch, dy)
    got = dy.numpy()
    exact = x.astype(np.float64) @ w32.astype(np.float64).T
    assert rel_err(got, exact) < 1e-5  # a transposed or misplaced fragment is O(1)
    for b in {0, batch // 2, batch - 1}:  # the reference's sequential fp32 matvec per row
        assert rel_err(got[b], oracle.matvec(w32, x[b])) < TOL
    # residual epilogue (device_matmul_add), residual aliasing the output
    res = rng.standard_normal((batch, rows)).astype(np.float32)
    dr = mmr.DeviceArray.from_numpy(res)
    mmr.matmul_f16(dw, rows, cols, dx, batch, dr, residual=dr)
    assert rel_err(dr.numpy(), res + exact) < 1e-5


@pytest.mark.parametrize("batch,rows,cols,grow", [(1409, 1793, 128, 0), (1536, 2048, 256, 0), (1500, 1800, 1408, 0),
                                                  (1409, 2047, 768, 1), (1409, 2047, 768, -1)])
def test_matmul_many_rows_matches_fp64(gpu, batch, rows, cols, grow):
    # the 128 x 256 tiles (96 of them): a last row tile of 1 row, a last column
    # tile of 1 column, the shortest K, an odd number of 128-column chunks;
    # rows whose values grow or shrink by 2^60 along K (a scale per 64 columns),
    # every row by another offset.  Against 64 bits, each row over its own
    # scale: the planes hold 22 bits of the row's largest values (2.4e-7), the
    # sums are fp32 over at most 1,408 products of like size (40 ulp at most).
    mmr = gpu
    print(f"[case] matmul many rows {batch}x{rows}x{cols} grow={grow}", flush=True)
    rng = np.random.default_rng(batch + rows + cols)
    w16, w32 = f16_weights(rng, rows, cols)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    if grow:
        x *= np.exp2(np.linspace(-30, 30, cols) * grow + rng.integers(-9, 9, (batch, 1))).astype(np.float32)
    x[7] = 0.0
    dw, dx = mmr.DeviceArray.from_numpy(w16.view(np.uint16)), mmr.DeviceArray.from_numpy(x)
    dy = mmr.DeviceArray((batch, rows), np.float32)
    mmr.matmul_f16(dw, rows, cols, dx, batch, dy)
    got = dy.numpy().astype(np.float64)
    exact = x.astype(np.float64) @ w32.astype(np.float64).T
    scale = np.maximum(np.abs(exact).max(axis=1, keepdims=True), 1e-30)
    assert np.max(np.abs(got - exact) / scale) < 1e-5
    assert not got[7].any()
    if not grow:
        res = rng.standard_normal((batch, rows)).astype(np.float32)
        dr = mmr.DeviceArray.from_numpy(res)
        mmr.matmul_f16(dw, rows, cols, dx, batch, dr, residual=dr)
        assert rel_err(dr.numpy(), res + exact) < 1e-5


@pytest.mark.parametrize("batch,rows,cols", [(100, 1152, 768), (1536, 2048, 768), (70, 24576, 384)])
def test_matmul_keeps_small_columns_beside_large_ones(gpu, batch, rows, cols):
    # columns 2^30 times the others' size in a chunk of 128 that no weight
    # reads: x is split under a scale per 128 columns or fewer, so the result
    # keeps its bits (the 64 x 64 tiles, then the many-rows ones)
    mmr = gpu
    print(f"[case] matmul beside large columns {batch}x{rows}x{cols}", flush=True)
    rng = np.random.default_rng(batch)
    w16, _ = f16_weights(rng, rows, cols)
    w16[:, 128:256] = 0
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    dw, dy = mmr.DeviceArray.from_numpy(w16.view(np.uint16)), mmr.DeviceArray((batch, rows), np.float32)
    out = []
    for size in (1.0, 2.0**30):
        x[:, 128:256] *= np.float32(size)
        mmr.matmul_f16(dw, rows, cols, mmr.DeviceArray.from_numpy(x), batch, dy)
        out.append(dy.numpy())
    np.testing.assert_array_equal(out[0], out[1])


@pytest.mark.parametrize("batch", [16, 17, 32, 33, 64, 65])
def test_matmul_few_rows_wide_output_matches_fp64(gpu, batch):
    # 160 tiles of 128 x 256 with few of their rows: the edges between the
    # few-rows kernel, the 64-row tiles and the many-rows ones
    mmr = gpu
    rows, cols = 40960, 256
    print(f"[case] matmul wide {batch}x{rows}x{cols}", flush=True)
    rng = np.random.default_rng(batch)
    w16, w32 = f16_weights(rng, rows, cols)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    dw, dx = mmr.DeviceArray.from_numpy(w16.view(np.uint16)), mmr.DeviceArray.from_numpy(x)
    dy = mmr.DeviceArray((batch, rows), np.float32)
    mmr.matmul_f16(dw, rows, cols, dx, batch, dy)
    assert rel_err(dy.numpy(), x.astype(np.float64) @ w32.astype(np.float64).T) < 1e-5


def test_matmul_rejects_bad_shapes(gpu):
    mmr = gpu
    d = mmr.DeviceArray(64, np.float32)
    with pytest.raises(mmr.InvalidArgument, match="multiple of 8"):
        mmr.check(mmr.lib().mmr_matmul_f16(d.ptr, 4, 44, d.ptr, 1, None, d.ptr, None))
    with pytest.raises(mmr.InvalidArgument, match="positive"):
        mmr.check(mmr.lib().mmr_matmul_f16(d.ptr, 4, 32, d.ptr, 0, None, d.ptr, None))


def cache_layout(rows_ref, tokens, hkv, d, rows):
    """[token][kv_head][d] (reference) -> [kv_head][rows][d] (cache)."""
    out = np.zeros((hkv, rows, d), rows_ref.dtype)
    out[:, :tokens, :] = rows_ref.reshape(tokens, hkv, d).transpose(1, 0, 2)
    return out


@pytest.mark.parametrize("d", [64, 96, 128])
@pytest.mark.parametrize("start", [0, 37])
def test_prefill_qkv_rows_match_per_token_postprocess(gpu, oracle, d, start):
    mmr = gpu
    hq, hkv, eps, theta, T = 8, 2, 1e-5, 1e6, 21
    rng = np.random.default_rng(d + start)
    qkv = rng.standard_normal((T, (hq + 2 * hkv) * d)).astype(np.float32)
    qn = (1 + 0.1 * rng.standard_normal(d)).astype(np.float32)
    kn = (1 + 0.1 * rng.standard_normal(d)).astype(np.float32)
    rope = mmr.RopeTable(1024, d, theta)
    cache = mmr.KvCache(hkv, d, start + T + 5, mmr.KV_F32)
    dqkv, dqn, dkn = (mmr.DeviceArray.from_numpy(a) for a in (qkv, qn, kn))
    query = mmr.DeviceArray((T, hq * d), np.float32)
    mmr.prefill_qkv_rows(dqkv, dqn, dkn, eps, rope, cache, start, T, hq, hkv, d, query)
    q_all, keys = query.numpy(), cache.download()[0]
    vals = cache.download()[1]
    for t in range(T):
        q_ref, k_ref = oracle.qk_norm_rope(qkv[t, : hq * d], qkv[t, hq * d: (hq + hkv) * d], qn, kn, hq, hkv, d,
                                           start + t, eps, theta)
        assert rel_err(q_all[t], q_ref) < 1e-5, t
        assert rel_err(keys[:, start + t, :].reshape(-1), k_ref) < 1e-5, t
        np.testing.assert_array_equal(vals[:, start + t, :].reshape(-1), qkv[t, (hq + hkv) * d:])
    assert not keys[:, :start, :].any() and not keys[:, start + T:, :].any()  # nothing else written


@pytest.mark.parametrize("kv", ["f16", "f32"])
@pytest.mark.parametrize("d", [32, 64, 96, 128])
@pytest.mark.parametrize("start,T", [(0, 1), (0, 16), (0, 17), (0, 100), (70, 33), (130, 64)])
def test_prefill_attention_matches_oracle(gpu, oracle, kv, d, start, T):
    mmr = gpu
    print(f"[case] prefill attention kv={kv} d={d} start={start} T={T}", flush=True)
    hq, hkv = 8, 2
    rng = np.random.default_rng(d * 1000 + start + T)
    np_kv = np.float16 if kv == "f16" else np.float32
    n = start + T
    k = rng.standard_normal(n * hkv * d).astype(np_kv).astype(np.float32)
    v = rng.standard_normal(n * hkv * d).astype(np_kv).astype(np.float32)
    q = rng.standard_normal((T, hq * d)).astype(np.float32)
    cache = mmr.KvCache(hkv, d, n + 3, mmr.KV_F16 if kv == "f16" else mmr.KV_F32)
    cache.upload(cache_layout(k, n, hkv, d, cache.rows), cache_layout(v, n, hkv, d, cache.rows))
    dq, out = mmr.DeviceArray.from_numpy(q), mmr.DeviceArray((T, hq * d), np.float32)
    mmr.prefill_attention(dq, cache, start, T, hq, hkv, d, out)
    got = out.numpy()
    for t in sorted({0, T // 3, T // 2, T - 1}):
        keys = start + t + 1  # causal: keys 0 .. own position
        ref = oracle.attention_step(q[t], k[: keys * hkv * d], v[: keys * hkv * d], keys, hq, hkv, d)
        assert rel_err(got[t], ref) < TOL, t


@pytest.mark.parametrize("hq,hkv", [(8, 1), (4, 4), (6, 2), (16, 2)])
def test_prefill_attention_group_sizes(gpu, oracle, hq, hkv):
    # query heads per KV head R = 8, 1, 3, 8 (the block holds 4 or 8 waves;
    # waves past R only stage K/V)
    mmr = gpu
    print(f"[case] prefill attention hq={hq} hkv={hkv}", flush=True)
    d, start, T = 64, 20, 45
    rng = np.random.default_rng(hq * 10 + hkv)
    n = start + T
    k = rng.standard_normal(n * hkv * d).astype(np.float32)
    v = rng.standard_normal(n * hkv * d).astype(np.float32)
    q = rng.standard_normal((T, hq * d)).astype(np.float32)
    cache = mmr.KvCache(hkv, d, n, mmr.KV_F32)
    cache.upload(cache_layout(k, n, hkv, d, cache.rows), cache_layout(v, n, hkv, d, cache.rows))
    dq, out = mmr.DeviceArray.from_numpy(q), mmr.DeviceArray((T, hq * d), np.float32)
    mmr.prefill_attention(dq, cache, start, T, hq, hkv, d, out)
    got = out.numpy()
    for t in (0, 17, T - 1):
        keys = start + t + 1
        ref = oracle.attention_step(q[t], k[: keys * hkv * d], v[: keys * hkv * d], keys, hq, hkv, d)
        assert rel_err(got[t], ref) < TOL, t


@pytest.mark.parametrize("d", [32, 64, 96, 128])
def test_prefill_attention_few_rows_keep_q_exact(gpu, d):
    # the 16-query kernel over an fp16 cache against 64 bits: q and p carry 22
    # bits, sums are fp32 over at most 300 keys, so 1e-5 of the largest value; a
    # q element whose two planes do not belong together is 1e-4
    mmr = gpu
    hq, hkv, T = 8, 2, 300
    print(f"[case] prefill attention few rows d={d}", flush=True)
    rng = np.random.default_rng(d)
    k = rng.standard_normal((hkv, T, d)).astype(np.float16)
    v = rng.standard_normal((hkv, T, d)).astype(np.float16)
    q = (2 * rng.standard_normal((T, hq, d))).astype(np.float32)
    cache = mmr.KvCache(hkv, d, T, mmr.KV_F16)
    cache.upload(k, v)
    dq, out = mmr.DeviceArray.from_numpy(q.reshape(T, hq * d)), mmr.DeviceArray((T, hq * d), np.float32)
    mmr.prefill_attention(dq, cache, 0, T, hq, hkv, d, out)
    got = out.numpy().reshape(T, hq, d)
    hidden = np.triu(np.ones((T, T), bool), 1)
    for h in range(hq):
        g = h // (hq // hkv)
        s = q[:, h].astype(np.float64) @ k[g].astype(np.float64).T / np.sqrt(d)
        s[hidden] = -np.inf
        p = np.exp(s - s.max(axis=1, keepdims=True))
        ref = p @ v[g].astype(np.float64) / p.sum(axis=1, keepdims=True)
        assert rel_err(got[:, h], ref) < 1e-5, h


@pytest.mark.parametrize("d", [32, 64, 96])
@pytest.mark.parametrize("hq,hkv,start,T", [(16, 2, 0, 449), (16, 2, 37, 480), (8, 2, 1000, 641), (8, 4, 511, 930),
                                            (12, 2, 20, 1300), (16, 2, 0, 993), (16, 2, 37, 992)])
def test_prefill_attention_many_rows(gpu, d, hq, hkv, start, T):
    # the 32-query kernel (the first two cases: the 16-query one): a last query
    # tile of 1, 2, 20, 1 and 32 rows, groups of 4, 2, 6 and 8 heads, key ranges
    # of unequal length, a context that crosses segments.  Against 64 bits:
    # q and p carry 22 bits (2.4e-7), sums are fp32 over at most 1,641 keys of
    # like size (random rounding, some 40 ulp of the sum at most): 1e-5 of the
    # largest value, where one wrong key among 1,641 is about 1e-2.
    mmr = gpu
    print(f"[case] prefill attention many rows d={d} hq={hq} hkv={hkv} start={start} T={T}", flush=True)
    assert mmr.prefill_attention_many_rows(hq, hkv, d, mmr.KV_F16, start, T) or T < 500
    rng = np.random.default_rng(d + hq + start + T)
    n = start + T
    k = rng.standard_normal((hkv, n, d)).astype(np.float16)
    v = rng.standard_normal((hkv, n, d)).astype(np.float16)
    q = (2 * rng.standard_normal((T, hq * d))).astype(np.float32)
    cache = mmr.KvCache(hkv, d, n, mmr.KV_F16)
    cache.upload(k, v)
    dq, out = mmr.DeviceArray.from_numpy(q), mmr.DeviceArray((T, hq * d), np.float32)
    mmr.prefill_attention(dq, cache, start, T, hq, hkv, d, out)
    got = out.numpy().reshape(T, hq, d)
    hidden = np.arange(n)[None, :] > start + np.arange(T)[:, None]
    for h in range(hq):
        g = h // (hq // hkv)
        s = q.reshape(T, hq, d)[:, h].astype(np.float64) @ k[g].astype(np.float64).T / np.sqrt(d)
        s[hidden] = -np.inf
        p = np.exp(s - s.max(axis=1, keepdims=True))
        ref = p @ v[g].astype(np.float64) / p.sum(axis=1, keepdims=True)
        assert rel_err(got[:, h], ref) < 1e-5, h


@pytest.mark.parametrize("d", [64, 96])
@pytest.mark.parametrize("hq,hkv,start,T,spread", [(32, 8, 0, 449, 0), (32, 4, 37, 480, 0), (16, 2, 1000, 993, 8),
                                                   (16, 4, 511, 961, 14)])
def test_prefill_attention_many_rows_f32(gpu, d, hq, hkv, start, T, spread):
    # the 32-query kernel over an fp32 cache: a last query tile of 1, 32, 1 and
    # 1 rows, groups of 4, 8, 8 and 4 heads, a context that crosses segments.
    # With a spread, V grows with the position by 2^spread and falls again, so
    # that the values' running scale moves, and K's rows (and, inversely, the
    # queries) differ in size.  Against 64 bits: K, V, q and p carry 22 bits
    # (2.4e-7 each; a score of size 10 turns two of these into 3.4e-6 of p at
    # most, averaged over the keys) and sums are fp32 over tiles of 32 keys:
    # 2e-6 of the largest value of the row, where one wrong key among 1,993 is
    # about 1e-2.
    mmr = gpu
    print(f"[case] prefill attention many rows f32 d={d} hq={hq} hkv={hkv} start={start} T={T}", flush=True)
    assert mmr.prefill_attention_many_rows(hq, hkv, d, mmr.KV_F32, start, T)
    rng = np.random.default_rng(d + hq + start + T)
    n = start + T
    k = rng.standard_normal((hkv, n, d)).astype(np.float32)
    v = rng.standard_normal((hkv, n, d)).astype(np.float32)
    q = rng.standard_normal((T, hq, d)).astype(np.float32)
    size = 2.0 ** (spread * (1 - np.abs(np.linspace(-1, 1, n))))
    v *= size[None, :, None].astype(np.float32)
    k *= np.float32(2.0**-spread)
    k[:, ::3] *= np.float32(0.25)
    q *= np.float32(2.0**spread)
    cache = mmr.KvCache(hkv, d, n, mmr.KV_F32)
    cache.upload(k, v)
    dq, out = mmr.DeviceArray.from_numpy(q.reshape(T, hq * d)), mmr.DeviceArray((T, hq * d), np.float32)
    mmr.prefill_attention(dq, cache, start, T, hq, hkv, d, out)
    got = out.numpy().reshape(T, hq, d)
    hidden = np.arange(n)[None, :] > start + np.arange(T)[:, None]
    for h in range(hq):
        g = h // (hq // hkv)
        s = q[:, h].astype(np.float64) @ k[g].astype(np.float64).T / np.sqrt(d)
        s[hidden] = -np.inf
        p = np.exp(s - s.max(axis=1, keepdims=True))
        ref = p @ v[g].astype(np.float64) / p.sum(axis=1, keepdims=True)
        err = np.abs(got[:, h] - ref).max(axis=1) / np.abs(ref).max(axis=1)
        assert err.max() < 2e-6, (h, int(err.argmax()), float(err.max()))


@pytest.mark.parametrize("d", [64, 96])
@pytest.mark.parametrize("hq,hkv,start,T", [(16, 4, 0, 993), (8, 2, 1990, 2000)])
def test_prefill_attention_f32_keeps_small_dims(gpu, d, hq, hkv, start, T):
    # V's dims have a scale of their own, per run of d / 4: dims 2^-40 of the
    # others' size come out as the same bits, 2^-40 times; and with dims spread
    # over 2^16 and, in the other half, keys over 2^16, every dim is within 5e-6
    # of its own largest value (22 bits of K, V, q and p; a score of size 10
    # turns two of these into 3.4e-6 of p at most).
    mmr = gpu
    print(f"[case] prefill attention f32 small dims d={d} hq={hq} hkv={hkv} start={start} T={T}", flush=True)
    assert mmr.prefill_attention_many_rows(hq, hkv, d, mmr.KV_F32, start, T)
    rng = np.random.default_rng(d + hq + start)
    n = start + T
    k = rng.standard_normal((hkv, n, d)).astype(np.float32)
    v = rng.standard_normal((hkv, n, d)).astype(np.float32)
    q = rng.standard_normal((T, hq, d)).astype(np.float32)
    dq, out = mmr.DeviceArray.from_numpy(q.reshape(T, hq * d)), mmr.DeviceArray((T, hq * d), np.float32)

    def attend(v):
        cache = mmr.KvCache(hkv, d, n, mmr.KV_F32)
        cache.upload(k, v)
        mmr.prefill_attention(dq, cache, start, T, hq, hkv, d, out)
        return out.numpy().reshape(T, hq, d)

    size = np.ones(d, np.float32)
    size[d // 4: d // 2] = 2.0**-40
    np.testing.assert_array_equal(attend(v * size), attend(v) * size)

    v[:, :, : d // 2] *= np.exp2(rng.uniform(-16, 0, (hkv, 1, d // 2))).astype(np.float32)
    v[:, :, d // 2:] *= np.exp2(rng.uniform(-16, 0, (hkv, n, 1))).astype(np.float32)
    got = attend(v)
    hidden = np.arange(n)[None, :] > start + np.arange(T)[:, None]
    for h in range(hq):
        g = h // (hq // hkv)
        s = q[:, h].astype(np.float64) @ k[g].astype(np.float64).T / np.sqrt(d)
        s[hidden] = -np.inf
        p = np.exp(s - s.max(axis=1, keepdims=True))
        ref = p @ v[g].astype(np.float64) / p.sum(axis=1, keepdims=True)
        err = np.abs(got[:, h] - ref).max(axis=0) / np.abs(ref).max(axis=0)
        assert err.max() < 5e-6, (h, int(err.argmax()), float(err.max()))


@pytest.mark.parametrize("kv", ["f16", "f32"])
@pytest.mark.parametrize("d", [64, 96])
def test_prefill_attention_many_rows_confines_infinities(gpu, d, kv):
    # An infinite value reaches its own dim of its own and later queries, a NaN
    # value likewise; an infinite key makes a score of -inf, which counts for
    # nothing, or of +inf, whose row is NaN.  All else is as without them.
    mmr = gpu
    hq, hkv, start, T = 8, 2, 40, 2000
    print(f"[case] prefill attention infinities d={d} kv={kv}", flush=True)
    rng = np.random.default_rng(d)
    n = start + T
    dt = np.float16 if kv == "f16" else np.float32
    k = rng.standard_normal((hkv, n, d)).astype(dt)
    v = (4 * rng.standard_normal((hkv, n, d))).astype(dt)
    q = rng.standard_normal((T, hq, d)).astype(np.float32)
    planted = v.copy()
    planted[0, 1005, 7], planted[0, 1790, 40] = np.inf, np.nan
    k[1, 1500, 9] = -np.inf
    cache = mmr.KvCache(hkv, d, n, mmr.KV_F16 if kv == "f16" else mmr.KV_F32)
    cache.upload(k, planted)
    dq, out = mmr.DeviceArray.from_numpy(q.reshape(T, hq * d)), mmr.DeviceArray((T, hq * d), np.float32)
    mmr.prefill_attention(dq, cache, start, T, hq, hkv, d, out)
    got = out.numpy().reshape(T, hq, d)
    position = start + np.arange(T)
    hidden = np.arange(n)[None, :] > position[:, None]
    with np.errstate(invalid="ignore"):
        for h in range(hq):
            g = h // (hq // hkv)
            s = q[:, h].astype(np.float64) @ k[g].astype(np.float64).T / np.sqrt(d)
            s[hidden] = -np.inf
            p = np.exp(s - s.max(axis=1, keepdims=True))
            ref = p @ v[g].astype(np.float64) / p.sum(axis=1, keepdims=True)
            if g == 0:
                ref[position >= 1005, 7] = np.inf
                ref[position >= 1790, 40] = np.nan
            np.testing.assert_array_equal(np.isnan(got[:, h]), np.isnan(ref))
            np.testing.assert_array_equal(np.isposinf(got[:, h]), np.isposinf(ref))
            finite = np.isfinite(ref)
            assert 0 < finite.sum() and np.abs(got[:, h] - ref)[finite].max() < 1e-5 * np.abs(ref[finite]).max(), h


def synth_model(mmr, g):
    return mmr.Model.synthetic(mmr.make_config(**g["config"]), g["seed"], g["std"], g["round_fp16"])


@pytest.mark.parametrize("case,chunk", [("mini", None), ("mini", 7), ("cfg0", None), ("cfg0", 64)])
def test_gemm_prefill_matches_tokenwise_prefill(gpu, monkeypatch, case, chunk):
    # the chunked GEMM prefill (one or several chunks) against the same prompt
    # fed token by token through the decode step: same next token, logits
    # within the bound, then identical greedy continuations
    mmr = gpu
    print(f"[case] prefill {case} chunk={chunk}", flush=True)
    g = load_golden(case)
    m = synth_model(mmr, g)
    rng = np.random.default_rng(5)
    prompt = [int(t) for t in rng.integers(0, g["config"]["vocab_size"], 150)]
    monkeypatch.setenv("MMR_PREFILL_TOKENWISE", "1")
    tok = m.make_state(200)
    monkeypatch.delenv("MMR_PREFILL_TOKENWISE")
    if chunk:
        monkeypatch.setenv("MMR_PREFILL_CHUNK", str(chunk))
    gem = m.make_state(200)
    for st in (tok, gem):
        st.enqueue_prefill(prompt)
        st.synchronize()
        assert st.position == len(prompt)
    assert rel_err(gem.read_logits(), tok.read_logits()) < 1e-4
    assert gem.read_sequence(0, len(prompt) + 1).tolist() == tok.read_sequence(0, len(prompt) + 1).tolist()
    for st in (tok, gem):
        st.enqueue_decode(24)
        st.synchronize()
    assert gem.read_sequence(len(prompt), 25).tolist() == tok.read_sequence(len(prompt), 25).tolist()


def test_gemm_prefill_on_used_state_and_fp16_cache(gpu, monkeypatch):
    # a second prompt appended to a state that already holds a sequence, and an
    # fp16 KV cache: GEMM prefill and token-by-token decode agree
    mmr = gpu
    g = load_golden("mini")
    m = synth_model(mmr, g)
    monkeypatch.setenv("MMR_PREFILL_TOKENWISE", "1")
    tok = m.make_state(128, mmr.KV_F16)
    monkeypatch.delenv("MMR_PREFILL_TOKENWISE")
    gem = m.make_state(128, mmr.KV_F16)
    for st in (tok, gem):
        st.enqueue_prefill(g["prompt"])
        st.enqueue_decode(5)
        st.enqueue_prefill([3, 1, 4, 1, 5, 9, 2, 6])
        st.synchronize()
    assert tok.position == gem.position == len(g["prompt"]) + 5 + 8
    n = tok.position + 1
    assert gem.read_sequence(0, n).tolist() == tok.read_sequence(0, n).tolist()
    assert rel_err(gem.read_logits(), tok.read_logits()) < 1e-4


@pytest.mark.parametrize("prompt_len", [256, 512])
def test_gemm_prefill_swiglu_presplit_tilings(gpu, monkeypatch, prompt_len):
    # hidden 256 with FFN 1536 (gate_up n = 3072, k = 256): unsplit 32 x 64
    # tiles at 256 and at 512 rows (the only K tile pair forbids splits),
    # writing the SwiGLU output pre-split for the down GEMM (MiniMind2's
    # gate_up covers the 64 x 64 tiles).  GEMM prefill against the same prompt
    # fed token by token.
    mmr = gpu
    print(f"[case] prefill swiglu tiling rows={prompt_len}", flush=True)
    cfg = mmr.make_config(hidden_size=256, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2,
                          head_dim=64, intermediate_size=1536, vocab_size=512, max_position_embeddings=1024,
                          rms_norm_eps=1e-5, rope_theta=1e6, tie_word_embeddings=0)
    m = mmr.Model.synthetic(cfg, 13, 0.02, True)
    rng = np.random.default_rng(prompt_len)
    prompt = [int(t) for t in rng.integers(0, 512, prompt_len)]
    monkeypatch.setenv("MMR_PREFILL_TOKENWISE", "1")
    tok = m.make_state(prompt_len + 16)
    monkeypatch.delenv("MMR_PREFILL_TOKENWISE")
    gem = m.make_state(prompt_len + 16)
    for st in (tok, gem):
        st.enqueue_prefill(prompt)
        st.synchronize()
    assert rel_err(gem.read_logits(), tok.read_logits()) < 1e-4
    for st in (tok, gem):
        st.enqueue_decode(12)
        st.synchronize()
    n = prompt_len + 13
    assert gem.read_sequence(0, n).tolist() == tok.read_sequence(0, n).tolist()


@pytest.mark.parametrize("prompt_len", [333, 600, 1300])
def test_minimind2_ragged_chunks_match_tokenwise(gpu, monkeypatch, prompt_len):
    # MiniMind2 shapes at row counts below the 512-row chunk (333 alone; 600 =
    # 512 + 88; 1300 = 2 x 512 + 276): fewer rows take more K splits, so the
    # split-K partial sets of these chunks are larger than the full chunk's.
    # GEMM prefill against the same prompt fed token by token through the
    # fp16 KV cache (from 1,025 positions on, the token-by-token steps run 16
    # attention splits over 17 or more tiles: blocks with two tiles).
    mmr = gpu
    print(f"[case] MiniMind2 prefill rows={prompt_len}", flush=True)
    g = load_golden("cfg3_short")
    m = synth_model(mmr, g)
    prompt = mmr.synthesize_prompt(11, prompt_len, 6400).tolist()
    monkeypatch.setenv("MMR_PREFILL_TOKENWISE", "1")
    tok = m.make_state(prompt_len + 8, mmr.KV_F16)
    monkeypatch.delenv("MMR_PREFILL_TOKENWISE")
    gem = m.make_state(prompt_len + 8, mmr.KV_F16)
    for st in (tok, gem):
        st.enqueue_prefill(prompt)
        st.synchronize()
    assert rel_err(gem.read_logits(), tok.read_logits()) < 1e-4
    assert gem.read_sequence(prompt_len, 1).tolist() == tok.read_sequence(prompt_len, 1).tolist()


@pytest.mark.parametrize("prompt_len", [2305, 2500, 3500, 5000])
def test_minimind2_long_passes_match_chunks(gpu, monkeypatch, prompt_len):
    # one pass of 2,500 rows and two of them (the many-rows GEMM for every
    # projection, O and down in 3 K splits, QKV in 2; the many-rows attention,
    # also after 2,500 cached rows), 2,305 (a last row tile of 1 row, K in uneven
    # splits of 5, 5 and 6 chunks) and 3,500 (2 splits, QKV 1) against the
    # same prompt in 512-row chunks: same next token, logits within 1e-4 (fp16
    # K/V roundings of differently grouped fp32 sums, as in the tests below)
    mmr = gpu
    print(f"[case] MiniMind2 long prefill rows={prompt_len}", flush=True)
    g = load_golden("cfg3_short")
    m = synth_model(mmr, g)
    prompt = mmr.synthesize_prompt(12, prompt_len, 6400).tolist()
    monkeypatch.setenv("MMR_PREFILL_CHUNK", "512")
    chunks = m.make_state(prompt_len + 8, mmr.KV_F16)
    monkeypatch.delenv("MMR_PREFILL_CHUNK")
    passes = m.make_state(prompt_len + 8, mmr.KV_F16)
    for st in (chunks, passes):
        st.enqueue_prefill(prompt)
        st.synchronize()
    assert rel_err(passes.read_logits(), chunks.read_logits()) < 1e-4
    assert passes.read_sequence(prompt_len, 1).tolist() == chunks.read_sequence(prompt_len, 1).tolist()


def test_long_prompts_without_the_pass_buffers(gpu, monkeypatch):
    # no memory for the buffers of long passes (and, in a second state, for those
    # of the longer of two prompts): passes of 512 tokens on the state's own,
    # with the bits of such passes
    mmr = gpu
    print("[case] long prompts without the pass buffers", flush=True)
    g = load_golden("mini")
    m = synth_model(mmr, g)
    rng = np.random.default_rng(4)
    first, second = ([int(t) for t in rng.integers(0, g["config"]["vocab_size"], n)] for n in (700, 1300))
    logits = {}
    for name, switch, value in (("chunks", "MMR_PREFILL_CHUNK", "512"), ("none", "MMR_PREFILL_BUFFER_MB", "0"),
                                ("some", "MMR_PREFILL_BUFFER_MB", "16")):
        monkeypatch.setenv(switch, value)
        st = m.make_state(2048, mmr.KV_F32)
        monkeypatch.delenv(switch)
        st.enqueue_prefill(first)
        one = st.read_logits()
        st.enqueue_prefill(second)
        st.enqueue_decode(3)
        logits[name] = one, st.read_logits()
    for one, two in zip(logits["chunks"], logits["none"]):
        np.testing.assert_array_equal(two, one)
    for one, two in zip(logits["chunks"], logits["some"]):
        assert rel_err(two, one) < 1e-4


def test_gemm_kernels_agree(gpu, monkeypatch):
    # the direct-to-LDS GEMM (pre-split A, K % 64 == 0) against the
    # register-staged one (MMR_GEMM_REGISTER_STAGED=1) on a MiniMind2 prefill
    # of 512 tokens: same next token, logits within 1e-4 (the two add the
    # same exact products in different groupings; through 16 layers and the
    # fp16 KV cache's roundings that leaves ~5e-5, as against token-by-token)
    mmr = gpu
    g = load_golden("cfg3_short")
    m = synth_model(mmr, g)
    prompt = mmr.synthesize_prompt(5, 512, 6400).tolist()
    dma = m.make_state(520, mmr.KV_F16)
    monkeypatch.setenv("MMR_GEMM_REGISTER_STAGED", "1")
    staged = m.make_state(520, mmr.KV_F16)
    staged.enqueue_prefill(prompt)
    staged.synchronize()
    monkeypatch.delenv("MMR_GEMM_REGISTER_STAGED")
    dma.enqueue_prefill(prompt)
    dma.synchronize()
    assert rel_err(dma.read_logits(), staged.read_logits()) < 1e-4
    assert dma.read_sequence(512, 1).tolist() == staged.read_sequence(512, 1).tolist()


MM2_LAYER = dict(hidden_size=768, num_hidden_layers=1, num_attention_heads=8, num_key_value_heads=2, head_dim=96,
                 intermediate_size=2048, vocab_size=6400, max_position_embeddings=32768, rms_norm_eps=1e-5,
                 rope_theta=1e6, tie_word_embeddings=1)


def layer_arrays(rng):
    H, D, F = 768, 96, 2048
    w = lambda rows, cols: f16_weights(rng, rows, cols)[1]  # noqa: E731
    gain = lambda n: (1 + 0.1 * rng.standard_normal(n)).astype(np.float32)  # noqa: E731
    return {"input_norm": gain(H), "post_attention_norm": gain(H), "q_norm": gain(D), "k_norm": gain(D),
            "q_proj": w(8 * D, H), "k_proj": w(2 * D, H), "v_proj": w(2 * D, H), "o_proj": w(H, 8 * D),
            "gate_proj": w(F, H), "up_proj": w(F, H), "down_proj": w(H, F)}


def run_prefill_layer(mmr, arrays, hs, kv):
    T, H = hs.shape
    lw = mmr.LayerWeights.create(mmr.make_config(**MM2_LAYER), **arrays)
    cache = mmr.KvCache(2, 96, T, kv)
    x, y = mmr.DeviceArray.from_numpy(hs.reshape(-1)), mmr.DeviceArray(T * H, np.float32)
    lw.prefill(cache, x, 0, T, y, mmr.DeviceArray(lw.prefill_workspace_size(T), np.uint8))
    out = y.numpy().reshape(T, H), *cache.download(T)
    lw.free()
    return out


@pytest.mark.parametrize("T", [512, 1500, 3000])
def test_layer_planes_keep_small_channels_beside_a_large_gain(gpu, T):
    # A channel whose gain is 2^30 times the others', in a chunk of 128 columns
    # that no weight reads: the normalised rows' planes have one scale per 128
    # columns, so every other chunk, and with them the layer's result and its
    # cache rows, keep their bits.  512 rows: 64 x 64 tiles; 1,500: gate_up on
    # the many-rows tiles and QKV on them in 3 K splits; 3,000: in 2.
    mmr = gpu
    print(f"[case] layer with a large gain T={T}", flush=True)
    rng = np.random.default_rng(T)
    arrays = layer_arrays(rng)
    for n in ("q_proj", "k_proj", "v_proj", "gate_proj", "up_proj"):
        arrays[n][:, 256:384] = 0.0
    hs = rng.standard_normal((T, 768)).astype(np.float32)
    want = run_prefill_layer(mmr, arrays, hs, mmr.KV_F32)
    for n in ("input_norm", "post_attention_norm"):
        arrays[n][300] *= np.float32(2.0**30)
    got = run_prefill_layer(mmr, arrays, hs, mmr.KV_F32)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)


@pytest.mark.parametrize("T", [512, 1500, 3000])
def test_layer_act_keeps_small_columns_beside_large_ones(gpu, T):
    # 32 FFN columns 2^18 times the others' size that the down projection does
    # not read: act is split under a scale per 32 columns, pre-split (512 and
    # 1,500 rows) and in the many-rows GEMM's K splits (3,000)
    mmr = gpu
    print(f"[case] layer with large FFN columns T={T}", flush=True)
    rng = np.random.default_rng(T)
    arrays = layer_arrays(rng)
    arrays["up_proj"][1056:1088] *= np.float32(2.0**-9)  # exact in fp16 on both sides
    arrays["up_proj"] = arrays["up_proj"].astype(np.float16).astype(np.float32)
    arrays["down_proj"][:, 1056:1088] = 0.0
    hs = rng.standard_normal((T, 768)).astype(np.float32)
    want = run_prefill_layer(mmr, arrays, hs, mmr.KV_F16)
    arrays["up_proj"][1056:1088] *= np.float32(2.0**27)
    got = run_prefill_layer(mmr, arrays, hs, mmr.KV_F16)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)
