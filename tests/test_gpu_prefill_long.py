"""Batch prefill of more than 64 rows (the tiled projections and the MFMA
attention) against float64 / oracle references: every weight kind, tile edges,
K tails, split and unsplit projections, each head layout, a cache that already
holds positions, and infinities in the cache."""
import os

import numpy as np
import pytest

from conftest import cosine, rel_err, tiny_config

pytestmark = pytest.mark.gpu

QNAME = {0: "fp16", 1: "int8", 2: "int4"}


def _weights(rng, kind, K, N):
    """(on-disk data, scales, the values as float64)."""
    if kind == 0:
        w = (rng.standard_normal((K, N)) * 0.02).astype(np.float16)
        return w.view(np.uint16), None, w.astype(np.float64)
    if kind == 1:
        q, s = rng.integers(-128, 128, (K, N)).astype(np.int8), rng.uniform(1e-4, 2e-4, N).astype(np.float32)
        return q, s, q.astype(np.float64) * s
    q, s = rng.integers(-8, 8, (K, N)), rng.uniform(1e-3, 3e-3, N).astype(np.float32)
    u = (q & 15).astype(np.uint8)
    return u[:, 0::2] | (u[:, 1::2] << 4), s, q.astype(np.float64) * s


# K fp32 sums of exact products of 16-bit values: an error of at most K 2^-24
# of the sum of magnitudes, in practice sqrt(K) 2^-24 of the result's rms
# times a few; 1e-5 of the largest result holds all of these with room.
GEMM_TOL = 1e-5


@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("M,K,N", [(65, 32, 96), (100, 96, 64), (203, 1024, 4096), (129, 352, 1030), (515, 1536, 512),
                                   (2048, 64, 4096), (1, 1024, 2), (2000, 160, 2054)])
def test_long_gemm(mdx, gpu, kind, M, K, N):
    rng = np.random.default_rng(M + 3 * K + 7 * N + kind)
    x = rng.standard_normal((M, K)).astype(np.float16).astype(np.float32)
    w, s, w64 = _weights(rng, kind, K, N)
    assert rel_err(mdx.gemm(kind, M, K, N, w, s, x, long=True), x.astype(np.float64) @ w64) < GEMM_TOL


@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("M,K,N", [(65, 3072, 1024), (203, 2048, 1024), (100, 2592, 128), (515, 4096, 1536), (2000, 512, 2048), (70, 32, 32)])
def test_long_residual_norm(mdx, gpu, kind, M, K, N):
    rng = np.random.default_rng(M + 3 * K + 7 * N + kind)
    x = rng.standard_normal((M, K)).astype(np.float16).astype(np.float32)
    w, s, w64 = _weights(rng, kind, K, N)
    h0 = rng.standard_normal((M, N)).astype(np.float32)
    nw = rng.uniform(0.5, 1.5, N).astype(np.float32)
    h, x16 = mdx.gemm_residual(kind, M, K, N, w, s, x, h0, nw, long=True)
    assert rel_err(h, h0 + x.astype(np.float64) @ w64) < GEMM_TOL
    h64 = h.astype(np.float64)
    ref = h64 / np.sqrt((h64 * h64).mean(1, keepdims=True) + 1e-6) * nw
    got = x16.view(np.float16).astype(np.float64)
    assert np.all(np.abs(got - ref) <= np.abs(ref) * 2.0 ** -10 + 2.0 ** -24)   # one fp16 ulp


@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("K", [256, 512, 576, 768, 1024, 1536, 2048, 3072, 3104, 4096, 5120])
def test_long_projections_as_exact_as_64_row_ones(mdx, gpu, kind, K):
    """fp32 sums of the same exact products: no further off (2-norm) than the
    kernels of up to 64 rows; 2 % for what the inputs make of it."""
    M, N = 128, 512
    rng = np.random.default_rng(K + kind)
    x = rng.standard_normal((M, K)).astype(np.float16).astype(np.float32)
    w, s, w64 = _weights(rng, kind, K, N)
    ref, h0 = x.astype(np.float64) @ w64, np.zeros((M, N), np.float32)
    halves = [slice(0, 64), slice(64, 128)]
    off = lambda y: np.linalg.norm(y - ref)  # noqa: E731
    assert off(mdx.gemm(kind, M, K, N, w, s, x, long=True)) <= 1.02 * off(
        np.concatenate([mdx.gemm(kind, 64, K, N, w, s, x[r]) for r in halves]))
    assert off(mdx.gemm_residual(kind, M, K, N, w, s, x, h0, None, long=True)[0]) <= 1.02 * off(
        np.concatenate([mdx.gemm_residual(kind, 64, K, N, w, s, x[r], h0[r], None)[0] for r in halves]))


@pytest.mark.parametrize("M,K,N", [(70, 32, 64), (100, 96, 64), (65, 352, 128), (203, 1056, 1024), (130, 128, 64)])
def test_long_gemm_infinite_weights(mdx, gpu, M, K, N):
    """Infinite fp16 weights, also among the last k of a K that ends inside a
    stage of 64, give infinities (of both signs in one column: NaN)."""
    rng = np.random.default_rng(K)
    x = rng.uniform(0.5, 1.5, (M, K)).astype(np.float16).astype(np.float32)
    w = (rng.standard_normal((K, N)) * 0.02).astype(np.float16)
    w[K - 1, 3], w[K - 8, 5], w[0, 7], w[K - 1, 9] = np.inf, -np.inf, np.inf, np.nan
    w[K - 2, 11], w[K - 3, 11] = np.inf, -np.inf
    with np.errstate(invalid="ignore"):
        ref = x.astype(np.float64) @ w.astype(np.float64)
    h0 = rng.standard_normal((M, N)).astype(np.float32)
    wu = w.view(np.uint16)
    for y, r in ((mdx.gemm(0, M, K, N, wu, None, x, long=True), ref),
                 (mdx.gemm_residual(0, M, K, N, wu, None, x, h0, None, long=True)[0], h0 + ref)):
        assert np.array_equal(np.isnan(y), np.isnan(r)) and np.array_equal(np.isinf(y), np.isinf(r))
        assert np.array_equal(np.sign(y[np.isinf(r)]), np.sign(r[np.isinf(r)]))
        ok = np.isfinite(r)
        assert rel_err(y[ok], r[ok]) < GEMM_TOL


def _attention64(q, k, v, S, M, nq, nkv, hd):
    out = np.empty((M, nq, hd))
    for h in range(nq):
        kh, vh = k[:, h // (nq // nkv)], v[:, h // (nq // nkv)]
        s = q[:, h] @ kh.T / np.sqrt(hd)
        s[np.arange(S + M)[None, :] > S + np.arange(M)[:, None]] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = p @ vh / p.sum(1, keepdims=True)
    return out.reshape(M, -1)


# The fp16 rounding of the output is 2^-11 of it; the fp32 sums, exponentials
# and the 23-bit parts of queries and probabilities are far below that.
@pytest.mark.parametrize("qstd", [1.0, 1e-3, 300.0])
@pytest.mark.parametrize("S,M", [(0, 65), (0, 129), (63, 70), (300, 515), (1, 1)])
@pytest.mark.parametrize("nq,nkv,hd", [(4, 2, 128), (8, 2, 64), (4, 2, 256), (2, 2, 64), (4, 1, 128), (2, 2, 256), (4, 1, 64)])
def test_long_attention(mdx, gpu, S, M, nq, nkv, hd, qstd):
    rng = np.random.default_rng(S + M + hd + nq)
    q = (rng.standard_normal((M, nq, hd)) * qstd).astype(np.float32)
    k = rng.standard_normal((S + M, nkv, hd)).astype(np.float16)
    v = rng.standard_normal((S + M, nkv, hd)).astype(np.float16)
    out = mdx.attn_prefill(nq, nkv, hd, S, M, q.ravel(), k.view(np.uint16).ravel(), v.view(np.uint16).ravel(), long=True)
    ref = _attention64(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), S, M, nq, nkv, hd)
    # at qstd 300 scores reach +-1500: their fp32 rounding (2^-24 of 1500) is up to 1e-4 of a probability
    assert rel_err(out, ref) < (2.0 ** -11 + 1e-5 if qstd < 10 else 2.0 ** -11 + 1e-3)
    old = np.concatenate([mdx.attn_prefill(nq, nkv, hd, S + a, min(64, M - a), q[a:a + 64].ravel(),
                                           k[:S + a + 64].view(np.uint16).ravel(), v[:S + a + 64].view(np.uint16).ravel())
                          for a in range(0, M, 64)])
    assert np.abs(out - ref).mean() <= 1.02 * np.abs(old - ref).mean() + 1e-9


@pytest.mark.parametrize("qstd", [1.0, 1e-3, 8.0, 100.0])
@pytest.mark.parametrize("nq,nkv,hd", [(16, 8, 128), (16, 4, 128), (16, 8, 64), (8, 2, 256)])
def test_long_attention_as_exact_as_fp32(mdx, gpu, nq, nkv, hd, qstd):
    """The share of outputs that are not the float64 result's fp16 rounding is
    a measure of the error before that rounding: no larger than in the kernel
    that holds queries and probabilities in fp32.  About 1 in 1000 of 0.5 to 1
    million: four standard deviations of the two counts' difference."""
    M = 515
    rng = np.random.default_rng(hd + nq)
    q = (rng.standard_normal((M, nq, hd)) * qstd).astype(np.float32)
    k = rng.standard_normal((M, nkv, hd)).astype(np.float16)
    v = rng.standard_normal((M, nkv, hd)).astype(np.float16)
    ku, vu = k.view(np.uint16), v.view(np.uint16)
    long = mdx.attn_prefill(nq, nkv, hd, 0, M, q.ravel(), ku.ravel(), vu.ravel(), long=True)
    old = np.concatenate([mdx.attn_prefill(nq, nkv, hd, a, min(64, M - a), q[a:a + 64].ravel(), ku[:a + 64].ravel(),
                                           vu[:a + 64].ravel()) for a in range(0, M, 64)])
    ref = _attention64(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), 0, M, nq, nkv, hd)
    want = ref.astype(np.float16).astype(np.float32)
    a, b = (long != want).sum(), (old != want).sum()
    assert a <= b + 4 * np.sqrt(a + b)


@pytest.mark.parametrize("where,val", [("v", np.inf), ("v", np.nan), ("k", np.inf), ("k", -np.inf), ("k", np.nan)])
@pytest.mark.parametrize("hd", [64, 128, 256])
def test_long_attention_non_finite_cache(mdx, gpu, hd, where, val):
    """A non-finite K or V value at one position leaves the rows before it
    alone, and gives the others what the one-row-per-block kernel gives."""
    M, nq, nkv, at = 130, 4, 2, 77
    rng = np.random.default_rng(hd)
    q = rng.standard_normal((M, nq, hd)).astype(np.float32)
    k = rng.standard_normal((M, nkv, hd)).astype(np.float16)
    v = rng.standard_normal((M, nkv, hd)).astype(np.float16)
    (k if where == "k" else v)[at, 1, 5] = val
    ku, vu = k.view(np.uint16), v.view(np.uint16)
    out = mdx.attn_prefill(nq, nkv, hd, 0, M, q.ravel(), ku.ravel(), vu.ravel(), long=True)
    old = np.concatenate([mdx.attn_prefill(nq, nkv, hd, a, min(64, M - a), q[a:a + 64].ravel(), ku[:a + 64].ravel(),
                                           vu[:a + 64].ravel()) for a in range(0, M, 64)])
    assert np.isfinite(out[:at]).all()
    assert np.array_equal(np.isnan(out), np.isnan(old)) and np.array_equal(np.isposinf(out), np.isposinf(old))
    ok = np.isfinite(old)
    assert np.abs(out[ok] - old[ok]).max() < 2.0 ** -10 * np.abs(old[ok]).max()


@pytest.mark.parametrize("quant", [0, 1, 2])
@pytest.mark.parametrize("over", [dict(rope_style=0), dict(num_q_heads=2, num_kv_heads=2, head_dim=128, rope_style=1),
                                  dict(num_q_heads=4, num_kv_heads=1, head_dim=256), dict(hidden_dim=160, ffn_dim=352, has_qk_norm=0)])
def test_long_prefill_decoder(mdx, gpu, oracle_lib, workdir, quant, over):
    """A 70-row prompt, a 131-row one behind it, and a step: cache rows and
    logits against the oracle."""
    cfg, d = tiny_config(mdx, max_seq_len=256, **over)
    path = os.path.join(workdir, "long_%d_%s" % (quant, "_".join(map(str, over.values()))))
    if not os.path.isdir(path):
        mdx.write_model(path, cfg, quant, 77 + quant)
    g = mdx.Decoder(path, cfg, QNAME[quant], 256)
    o = oracle_lib.Model(path, d, quant, 256, kv_fp16=True)
    rng = np.random.default_rng(3)
    for n in (70, 131):
        emb = rng.standard_normal((n, d["hidden_dim"])).astype(np.float32)
        tok, lg = g.prefill_logits(emb)
        assert o.prefill_batch(emb) == 0 and tok >= 0
        x16 = oracle_lib.f16_to_f32(oracle_lib.f32_to_f16(o.last_normed())).astype(np.float64)
        hq, hs = o.lm_head_q()
        assert rel_err(lg, (hq.astype(np.float64) @ x16) * hs) < 1e-3
    for layer in range(d["num_layers"]):
        for a, b in zip(g.kv_read(layer, 0, 201), o.kv_read(layer, 0, 201)):
            assert rel_err(a, b) < 2e-3
    tg, lg = g.step(5)
    to, lo = o.step(5)
    assert tg == to and rel_err(lg, lo) < 1e-3 and cosine(lg, lo) > 0.9999
    assert g.seq_len == o.seq_len == 202


def _prompts_and_a_step(mdx, oracle_lib, path, cfg, d, max_seq, prompts, rows):
    """Prompts one behind the other, then a step: last-row logits and the given
    cache rows against the oracle."""
    g = mdx.Decoder(path, cfg, "fp16", max_seq)
    o = oracle_lib.Model(path, d, 0, max_seq, kv_fp16=True)
    rng = np.random.default_rng(4)
    for n in prompts:
        emb = rng.standard_normal((n, d["hidden_dim"])).astype(np.float32)
        tok, lg = g.prefill_logits(emb)
        assert o.prefill_batch(emb) == 0 and tok >= 0
        x16 = oracle_lib.f16_to_f32(oracle_lib.f32_to_f16(o.last_normed())).astype(np.float64)
        hq, hs = o.lm_head_q()
        assert rel_err(lg, (hq.astype(np.float64) @ x16) * hs) < 1e-3
    for layer in range(d["num_layers"]):
        for at, n in rows:
            for a, b in zip(g.kv_read(layer, at, n), o.kv_read(layer, at, n)):
                assert rel_err(a, b) < 2e-3
    tg, lg = g.step(5)
    to, lo = o.step(5)
    assert tg == to and rel_err(lg, lo) < 1e-3 and g.seq_len == o.seq_len == sum(prompts) + 1


@pytest.mark.parametrize("over", [dict(), dict(num_q_heads=4, num_kv_heads=1, head_dim=256)])
def test_long_prefill_in_passes(mdx, gpu, oracle_lib, workdir, over):
    """2300 rows (two passes of 1150, which reuse the activations and the
    upload ring; head_dim 256 takes its position from the device), and 2100
    more behind them: the rows on both sides of every pass's end."""
    cfg, d = tiny_config(mdx, max_seq_len=4500, num_layers=1, **over)
    path = os.path.join(workdir, "passes_%d" % d["head_dim"])
    mdx.write_model(path, cfg, 0, 78)
    _prompts_and_a_step(mdx, oracle_lib, path, cfg, d, 4500, (2300, 2100), [(0, 4), (1100, 100), (2290, 20), (3340, 20), (4390, 10)])


@pytest.mark.parametrize("chunk,prompts", [(16, (70, 16, 1)), (63, (127, 64)), (1, (5,))])
def test_prefill_in_short_chunks(mdx, gpu, oracle_lib, workdir, chunk, prompts):
    """A max_batch_prefill below 64 is kept to, whatever the prompt's length."""
    cfg, d = tiny_config(mdx, max_seq_len=256, max_batch_prefill=chunk)
    path = os.path.join(workdir, "chunks")
    if not os.path.isdir(path):
        mdx.write_model(path, cfg, 0, 79)
    _prompts_and_a_step(mdx, oracle_lib, path, cfg, d, 256, prompts, [(0, sum(prompts))])
