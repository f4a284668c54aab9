"""Decode attention around its split and round edges (one split up to 128 or
256 positions, splits of 128, more than 64 splits' worth), for every head
layout, against float64."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pos", [0, 1, 7, 63, 64, 127, 128, 255, 256, 300, 1000, 8191, 8300])
@pytest.mark.parametrize("nq,nkv,hd", [(2, 2, 64), (4, 2, 64), (8, 2, 64), (8, 1, 64), (2, 2, 128), (4, 2, 128), (8, 2, 128),
                                       (8, 1, 128), (1, 1, 256), (4, 2, 256), (8, 2, 256)])
def test_attn_decode_edges(mdx, gpu, nq, nkv, hd, pos):
    rng = np.random.default_rng(pos + hd + nq)
    kvd = nkv * hd
    qkv = rng.standard_normal(nq * hd + 2 * kvd).astype(np.float32)
    k = rng.standard_normal((pos, kvd)).astype(np.float16)
    v = rng.standard_normal((pos, kvd)).astype(np.float16)
    # norms off
    out, k_new, v_new = mdx.attn_decode(nq, nkv, hd, pos, 1, 1e6, 1e-6, None, None, qkv, k.view(np.uint16).ravel(),
                                        v.view(np.uint16).ravel())
    ang = pos * (1e6 ** (-np.arange(0, hd, 2) / hd)).astype(np.float32).astype(np.float64)
    q = qkv[:nq * hd].astype(np.float64).reshape(nq, hd)
    a, b = q[:, :hd // 2], q[:, hd // 2:]
    q = np.concatenate([a * np.cos(ang) - b * np.sin(ang), b * np.cos(ang) + a * np.sin(ang)], 1)
    kk = np.concatenate([k.astype(np.float64), k_new.view(np.float16).astype(np.float64)[None]]).reshape(pos + 1, nkv, hd)
    vv = np.concatenate([v.astype(np.float64), v_new.view(np.float16).astype(np.float64)[None]]).reshape(pos + 1, nkv, hd)
    ref = np.empty((nq, hd))
    for h in range(nq):
        s = kk[:, h // (nq // nkv)] @ q[h] / np.sqrt(hd)
        p = np.exp(s - s.max())
        ref[h] = p @ vv[:, h // (nq // nkv)] / p.sum()
    # the output's fp16 rounding (2^-11 of a value), and the rotation angle in
    # fp32: 2^-24 of an angle of up to 8300 turns a query by 5e-4
    assert rel_err(out, ref.ravel()) < 2.0 ** -11 + 5e-4


def _softmax64(q, kk, vv, hd):
    """One head as IEEE arithmetic has it: the maximum looks past NaN, everything after it carries them."""
    with np.errstate(all="ignore"):
        s = kk @ q / np.sqrt(hd)
        p = np.exp(s - np.fmax.reduce(s))
        return (p[:, None] * vv).sum(0) / p.sum()


# first..last - 1: all of the first split of two, of the second of three, of two
# in the middle of six, one position, all but the newest.  The layouts merge
# their splits in 32, 8, 8, 4, 2, 8 and 2 groups.
@pytest.mark.parametrize("what", ["nan", "overflow", "minus_inf", "minus_inf_v", "v_nan"])
@pytest.mark.parametrize("first,last,pos", [(0, 100, 199), (101, 202, 300), (234, 468, 700), (3, 4, 40), (0, 700, 700)])
@pytest.mark.parametrize("nq,nkv,hd", [(2, 2, 64), (8, 2, 64), (4, 2, 128), (8, 2, 128), (16, 2, 128), (2, 2, 256), (8, 2, 256)])
def test_attn_decode_non_finite_cache(mdx, gpu, nq, nkv, hd, first, last, pos, what):
    """Non-finite K or V values of the first KV head give its query heads what
    the arithmetic gives, and leave the others alone."""
    rng = np.random.default_rng(pos + hd + nq)
    kvd = nkv * hd
    ang = pos * (1e6 ** (-np.arange(0, hd, 2) / hd)).astype(np.float32).astype(np.float64)
    qkv = rng.standard_normal(nq * hd + 2 * kvd).astype(np.float32)
    q32 = qkv[:nq * hd].reshape(nq, hd)
    q32[:, 0], q32[:, hd // 2] = np.cos(ang[0]), -np.sin(ang[0])      # dimension 0 is 1 once rotated
    k = rng.standard_normal((pos, nkv, hd)).astype(np.float16)
    v = rng.standard_normal((pos, nkv, hd)).astype(np.float16)
    if what == "nan":
        k[first:last, 0, 5] = np.nan
    elif what == "overflow":
        k[first:last, 0, 1:9], k[first:last, 0, 9:17] = np.inf, -np.inf      # of both signs for any query
    elif what == "v_nan":
        v[first, 0, 3] = np.nan
    else:
        k[first:last, 0, 0] = -np.inf
        if what == "minus_inf_v":
            v[first, 0, 3] = np.inf          # of probability 0
    out, k_new, v_new = mdx.attn_decode(nq, nkv, hd, pos, 1, 1e6, 1e-6, None, None, qkv, k.view(np.uint16).ravel(),
                                        v.view(np.uint16).ravel())
    q = q32.astype(np.float64)
    a, b = q[:, :hd // 2], q[:, hd // 2:]
    q = np.concatenate([a * np.cos(ang) - b * np.sin(ang), b * np.cos(ang) + a * np.sin(ang)], 1)
    kk = np.concatenate([k, k_new.view(np.float16).reshape(1, nkv, hd)]).astype(np.float64)
    vv = np.concatenate([v, v_new.view(np.float16).reshape(1, nkv, hd)]).astype(np.float64)
    ref = np.stack([_softmax64(q[h], kk[:, h // (nq // nkv)], vv[:, h // (nq // nkv)], hd) for h in range(nq)]).ravel()
    assert np.array_equal(np.isnan(out), np.isnan(ref))
    ok = np.isfinite(ref)
    assert ok[nq // nkv * hd:].all() and rel_err(out[ok], ref[ok]) < 2.0 ** -11 + 5e-4
