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
