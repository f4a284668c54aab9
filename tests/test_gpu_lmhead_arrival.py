"""The lm_head's argmax over many workgroups: every arrival pattern (fewer
workgroups than counter groups, uneven groups, the largest grid), launched
again and again on the same scratch, through the greedy loop and single steps."""
import os

import numpy as np
import pytest

from conftest import tiny_config

pytestmark = pytest.mark.gpu


# int8 rows of 64/128 (k_gemv: 1, 2 or 8 rows per wave by the row count) with
# 1, 31, 33, 1000, 1024 (capped) workgroups
@pytest.mark.parametrize("V", [3, 124, 130, 8000, 70001])
def test_argmax_over_workgroups(mdx, gpu, workdir, V):
    cfg, d = tiny_config(mdx, vocab_size=V)
    path = os.path.join(workdir, "lm_%d" % V)
    mdx.write_model(path, cfg, 1, 5)
    g = mdx.Decoder(path, cfg, "int8", 64)
    rng = np.random.default_rng(V)
    for _ in range(12):
        tok, lg = g.step(0, embedding=rng.standard_normal(d["hidden_dim"]).astype(np.float32))
        assert tok == int(np.argmax(lg))
    g.clear()
    singles, t = [], 1
    for _ in range(20):
        t, lg = g.step(t)
        assert t == int(np.argmax(lg))
        singles.append(t)
    g.clear()
    assert list(g.generate_greedy(1, 20)[0]) == singles
