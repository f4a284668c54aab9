"""rmp_run over its pinned slots: inputs read in place and copied in, ragged K,
one pass and several (more than there are slots), and new inputs call after
call on one context, against float64."""
import ctypes as C

import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


# 8 KB inputs are read in host memory: (1,4096), (2,2048) and (64,64) lie on
# it, (1,4097) and (2,2080) past it.  Passes of 2 MB of output in runs of 64
# rows: (300,1000,3074) two, (900,64,4098) eight through four slots, the
# others one.
@pytest.mark.parametrize("M,K,N", [(1, 8, 2), (1, 4096, 130), (1, 64, 5002), (1, 40, 122), (1, 4097, 64), (2, 2048, 2), (2, 2080, 66), (64, 64, 34),
                                   (65, 33, 30), (129, 96, 2), (300, 1000, 3074), (900, 64, 4098)])
def test_rmp_passes(mdx, gpu, M, K, N):
    rng = np.random.default_rng(M + K + N)
    w = (rng.standard_normal((K, N)) * 0.02).astype(np.float16)
    L = mdx.lib()
    h = L.rmp_create(C.byref(mdx.RmpConfig(M, K, N, 0, 0, 2)), w.ctypes.data, None)
    assert h
    try:
        for _ in range(3):
            x = rng.standard_normal((M, K)).astype(np.float16)
            y = np.full((M, N), np.nan, np.float32)
            assert L.rmp_run(h, x.view(np.uint16).ctypes.data_as(mdx._U16), y.ctypes.data_as(mdx._F)) == 0
            # fp32 sums of exact products
            assert rel_err(y, x.astype(np.float64) @ w.astype(np.float64)) < 1e-5
    finally:
        L.rmp_destroy(h)


def test_rmp_output_over_input(mdx, gpu):
    """Input rows at the start of the output buffer, eight passes through four
    slots: the first passes' rows are stored before the last are read."""
    M, K, N = 900, 64, 4098
    rng = np.random.default_rng(1)
    w = (rng.standard_normal((K, N)) * 0.02).astype(np.float16)
    x = rng.standard_normal((M, K)).astype(np.float16)
    y = np.zeros((M, N), np.float32)
    L = mdx.lib()
    h = L.rmp_create(C.byref(mdx.RmpConfig(M, K, N, 0, 0, 2)), w.ctypes.data, None)
    assert h
    try:
        for at in (0, M * N * 4 - x.nbytes, 4 * N * 500):
            y.view(np.uint8).ravel()[at:at + x.nbytes] = x.view(np.uint8).ravel()
            xin = C.cast(C.c_void_p(y.ctypes.data + at), mdx._U16)
            assert L.rmp_run(h, xin, y.ctypes.data_as(mdx._F)) == 0
            assert rel_err(y, x.astype(np.float64) @ w.astype(np.float64)) < 1e-5
    finally:
        L.rmp_destroy(h)
