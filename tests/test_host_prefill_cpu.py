"""The host side of batch prefill over a device that runs its queue as late as
it may (fake_device.c): the passes of a long prompt, the chunks of a short
one, what the last row's logits are taken from, and a call that fails."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import PKG, ROOT, tiny_config

HERE = os.path.dirname(os.path.abspath(__file__))
F32P = C.POINTER(C.c_float)


@pytest.fixture(scope="session")
def fake(tmp_path_factory):
    """The host C runtime linked against fake_device.c."""
    tmp = str(tmp_path_factory.mktemp("fake"))
    host = os.path.join(PKG, "csrc", "host")
    flags = ["gcc", "-O1", "-fPIC", "-std=gnu11", "-w"] + ["-I" + d for d in (
        os.path.join(ROOT, "include"), os.path.join(PKG, "csrc", "kernels"), host)]
    objs = []
    for src in [os.path.join(host, f) for f in sorted(os.listdir(host)) if f.endswith(".c")] + [os.path.join(HERE, "fake_device.c")]:
        objs.append(os.path.join(tmp, os.path.basename(src) + ".o"))
        subprocess.run(flags + ["-c", src, "-o", objs[-1]], check=True)
    syms = subprocess.run(["nm"] + objs, capture_output=True, text=True, check=True).stdout.split("\n")
    have = {s.split()[-1] for s in syms if " T " in s}
    need = {s.split()[-1] for s in syms if " U mdx" in s} - have
    rest = os.path.join(tmp, "rest.c")
    with open(rest, "w") as f:
        f.writelines("int %s() { return 0; }\n" % n for n in sorted(need))
    out = os.path.join(tmp, "libfake.so")
    subprocess.run(flags + ["-shared", rest] + objs + ["-o", out, "-lpthread", "-lm"], check=True)
    L = C.CDLL(out)
    L.matmul_decoder_create.restype = C.c_void_p
    L.matmul_decoder_create.argtypes = [C.c_char_p, C.c_void_p, C.c_int, C.c_int]
    L.matmul_decoder_destroy.argtypes = L.matmul_decoder_clear_kv_cache.argtypes = L.matmul_decoder_get_seq_len.argtypes = [C.c_void_p]
    L.matmul_decoder_prefill_batch.argtypes = [C.c_void_p, F32P, C.c_int]
    L.mdx_prefill_logits.argtypes = [C.c_void_p, F32P, C.c_int, F32P]
    L.mdx_time_prefill.argtypes = [C.c_void_p, F32P, C.c_int, C.c_int, F32P]
    return L


def _decoder(fake, mdx, workdir, max_seq, **over):
    cfg, d = tiny_config(mdx, max_seq_len=max_seq, num_layers=1, **over)
    path = os.path.join(workdir, "fake_%d" % cfg.head_dim)
    if not os.path.isdir(path):
        mdx.write_model(path, cfg, 0, 9)
    fake.fake_reset()
    h = fake.matmul_decoder_create(path.encode(), C.byref(cfg), 0, max_seq)
    assert h
    return h, d["hidden_dim"]


def _rows(n, d, first):
    e = np.zeros((n, d), np.float32)
    e[:, 0] = first + np.arange(n)
    return e, e.ctypes.data_as(F32P)


# rows, max_batch_prefill -> the rows of each pass: long prompts in equal
# passes of up to 2048, whose pieces go round the upload ring up to four times;
# up to 64 rows and a smaller max_batch_prefill in chunks
@pytest.mark.parametrize("head_dim", [64, 256])
@pytest.mark.parametrize("n,chunk,passes", [(65, 64, [65]), (2048, 64, [2048]), (2049, 0, [1025, 1024]), (5000, 64, [1667, 1667, 1666]),
                                            (64, 64, [64]), (70, 16, [16, 16, 16, 16, 6]), (5, 16, [5])])
def test_passes(fake, mdx, workdir, n, chunk, passes, head_dim):
    h, d = _decoder(fake, mdx, workdir, 6000, max_batch_prefill=chunk, head_dim=head_dim)
    logits = np.zeros(512, np.float32)
    try:
        for start in (0, n) if 2 * n <= 6000 else (0,):       # the second prompt behind the first
            fake.fake_reset()
            emb, p = _rows(n, d, 10.0 + start)
            assert fake.mdx_prefill_logits(h, p, n, logits.ctypes.data_as(F32P)) >= 0
            assert fake.matmul_decoder_get_seq_len(h) == start + n and fake.fake_pending() == 0
            got = np.ctypeslib.as_array((C.c_float * n).in_dll(fake, "fake_rows"))
            assert C.c_int.in_dll(fake, "fake_n_rows").value == n and np.array_equal(got, emb[:, 0])
            pos = list((C.c_int * 64).in_dll(fake, "fake_pos"))[:C.c_int.in_dll(fake, "fake_n_pos").value]
            assert pos == [start + sum(passes[:i]) for i in range(len(passes))]
            assert C.c_int.in_dll(fake, "fake_copied_row").value == passes[-1] - 1
            assert logits[0] == emb[n - 1, 0]
    finally:
        fake.matmul_decoder_destroy(h)


@pytest.mark.parametrize("n,ok", [(70, 0), (70, 1), (20, 0), (20, 1)])
def test_failed_call_leaves_nothing_running(fake, mdx, workdir, n, ok):
    """A signal that cannot be issued, behind the prompt (ok 0) or the head
    (1): the call fails with the device idle, so the next one may reuse the
    pinned buffers, and works."""
    h, d = _decoder(fake, mdx, workdir, 256)
    logits = np.zeros(512, np.float32)
    lp = logits.ctypes.data_as(F32P)
    try:
        emb, p = _rows(n, d, 3.0)
        C.c_int.in_dll(fake, "fake_fail_signal").value = ok
        assert fake.mdx_prefill_logits(h, p, n, lp) < 0
        assert fake.fake_pending() == 0
        C.c_int.in_dll(fake, "fake_fail_signal").value = -1
        fake.matmul_decoder_clear_kv_cache(h)
        assert fake.mdx_prefill_logits(h, p, n, lp) >= 0 and logits[0] == emb[-1, 0]
    finally:
        fake.matmul_decoder_destroy(h)


def test_split_partials_of_long_prompts(mdx):
    """The partials' scratch holds every launch of up to M rows and little more
    (hidden 1024, passes of 2048 rows: 8.4 MB)."""
    need = mdx.lib().mdx_long_scratch_floats
    need.restype = C.c_size_t
    assert need(2048, 1024) * 4 <= 8.5e6
    for N in (32, 160, 1024, 1536, 2048, 5120, 16384):
        for M in (65, 127, 128, 203, 515, 1000, 1024, 2000, 2048):
            for m in (1, 64, M // 2, M - 1, M):
                # 128 x 128 tiles from 256 of them on, else 64 x 64; up to 8 splits while there are fewer than 512 blocks
                t = 128 if -(-m // 128) * -(-N // 128) >= 256 else 64
                splits = max(1, min(8, 512 // (-(-m // t) * -(-N // t))))
                assert need(M, N) >= splits * m * N, (M, N, m)


def test_timed_prefill_is_what_callers_run(fake, mdx, workdir):
    """mdx_time_prefill issues what matmul_decoder_prefill_batch issues, over and
    over at the same position, and no graph that callers never replay."""
    h, d = _decoder(fake, mdx, workdir, 256)
    ms = C.c_float()
    try:
        emb, p = _rows(20, d, 5.0)
        assert fake.matmul_decoder_prefill_batch(h, p, 20) == 0
        fake.fake_reset()
        graphs = C.c_int.in_dll(fake, "fake_graphs").value
        assert fake.mdx_time_prefill(h, p, 20, 3, C.byref(ms)) == 0 and ms.value > 0
        assert C.c_int.in_dll(fake, "fake_graphs").value == graphs
        got = np.ctypeslib.as_array((C.c_float * 60).in_dll(fake, "fake_rows"))
        assert C.c_int.in_dll(fake, "fake_n_rows").value == 60 and np.array_equal(got, np.tile(emb[:, 0], 3))
        assert list((C.c_int * 3).in_dll(fake, "fake_pos")) == [20, 20, 20]
        assert fake.matmul_decoder_get_seq_len(h) == 20 and fake.fake_pending() == 0
    finally:
        fake.matmul_decoder_destroy(h)
