"""Page-table updates that went into a recording (kv_pages.hpp): they reach the
device table only when the recording runs, so they stay to be done for every
call before that, and again after each replay.  On the CPU, the bookkeeping
alone (tests/c/kv_pages_recorded.cpp); on the GPU, the calls that read the
device table after a dropped recording and after an old one is replayed."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from hymt2sharp_amd import F16, F32, HipBackend
from tests.attn_cases import BASE, D, EPS, HKV, HQ, cache_rows, new_token

HERE = os.path.dirname(os.path.abspath(__file__))


def test_changed_entries_across_recordings(tmp_path):
    cxx = shutil.which("g++")
    if not cxx or os.environ.get("HYMT_SANITIZED_CHILD") == "1":
        pytest.skip("no g++, or the preloaded sanitizer would reach it")
    exe = tmp_path / "kv_pages_recorded"
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", "-o", str(exe),
                    os.path.join(HERE, "c", "kv_pages_recorded.cpp")], check=True)
    assert subprocess.run([str(exe)]).returncode == 0


def steps(dtype, record):
    """Decode at 320 (which maps page 5) and 321 over 320 cached rows, and the
    cache read back; with `record`, after a recording of the first was dropped."""
    kb, vb = cache_rows(23, 320)
    q, k, v, qnw, knw = new_token(23, 1, "gamma", seq=2)
    be = HipBackend(0).configure(HQ, HKV, D, D, BASE, EPS).create_cache(1, 640, dtype)
    try:
        be.UploadKv(0, 0, 320, kb, vb)
        if record:
            ptrs = []
            for a in (q, k, v, qnw, knw):
                ptrs.append(be.alloc(a.nbytes))
                be.upload(ptrs[-1], a)
            out = be.alloc(q.nbytes)
            be.graph_begin()
            be.decode_dev(0, 320, *ptrs, out)
            g = be.graph_end()
            be.graph_destroy(g)
        outs = [be.DecodeAttention(0, 320 + i, q[i], k[i], v[i], qnw, knw) for i in range(2)]
        return outs + list(be.ReadKv(0, 0, 322))
    finally:
        be.Dispose()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F16, F32])
def test_dropped_recording(hip_available, dtype):
    for a, b in zip(steps(dtype, True), steps(dtype, False)):
        assert np.array_equal(a, b)


@pytest.mark.gpu
def test_replay_after_the_table_moved_on(hip_available):
    """A replay writes the page it was recorded with into the device table; the
    next call that reads the table reads the live one."""
    kb, vb = cache_rows(24, 384)
    q, k, v, qnw, knw = new_token(24, 1, "gamma")
    be = HipBackend(0).configure(HQ, HKV, D, D, BASE, EPS).create_cache(1, 640, F16)
    try:
        be.UploadKv(0, 0, 256, kb, vb)
        be.ReadKv(0, 0, 128)  # its buffer: one allocated later would void the recording
        ptrs = []
        for a in (q, k, v, qnw, knw):
            ptrs.append(be.alloc(a.nbytes))
            be.upload(ptrs[-1], a)
        out = be.alloc(q.nbytes)
        be.graph_begin()
        be.decode_dev(0, 256, *ptrs, out)  # maps page 4
        g = be.graph_end()
        be.graph_launch(g)
        recorded = be.page_of(4)
        be.SetCacheLen(192)
        be.MapRange(192, 64)  # block 3 takes the page block 4 had, so block 4 gets another
        be.UploadKv(0, 192, 192, kb, vb)
        assert be.page_of(4) != recorded
        want = be.ReadKv(0, 256, 128)
        be.graph_launch(g)  # its row goes to the recorded page, which is block 3's now
        be.sync()
        for a, b in zip(be.ReadKv(0, 256, 128), want):
            assert np.array_equal(a, b)
        be.graph_destroy(g)
    finally:
        be.Dispose()


@pytest.mark.gpu
def test_replay_after_another_replay(hip_available):
    """The page that one recording's replay writes into the device table is not
    what the next one reads there."""
    kb, vb = cache_rows(25, 320)
    q, k, v, qnw, knw = new_token(25, 1, "gamma", seq=64)
    be = HipBackend(0).configure(HQ, HKV, D, D, BASE, EPS).create_cache(1, 640, F16)
    try:
        be.UploadKv(0, 0, 256, kb, vb)
        be.ReadKv(0, 0, 128)
        ptrs = []
        for a in (q, k, v, qnw, knw):
            ptrs.append(be.alloc(a.nbytes))
            be.upload(ptrs[-1], a)
        out = be.alloc(q.nbytes)

        def chunk():
            be.prefill_dev(0, 256, 64, *ptrs[:3], F32, *ptrs[3:], out)

        chunk()  # its workspace; maps page 4
        be.SetCacheLen(256)
        be.graph_begin()
        be.decode_dev(0, 256, *ptrs, out)  # maps page 4
        g1 = be.graph_end()
        recorded = be.page_of(4)
        be.SetCacheLen(192)
        be.MapRange(192, 64)
        be.UploadKv(0, 192, 64, kb, vb)
        chunk()  # block 4 has another page
        assert be.page_of(3) == recorded
        be.graph_begin()
        chunk()
        g2 = be.graph_end()
        want = be.ReadKv(0, 256, 64)
        be.graph_launch(g1)          # a row of block 4 into block 3's page: undone by the upload
        be.sync()
        be.UploadKv(0, 192, 64, kb, vb)
        three = be.ReadKv(0, 192, 64)
        be.upload(ptrs[1], np.zeros_like(k))
        be.upload(ptrs[2], np.zeros_like(v))
        be.graph_launch(g1)
        be.graph_launch(g2)          # block 4's own page, rows of 0
        be.sync()
        four = be.ReadKv(0, 256, 64)
        assert not four[1].any() and want[1].any()
        now = be.ReadKv(0, 192, 64)
        assert np.array_equal(now[0][1:], three[0][1:]) and np.array_equal(now[1][1:], three[1][1:])
        be.graph_destroy(g1)
        be.graph_destroy(g2)
    finally:
        be.Dispose()
