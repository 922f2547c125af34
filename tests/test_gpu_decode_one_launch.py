"""Decode attention over a short cache, which one launch serves: positions at
the page edges, at the edges between its forms (one or two pages a wave group,
then the split form with its merge), against the oracle with the bars of
test_gpu_decode.py; every head and dim slice, the appended row and a cache
whose pages are not in order."""
import numpy as np
import pytest

from hymt2sharp_amd import HipBackend
from hymt2sharp_amd import synth as S
from hymt2sharp_amd._native import BF16, F16, F32, ArgumentError
from tests.attn_cases import BASE, D, EPS, HKV, HQ, cache_rows, max_rel, new_token
from tests.test_gpu_random_sweep import decode_case
from tests.test_gpu_decode import ulp_close
from tests.test_gpu_graph import dev_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [F32, F16, BF16])
@pytest.mark.parametrize("pos", [1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 256, 257, 383, 511, 512, 513, 576])
def test_short_cache(oracle, hip_available, dtype, pos):
    got, ref, (kd, vd), (kr, vr) = decode_case(oracle, dtype, pos, "gamma", config=17, salt=pos)
    assert max_rel(got, ref) <= 1e-3
    assert ulp_close(kd, kr, dtype) and ulp_close(vd, vr, dtype)


@pytest.mark.parametrize("dtype,last", [(F32, 192), (F16, 512), (BF16, 512)])
def test_one_launch_up_to(hip_available, dtype, last):
    """No merge follows up to `last` cached positions; one does from the next."""
    q, k, v, qnw, knw = new_token(17, 9, "gamma")
    be = HipBackend(0).configure(HQ, HKV, D, D, BASE, EPS).create_cache(1, 640, dtype)
    try:
        be.MapRange(0, 640)
        ptrs = dev_inputs(be, [q, k, v, qnw, knw])
        out = be.alloc(q.nbytes)
        be.timing_enable(2)
        for n, pos in enumerate((1, 64, 65, 130, last), 1):
            be.decode_dev(0, pos, *ptrs, out)
            be.sync()
            assert be.timing("decode_attn")[0] == n
        with pytest.raises(ArgumentError):  # none was timed
            be.timing("decode_merge")
        be.decode_dev(0, last + 1, *ptrs, out)
        be.sync()
        assert be.timing("decode_merge")[0] == 1
    finally:
        be.Dispose()


@pytest.mark.parametrize("kv_heads", [1, 2, 8])
@pytest.mark.parametrize("dtype,pos", [(F32, 190), (F16, 100), (BF16, 400)])
def test_other_kv_head_counts(oracle, hip_available, dtype, pos, kv_heads):
    """The first kv heads of the usual inputs, or those twice over."""
    def cut(a, per):  # per: heads for each kv head
        return np.ascontiguousarray(np.concatenate([a, a], 1)[:, :per * kv_heads * D])
    kb, vb = (cut(a, 1) for a in cache_rows(19, pos))
    q, k, v, qnw, knw = new_token(19, 0, "gamma")
    q, k, v = cut(q, 4), cut(k, 1), cut(v, 1)
    be = HipBackend(0).configure(4 * kv_heads, kv_heads, D, D, BASE, EPS).create_cache(1, 640, dtype)
    try:
        be.UploadKv(0, 0, pos, kb, vb)
        got = be.DecodeAttention(0, pos, q[0], k[0], v[0], qnw, knw)
    finally:
        be.Dispose()
    caches = []
    for b in (kb, vb):
        caches.append(oracle.new_cache(640, kv_heads, D, dtype))
        caches[-1][:pos] = oracle.to_storage(S.bf16_bits_to_f32(b), dtype)
    ref = oracle.decode_attention(q[0], k[0], v[0], qnw, knw, *caches, dtype, 4 * kv_heads, kv_heads, D, BASE, EPS, pos)
    assert max_rel(got, ref) <= 1e-3


@pytest.mark.parametrize("dtype,rope_dim", [(F16, 64), (BF16, 2), (F32, 0)])
def test_short_cache_partial_rotary(oracle, hip_available, dtype, rope_dim):
    for pos in (100, 180):
        got, ref, _, _ = decode_case(oracle, dtype, pos, "gamma", config=17, salt=pos, rope_dim=rope_dim)
        assert max_rel(got, ref) <= 1e-3


@pytest.mark.parametrize("dtype", [F16, F32])
def test_pages_out_of_order(hip_available, dtype):
    """The same rows give the same bits whatever physical pages hold them."""
    outs = []
    for shuffle in (False, True):
        kb, vb = cache_rows(17, 160, salt=3)
        q, k, v, qnw, knw = new_token(17, 3, "gamma")
        be = HipBackend(0).configure(HQ, HKV, D, D, BASE, EPS).create_cache(1, 640, dtype)
        try:
            if shuffle:  # map far blocks first, then give them back: the free list hands out others
                be.MapRange(0, 640)
                be.SetCacheLen(64)
                be.MapRange(320, 64)
            be.UploadKv(0, 0, 160, kb, vb)
            pages = [be.page_of(b) for b in range(3)]
            outs.append((pages, be.DecodeAttention(0, 160, q[0], k[0], v[0], qnw, knw)))
        finally:
            be.Dispose()
    assert outs[0][0] != outs[1][0]
    assert np.array_equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("dtype,pos", [(F32, 180), (F16, 180), (BF16, 350), (F16, 500)])
def test_replay_keeps_its_pages(hip_available, dtype, pos):
    """A recorded call takes the page of every run from its arguments: the
    table may have moved on by the time it is replayed."""
    kb, vb = cache_rows(17, pos, salt=5)
    q, k, v, qnw, knw = new_token(17, 5, "gamma")
    be = HipBackend(0).configure(HQ, HKV, D, D, BASE, EPS).create_cache(1, 640, dtype)
    try:
        be.UploadKv(0, 0, pos, kb, vb)
        ptrs = dev_inputs(be, [q, k, v, qnw, knw])
        dout = be.alloc(q.nbytes)

        def out():
            be.sync()
            return be.download(np.empty(HQ * D, np.float32), dout)

        be.decode_dev(0, pos, *ptrs, dout)
        eager = out()
        be.graph_begin()
        be.decode_dev(0, pos, *ptrs, dout)
        g = be.graph_end()
        pages = [be.page_of(b) for b in range(pos // 64 + 1)]
        be.SetCacheLen(64)                # blocks 1 and up give their pages back
        be.MapRange(64, pos + 1 - 64)     # and get them again, the last given back first
        assert [be.page_of(b) for b in range(pos // 64 + 1)] == pages[:1] + pages[:0:-1]
        be.upload(dout, np.zeros_like(q))
        be.graph_launch(g)
        assert np.array_equal(out(), eager)
        be.graph_destroy(g)
    finally:
        be.Dispose()


@pytest.mark.parametrize("dtype,pos", [(F32, 150), (F16, 70), (BF16, 300), (F16, 512)])
def test_output_in_place_of_q(hip_available, dtype, pos):
    """out may be the q buffer: the call then writes it after every read."""
    kb, vb = cache_rows(17, pos, salt=7)
    q, k, v, qnw, knw = new_token(17, 7, "gamma")
    be = HipBackend(0).configure(HQ, HKV, D, D, BASE, EPS).create_cache(1, 640, dtype)
    try:
        be.UploadKv(0, 0, pos, kb, vb)
        ptrs = dev_inputs(be, [q, k, v, qnw, knw])
        dout = be.alloc(q.nbytes)
        outs = []
        for d in (dout, ptrs[0]):
            be.decode_dev(0, pos, *ptrs, d)
            be.sync()
            outs.append(be.download(np.empty(HQ * D, np.float32), d))
    finally:
        be.Dispose()
    # two forms of the same sums: q and P enter the MFMA in 16-bit pairs
    assert max_rel(outs[1], outs[0]) <= 1e-3
