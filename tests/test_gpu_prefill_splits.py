"""The split of a prefill's kv range over work items, at the lengths where its
rule changes: 305 rows and up (the same number of items for every block pair,
chosen by cost), long caches under that (as many as fill one round of the
chip), the last row counts with two items per pair and the first
with one.  Against the
oracle, to the bounds of test_gpu_prefill.py."""
import numpy as np
import pytest

from hymt2sharp_amd import HipBackend
from hymt2sharp_amd import synth as S
from hymt2sharp_amd._native import BF16, F16, ArgumentError
from tests.attn_cases import BASE, D, EPS, cache_rows, new_token
from tests.test_gpu_prefill import check, run_prefill

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,pos,seq", [
    (BF16, 0, 304), (BF16, 0, 305),        # either side of the row limit
    (BF16, 5, 320), (F16, 640, 310),       # unsplit; 2 items a pair
    (BF16, 1030, 512), (F16, 2048, 333),   # 3 and 5 or 6
    (BF16, 4100, 200), (F16, 3000, 290),   # under the limit, over 47 tiles: 9 and 6
    (BF16, 2900, 992), (BF16, 2900, 1024), (BF16, 2900, 1025),  # 124 pairs (2 items), 128 and 130 (unsplit)
])
def test_split_rule_edges(oracle, hip_available, dtype, pos, seq):
    got, ref, _, vf, (kd, vd), (kref, vref) = run_prefill(oracle, dtype, pos, seq, "gamma", 16, salt=pos + seq,
                                                          with_model=False)
    check(got, ref, vf, dtype)
    assert np.array_equal(vd, vref)


def merges_of(kv_heads, pos, seq, record):
    """Merge launches of one call (1: split), after a recording of it without a
    warm-up if `record`."""
    be = HipBackend(0).configure(4 * kv_heads, kv_heads, D, D, BASE, EPS).create_cache(1, pos + seq, BF16)
    try:
        be.MapRange(0, pos + seq)
        bufs = [be.alloc(n) for n in (seq * 4 * kv_heads * D * 2, seq * kv_heads * D * 2, seq * kv_heads * D * 2,
                                      seq * 4 * kv_heads * D * 4)]
        for b, n in zip(bufs, (4, 1, 1, 8)):
            be.upload(b, np.zeros(seq * n * kv_heads * D, np.uint16))

        def call():
            be.prefill_dev(0, pos, seq, *bufs[:3], BF16, None, None, bufs[3])

        if record:
            be.graph_begin()
            call()
            be.graph_destroy(be.graph_end())
        be.timing_enable(2)
        call()
        be.sync()
        assert be.timing("prefill_flash")[0] == 1
        try:
            return be.timing("prefill_merge")[0]
        except ArgumentError:  # none was timed
            return 0
    finally:
        be.Dispose()


@pytest.mark.parametrize("kv_heads,seq,merges", [(4, 992, 1), (4, 993, 0), (4, 1024, 0), (8, 480, 1), (8, 512, 0),
                                                 (2, 1984, 1), (2, 2048, 0)])
def test_128_pairs_stay_whole(hip_available, kv_heads, seq, merges):
    """From 128 (block pair, kv head) items on a call keeps every sum in fp32
    to its output: no partial in the cache type, no merge, and so no workspace
    that a first call under recording would have to grow."""
    assert merges_of(kv_heads, 6144, seq, record=not merges) == merges


@pytest.mark.parametrize("kv_heads,pos,seq,merges", [
    (1, 0, 512, 1), (1, 512, 600, 1), (2, 0, 400, 1),  # cheap partials: split already over a short cache
    (4, 0, 512, 0), (4, 2048, 512, 1),
    (8, 512, 400, 0), (8, 2048, 400, 1),               # dear ones: whole a little longer
])
def test_splits_weigh_the_kv_heads(hip_available, kv_heads, pos, seq, merges):
    assert merges_of(kv_heads, pos, seq, record=False) == merges


@pytest.mark.parametrize("kv_heads", [1, 2, 8])
@pytest.mark.parametrize("pos,seq", [(0, 512), (700, 400), (3000, 330), (3000, 200)])
def test_other_kv_head_counts(oracle, hip_available, kv_heads, pos, seq):
    """The first kv heads of the usual inputs, or those twice over."""
    def cut(a, per):  # per: heads for each kv head
        return np.ascontiguousarray(np.concatenate([a, a], 1)[:, :per * kv_heads * D])
    kb, vb = (cut(a, 1) for a in cache_rows(18, pos))
    q, k, v, qnw, knw = new_token(18, 0, "gamma", seq=seq)
    q, k, v = cut(q, 4), cut(k, 1), cut(v, 1)
    be = HipBackend(0).configure(4 * kv_heads, kv_heads, D, D, BASE, EPS).create_cache(1, pos + seq, BF16)
    try:
        if pos:
            be.UploadKv(0, 0, pos, kb, vb)
        got = be.PrefillAttention(0, pos, q, k, v, qnw, knw)
    finally:
        be.Dispose()
    caches = []
    for b in (kb, vb):
        caches.append(oracle.new_cache(pos + seq, kv_heads, D, BF16))
        caches[-1][:pos] = oracle.to_storage(S.bf16_bits_to_f32(b), BF16)
    ref = oracle.prefill_attention(q, k, v, qnw, knw, *caches, BF16, 4 * kv_heads, kv_heads, D, BASE, EPS, pos,
                                   threads=8)
    check(got, ref, oracle.from_storage(caches[1], BF16), BF16)
