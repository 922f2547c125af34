"""The split of a prefill's kv range over work items, at the lengths where its
rule changes: 305 rows and up (the same number of items for every block pair,
chosen by cost), long caches under that (as many as fill one round of the
chip), the last row counts with two items per pair and the first
with one.  Against the
oracle, to the bounds of test_gpu_prefill.py."""
import numpy as np
import pytest

from hymt2sharp_amd import HipBackend
from hymt2sharp_amd._native import BF16, F16, ArgumentError
from tests.attn_cases import BASE, D, EPS
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


@pytest.mark.parametrize("kv_heads,seq,merges", [(4, 992, 1), (4, 993, 0), (4, 1024, 0), (8, 480, 1), (8, 512, 0),
                                                 (2, 1984, 1), (2, 2048, 0)])
def test_128_pairs_stay_whole(hip_available, kv_heads, seq, merges):
    """From 128 (block pair, kv head) items on a call keeps every sum in fp32
    to its output: no partial in the cache type, no merge, and so no workspace
    that a first call under recording would have to grow."""
    be = HipBackend(0).configure(4 * kv_heads, kv_heads, D, D, BASE, EPS).create_cache(1, 6144 + seq, BF16)
    try:
        be.MapRange(0, 6144 + seq)
        bufs = [be.alloc(n) for n in (seq * 4 * kv_heads * D * 2, seq * kv_heads * D * 2, seq * kv_heads * D * 2,
                                      seq * 4 * kv_heads * D * 4)]
        for b, n in zip(bufs, (4, 1, 1, 8)):
            be.upload(b, np.zeros(seq * n * kv_heads * D, np.uint16))

        def call():
            be.prefill_dev(0, 6144, seq, *bufs[:3], BF16, None, None, bufs[3])

        if not merges:
            be.graph_begin()
            call()
            be.graph_destroy(be.graph_end())
        be.timing_enable(2)
        call()
        be.sync()
        assert be.timing("prefill_flash")[0] == 1
        try:
            count = be.timing("prefill_merge")[0]
        except ArgumentError:  # none was timed
            count = 0
        assert count == merges
    finally:
        be.Dispose()
