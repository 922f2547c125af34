"""The split of a prefill's kv range over work items, at the lengths where its
rule changes: 305 rows and up (the same number of items for every block pair,
chosen by cost), long caches under that (as many as fill one round of the
chip), the last row counts with one and with two items per pair.  Against the
oracle, to the bounds of test_gpu_prefill.py."""
import numpy as np
import pytest

from hymt2sharp_amd._native import BF16, F16
from tests.test_gpu_prefill import check, run_prefill

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,pos,seq", [
    (BF16, 0, 304), (BF16, 0, 305),        # either side of the row limit
    (BF16, 5, 320), (F16, 640, 310),       # unsplit; 2 items a pair
    (BF16, 1030, 512), (F16, 2048, 333),   # 3 and 5 or 6
    (BF16, 4100, 200), (F16, 3000, 290),   # under the limit, over 47 tiles: 9 and 6
    (BF16, 2900, 1024), (BF16, 2900, 1025),  # 128 pairs (2 items) and 130 (unsplit)
])
def test_split_rule_edges(oracle, hip_available, dtype, pos, seq):
    got, ref, _, vf, (kd, vd), (kref, vref) = run_prefill(oracle, dtype, pos, seq, "gamma", 16, salt=pos + seq,
                                                          with_model=False)
    check(got, ref, vf, dtype)
    assert np.array_equal(vd, vref)
