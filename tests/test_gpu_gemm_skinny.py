"""The short-prompt GEMM (hymt2sharp_amd/csrc/gemm_skinny.hip): every tile of
its family at its token and width edges through hymt_gemm, against the fp64
product (the bounds of test_gpu_gemm_mfma.py: fp32 sums within 1e-5 of
sum |x w|), and the fused gate/up + SwiGLU against the two calls it replaces,
bit for bit."""
import numpy as np
import pytest

from tests.test_gpu_gemm_mfma import MFMA, check, run_case
from tests.test_gpu_gemm_swiglu import fused_and_composed

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def default_choice(monkeypatch):
    monkeypatch.delenv("HYMT_HIP_GEMM", raising=False)
    monkeypatch.delenv("HYMT_HIP_GEMM_TILE", raising=False)


@pytest.mark.parametrize("rows,cols,m", [
    (128, 2048, 1), (2048, 2048, 16),                      # 16 x 16
    (128, 2048, 17), (2048, 6144, 33), (2048, 8192, 64),   # 16 x 32 once 16 x 16 passes 256 workgroups
    (12288, 2048, 1), (12288, 2048, 16),                   # 48 x 16
    (3072, 2048, 33), (2048, 2048, 128),                   # 32 x 32
    (12288, 2048, 17), (3072, 2048, 128),                  # 48 x 32
    (2048, 6144, 129), (2048, 2048, 256),                  # 32 x 64
    (12288, 2048, 64), (3072, 4096, 256),                  # 48 x 64
    (2048, 2048, 257), (2048, 6144, 448),                  # 64 x 64
    (12288, 2048, 65), (3072, 2048, 511),                  # 96 x 64
    (2048, 2048, 513), (2048, 6144, 768),                  # 64 x 96, its last token count
    (2048, 2048, 769),                                     # past it: the 128-wide tiles
])
def test_tiles_and_edges(hip_available, rows, cols, m):
    out, counts, ref, mag, y0 = run_case(rows, cols, m, 6000 + rows + cols + m, MFMA)
    check(out, ref, mag, y0)
    assert counts == {"gemm_mfma_out_f32": 2, "gemm_mfma_out_bf16": 1}


def test_bits_do_not_depend_on_the_tile(hip_available):
    """The rows of a prompt give the same bits alone (a smaller tile) and as
    part of a longer one: k is split the same way in every tile."""
    whole, _, _, _, _ = run_case(256, 2048, 1, 11, MFMA)
    for m in (17, 100, 400):  # run_case draws x row by row from the seed: row 0 is the same
        part, _, _, _, _ = run_case(256, 2048, m, 11, MFMA)
        assert np.array_equal(part["f32"][:1], whole["f32"]), m
        assert np.array_equal(part["bf16"][:1], whole["bf16"]), m


@pytest.mark.parametrize("f,k,m,separate", [
    (6144, 2048, 65, False),    # 96 x 64
    (6144, 2048, 128, False),
    (6144, 2048, 256, True),    # the unfused calls, 6144 rows each, on 96 x 64; the fused one on the same k parts
    (1536, 2048, 512, False),   # 96 x 64 over 3072 rows
])
def test_fused_equals_composed(hip_available, f, k, m, separate):
    fused, composed = fused_and_composed(f, k, m, 40 + m, separate)
    assert fused is not None
    assert np.array_equal(fused, composed)


@pytest.mark.parametrize("m", [2, 16, 33, 64])
def test_short_prompt_lengths_stay_refused(hip_available, m):
    """hymt_gemm_swiglu refuses the lengths whose plan splits k, as before
    (the model's prefill fuses them itself)."""
    fused, _ = fused_and_composed(6144, 2048, m, 3)
    assert fused is None
