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


# features x tokens of the family's tiles, smallest first, in blocks of 16
TILES = [(1, 1), (1, 2), (3, 1), (2, 2), (3, 2), (2, 4), (3, 4), (4, 4), (6, 4), (4, 6)]


def tile(rows, m):
    """The first tile that makes at most one round of 256 workgroups."""
    for a, b in TILES:
        if rows % (16 * a) == 0 and rows // (16 * a) * -(-m // (16 * b)) <= 256:
            return a, b
    return None


@pytest.mark.parametrize("rows,cols,m,want", [
    (128, 2048, 1, (1, 1)), (2048, 2048, 16, (1, 1)), (128, 2048, 17, (1, 1)),
    (2048, 6144, 33, (1, 2)), (2048, 8192, 64, (1, 2)),
    (12288, 2048, 1, (3, 1)), (12288, 2048, 16, (3, 1)), (3072, 2048, 33, (3, 1)),
    (2048, 2048, 65, (2, 2)), (2048, 2048, 128, (2, 2)),
    (12288, 2048, 17, (3, 2)), (3072, 2048, 128, (3, 2)),
    (2048, 6144, 129, (2, 4)), (2048, 2048, 256, (2, 4)),
    (12288, 2048, 64, (3, 4)), (3072, 4096, 256, (3, 4)),
    (2048, 2048, 257, (4, 4)), (2048, 6144, 448, (4, 4)),
    (12288, 2048, 65, (6, 4)), (3072, 2048, 511, (6, 4)),
    (2048, 2048, 513, (4, 6)), (2048, 6144, 768, (4, 6)),  # its last token count
    (2048, 2048, 769, None),                               # past it: the 128-wide tiles
])
def test_tiles_and_edges(hip_available, monkeypatch, rows, cols, m, want):
    assert tile(rows, m) == want
    out, counts, ref, mag, y0 = run_case(rows, cols, m, 6000 + rows + cols + m, MFMA)
    check(out, ref, mag, y0)
    assert counts == {"gemm_mfma_out_f32": 2, "gemm_mfma_out_bf16": 1}
    # which kernel it was: k in four parts here, whole in an unsplit tile of the
    # other, whose tiles all give the same bits
    monkeypatch.setenv("HYMT_HIP_GEMM_TILE", "128x64")
    other, _, _, _, _ = run_case(rows, cols, m, 6000 + rows + cols + m, MFMA)
    assert np.array_equal(out["f32"], other["f32"]) == (want is None)


@pytest.mark.parametrize("rows,lengths", [(2048, [33, 100, 200, 400, 700]), (3072, [20, 50, 100, 200, 300, 500])])
def test_bits_do_not_depend_on_the_tile(hip_available, rows, lengths):
    """The rows of a prompt give the same bits alone (the smallest tile) and as
    part of a longer one: k is split the same way in every tile."""
    whole, _, _, _, _ = run_case(rows, 2048, 1, 11, MFMA)
    for m in lengths:  # run_case draws x row by row from the seed: row 0 is the same
        part, _, _, _, _ = run_case(rows, 2048, m, 11, MFMA)
        assert np.array_equal(part["f32"][:1], whole["f32"]), m
        assert np.array_equal(part["bf16"][:1], whole["bf16"]), m


def test_every_tile_is_compared():
    seen = {tile(2048, m) for m in (1, 33, 100, 200, 400, 700)} | {tile(3072, m) for m in (20, 50, 100, 200, 300, 500)}
    assert seen == set(TILES)


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
