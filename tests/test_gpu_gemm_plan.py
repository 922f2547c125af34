"""The GEMM plan's choice of 256 x 128 tiles (hymt2sharp_amd/csrc/gemm_mfma.hip),
at the first and last token counts where its rounds are the shorter ones: the
products against fp64, and the fused gate/up + SwiGLU against the calls it
replaces, bit for bit."""
import numpy as np
import pytest

from tests.test_gpu_gemm_mfma import MFMA, check, run_case
from tests.test_gpu_gemm_swiglu import fused_and_composed

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def default_choice(monkeypatch):
    monkeypatch.delenv("HYMT_HIP_GEMM", raising=False)
    monkeypatch.delenv("HYMT_HIP_GEMM_TILE", raising=False)


@pytest.mark.parametrize("rows,cols,m", [(12288, 2048, 513), (12288, 2048, 640), (6144, 2048, 1025)])
def test_256_x_128_rounds(hip_available, rows, cols, m):
    out, counts, ref, mag, y0 = run_case(rows, cols, m, 7000 + m, MFMA)
    check(out, ref, mag, y0)
    assert counts == {"gemm_mfma_out_f32": 2, "gemm_mfma_out_bf16": 1}


@pytest.mark.parametrize("m,separate", [(600, False), (1200, False), (1200, True)])
def test_256_x_128_fused(hip_available, m, separate):
    fused, composed = fused_and_composed(6144, 2048, m, 70 + m, separate)
    assert fused is not None
    assert np.array_equal(fused, composed)
