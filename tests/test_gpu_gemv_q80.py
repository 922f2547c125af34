"""The Q8_0 GEMV on the matrix cores (hymt2sharp_amd/csrc/gemv.hip,
gemv_kq_kernel<kW_Q8_0>) and the tiles its upload makes: row counts that do not
fill a tile, every width, the input and output modes, values of extreme range,
and the rows read back from the tiles.

Bound of a product: x' enters exactly and a block's products are summed in
integers, so what remains is fp32: the eight blocks' scaled sums and one fma per
super-block and digit, then the partial sums, under 16 roundings of 2^-24 on
terms that add up to sum |w x|: 1e-6 of it; the norm's factor and the sigmoid add
a few more: 2e-6."""
import numpy as np
import pytest

from hymt2sharp_amd import HipBackend
from hymt2sharp_amd import _native as N
from hymt2sharp_amd import synth as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def run(rows, cols, x, seed, gamma=None, y0=None, **kw):
    raw = S.random_weight(seed, N.W_Q8_0, rows, cols)
    W = O.dequant(N.W_Q8_0, raw, rows, cols).astype(np.float64)
    outs = rows // 2 if kw.get("swiglu_out") else rows
    be = HipBackend(0)
    try:
        w = be.weight_upload(N.W_Q8_0, rows, cols, raw)
        dx, dy, dg = be.alloc(4 * x.size), be.alloc(4 * outs), None
        be.upload(dx, x)
        be.upload(dy, np.zeros(outs, np.float32) if y0 is None else y0)
        if gamma is not None:
            dg = be.alloc(4 * gamma.size)
            be.upload(dg, gamma)
        be.gemv(w, dx, dy, rmsnorm=dg, eps=1e-6, **kw)
        be.sync()
        y = be.download(np.empty(outs, np.float32), dy).astype(np.float64)
    finally:
        be.Dispose()
    return W, y


def close(y, ref, mag):
    assert np.all(np.abs(y - ref) <= 2e-6 * mag), float(np.max(np.abs(y - ref)))


@pytest.mark.parametrize("cols", [2048, 4096, 6144, 8192])
@pytest.mark.parametrize("rows", [1, 17, 250, 8200])
def test_tiles_and_waves(hip_available, rows, cols):
    rng = np.random.default_rng(rows + cols)
    x, y0 = rng.standard_normal(cols).astype(np.float32), rng.standard_normal(rows).astype(np.float32)
    W, y = run(rows, cols, x, 5, y0=y0, accumulate=True)
    close(y, W @ x + y0, np.abs(W) @ np.abs(x) + np.abs(y0))


@pytest.mark.parametrize("F,cols", [(1, 2048), (15, 2048), (40, 8192), (8208, 2048)])
def test_norm_and_swiglu_output(hip_available, F, cols):
    rng = np.random.default_rng(F)
    x, g = rng.standard_normal(cols).astype(np.float32), rng.uniform(0.9, 1.1, cols).astype(np.float32)
    W, y = run(2 * F, cols, x, 6, gamma=g, swiglu_out=True)
    xn = x.astype(np.float64) / np.sqrt(np.mean(x.astype(np.float64) ** 2) + 1e-6) * g
    gt, up, mg, mu = W[:F] @ xn, W[F:] @ xn, np.abs(W[:F]) @ np.abs(xn), np.abs(W[F:]) @ np.abs(xn)
    with np.errstate(over="ignore"):
        sig = 1.0 / (1.0 + np.exp(-gt))
    ref = gt * sig * up
    close(y, ref, 1.1 * mg * np.abs(up) + np.abs(gt * sig) * mu + np.abs(ref))


def test_swiglu_input(hip_available):
    gu = np.random.default_rng(1).standard_normal(2 * 6144).astype(np.float32)
    W, y = run(100, 6144, gu, 7, swiglu=True)
    g = gu[:6144].astype(np.float64)
    x = g / (1.0 + np.exp(-g)) * gu[6144:]
    close(y, W @ x, np.abs(W) @ np.abs(x))


@pytest.mark.parametrize("scale", [0.0, 1e-36, 1e-34, 1e-30, 1e28])
def test_range(hip_available, scale):
    x = (np.random.default_rng(9).standard_normal(2048) * scale).astype(np.float32)
    W, y = run(48, 2048, x, 8)
    x = x.astype(np.float64)
    close(y, W @ x, np.abs(W) @ np.abs(x))


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_non_finite_input_shows(hip_available, bad):
    x = np.random.default_rng(3).standard_normal(2048).astype(np.float32)
    x[777] = bad
    _, y = run(32, 2048, x, 8)
    assert not np.any(np.isfinite(y))


@pytest.mark.parametrize("rows,cols", [(1, 2048), (33, 6144), (16000, 2048)])
def test_rows_of_the_tiles(hip_available, rows, cols):
    """Dequantized rows are the oracle's values bit for bit; 16000 rows are
    uploaded in two pieces."""
    raw = S.random_weight(4, N.W_Q8_0, rows, cols)
    want = O.dequant(N.W_Q8_0, raw, rows, cols)
    be = HipBackend(0)
    try:
        w, out = be.weight_upload(N.W_Q8_0, rows, cols, raw), be.alloc(4 * cols)
        for r in {0, rows // 2, rows - 1}:
            be.embed(w, r, out)
            be.sync()
            assert np.array_equal(be.download(np.empty(cols, np.float32), out), want[r])
    finally:
        be.Dispose()
