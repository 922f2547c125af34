"""The Q4_K GEMV on the matrix cores (hymt2sharp_amd/csrc/gemv.hip,
gemv_kq_kernel): every form of its dispatch (waves over 2048 to 8192 columns,
one or two 16-row tiles a workgroup), row counts that do not fill a tile,
the input and output modes, and inputs of extreme range, against the fp64
product of the dequantized weights.

Bound: x' enters exactly, the products are summed in integers and with the
minima in fp64; what remains is fp32, a rounding of each wave's share of a row
and their sum: under 16 roundings of 2^-24 on terms that add up to sum |w x|,
1e-6 of it.  The norm's factor and the sigmoid, and super-blocks that take fp32
products (values 2^36 apart), add a few more: 4e-6."""
import numpy as np
import pytest

from hymt2sharp_amd import HipBackend
from hymt2sharp_amd import _native as N
from hymt2sharp_amd import synth as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def run(rows, cols, x, seed, y0=None, **kw):
    raw = S.random_weight(seed, N.W_Q4_K, rows, cols)
    W = O.dequant(N.W_Q4_K, raw, rows, cols).astype(np.float64)
    outs = rows // 2 if kw.get("swiglu_out") else rows
    gamma = kw.pop("gamma", None)
    be = HipBackend(0)
    try:
        w = be.weight_upload(N.W_Q4_K, rows, cols, raw)
        dx, dy = be.alloc(4 * x.size), be.alloc(4 * outs)
        be.upload(dx, x)
        be.upload(dy, np.zeros(outs, np.float32) if y0 is None else y0)
        dg = None
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
    assert np.all(np.abs(y - ref) <= 4e-6 * mag), float(np.max(np.abs(y - ref) / mag))


@pytest.mark.parametrize("cols", [2048, 4096, 6144, 8192])
@pytest.mark.parametrize("rows", [1, 16, 17, 250, 8192, 8200])
def test_tiles_and_waves(hip_available, rows, cols):
    rng = np.random.default_rng(rows + cols)
    x, y0 = rng.standard_normal(cols).astype(np.float32), rng.standard_normal(rows).astype(np.float32)
    W, y = run(rows, cols, x, 5, y0, accumulate=True)
    close(y, W @ x + y0, np.abs(W) @ np.abs(x) + np.abs(y0))


@pytest.mark.parametrize("F", [1, 15, 16, 40, 8208])
def test_norm_and_swiglu_output(hip_available, F):
    """[gate; up] with F rows each: gate and up rows need not start a tile."""
    rng = np.random.default_rng(F)
    x, g = rng.standard_normal(2048).astype(np.float32), rng.uniform(0.9, 1.1, 2048).astype(np.float32)
    W, y = run(2 * F, 2048, x, 6, gamma=g, swiglu_out=True)
    xn = x.astype(np.float64) / np.sqrt(np.mean(x.astype(np.float64) ** 2) + 1e-6) * g
    gt, up, mg, mu = W[:F] @ xn, W[F:] @ xn, np.abs(W[:F]) @ np.abs(xn), np.abs(W[F:]) @ np.abs(xn)
    with np.errstate(over="ignore"):
        sig = 1.0 / (1.0 + np.exp(-gt))
    ref = gt * sig * up
    # |d silu| <= 1.1; the exponential's argument is a sum of magnitude mg
    mag = 1.1 * mg * np.abs(up) + np.abs(gt * sig) * mu + 0.3 * np.abs(ref)
    close(y, ref, mag)


@pytest.mark.parametrize("cols", [2048, 6144])
def test_swiglu_input(hip_available, cols):
    rng = np.random.default_rng(cols)
    gu = rng.standard_normal(2 * cols).astype(np.float32)
    W, y = run(100, cols, gu, 7, swiglu=True)
    g = gu[:cols].astype(np.float64)
    x = g / (1.0 + np.exp(-g)) * gu[cols:]
    close(y, W @ x, np.abs(W) @ np.abs(x))


@pytest.mark.parametrize("kind", ["zero", "tiny", "huge", "outlier", "mixed"])
def test_range(hip_available, kind):
    rng = np.random.default_rng(9)
    x = rng.standard_normal(2048)
    if kind == "zero":
        x[:] = 0
    elif kind == "tiny":
        x *= 1e-36
    elif kind == "huge":
        x *= 1e33
    elif kind == "outlier":
        x[rng.integers(0, 2048, 5)] *= 3e4
    else:  # a different magnitude for every super-block
        x *= np.repeat(10.0 ** np.arange(-16, 16, 4), 256)
    x = x.astype(np.float32)
    W, y = run(48, 2048, x, 8)
    x = x.astype(np.float64)
    if kind == "zero":
        assert np.all(y == 0)
    else:
        close(y, W @ x, np.abs(W) @ np.abs(x))


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_non_finite_input_shows(hip_available, bad):
    x = np.random.default_rng(3).standard_normal(2048).astype(np.float32)
    x[777] = bad
    _, y = run(32, 2048, x, 8)
    assert not np.any(np.isfinite(y))
