"""What the matrix-core GEMVs (hymt2sharp_amd/csrc/gemv.hip, gemv_kq_kernel) make
of inputs whose values lie far apart: infinities and NaN, values far below
their super-block's largest, which lose nothing to it, and sums that cancel.

Bound of the finite ones, root mean square over the rows: 2e-7 of the root mean
square of y, about 3.4 roundings of 2^-24.  fp32 products added in fp32 make
1.2e-7 to 1.6e-7 of these inputs; digits that ended 2^-30 below the largest value
made 2e-6 and more where the largest meets zero weights."""
import numpy as np
import pytest

from hymt2sharp_amd import HipBackend
from hymt2sharp_amd import _native as N
from hymt2sharp_amd import synth as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TYPES = [N.W_Q4_K, N.W_Q6_K, N.W_Q8_0]


def weights(wtype, seed, rows, cols, zero=()):
    """A random matrix and its fp64 values; the columns `zero` have weight 0 in
    every row (for Q4_K their super-blocks have no minima)."""
    raw = np.frombuffer(S.random_weight(seed, wtype, rows, cols), np.uint8).copy()
    size = {N.W_Q4_K: 144, N.W_Q6_K: 210, N.W_Q8_0: 34 * 8}[wtype]
    b = raw.reshape(rows, cols // 256, size)
    for col in zero:
        sb, j = divmod(col, 256)
        if wtype == N.W_Q8_0:
            b[:, sb, 34 * (j // 32) + 2 + j % 32] = 0
        elif wtype == N.W_Q4_K:
            b[:, sb, 2:4] = 0
            b[:, sb, 16 + 32 * (j // 64) + j % 32] &= 0x0F if j % 64 >= 32 else 0xF0
        else:  # code 32: low bits 0, high bits 2
            n, quarter, l = j // 128, j % 128 // 32, j % 32
            b[:, sb, 64 * n + 32 * (quarter & 1) + l] &= 0x0F if quarter >= 2 else 0xF0
            h = b[:, sb, 128 + 32 * n + l]
            b[:, sb, 128 + 32 * n + l] = (h & ~np.uint8(3 << 2 * quarter)) | np.uint8(2 << 2 * quarter)
    raw = raw.tobytes()
    W = O.dequant(wtype, raw, rows, cols).astype(np.float64)
    assert not W[:, list(zero)].any()
    return raw, W


def gemv(wtype, raw, rows, cols, x, **kw):
    outs = rows // 2 if kw.get("swiglu_out") else rows
    be = HipBackend(0)
    try:
        w = be.weight_upload(wtype, rows, cols, raw)
        dx, dy, dg = be.alloc(4 * x.size), be.alloc(4 * outs), None
        be.upload(dx, x)
        be.upload(dy, np.zeros(outs, np.float32))
        if "gamma" in kw:
            dg = be.alloc(4 * cols)
            be.upload(dg, kw.pop("gamma"))
        be.gemv(w, dx, dy, rmsnorm=dg, eps=1e-6, **kw)
        be.sync()
        return be.download(np.empty(outs, np.float32), dy)
    finally:
        be.Dispose()


@pytest.mark.parametrize("rows,cols", [(33, 2048), (8208, 2048), (20, 8192)])
@pytest.mark.parametrize("bad", [{777: np.inf}, {5: -np.inf}, {300: np.inf, 1999: np.inf}, {300: np.inf, 301: -np.inf},
                                 {0: np.nan}])
@pytest.mark.parametrize("wtype", TYPES)
def test_infinities_and_nan(hip_available, wtype, bad, rows, cols):
    """As the products have it: Q8_0's are code times value, Q4_K's and Q6_K's
    take an offset off afterwards, where infinity less infinity is NaN.  The
    rows' other super-blocks do not hide it."""
    raw, W = weights(wtype, 12, rows, cols)
    x = np.random.default_rng(3).standard_normal(cols).astype(np.float32)
    for c, v in bad.items():
        x[c] = v
    y = gemv(wtype, raw, rows, cols, x)
    with np.errstate(invalid="ignore"):
        want = W @ x.astype(np.float64) if wtype == N.W_Q8_0 else np.full(rows, np.nan)
    assert np.array_equal(y.astype(np.float64), want, equal_nan=True)
    if wtype == N.W_Q8_0 and len(bad) == 1:
        assert np.isinf(y).any() or np.isnan(x).any()


def rms(a):
    return float(np.sqrt(np.mean(np.square(a))))


def check(y, ref):
    err = rms(y.astype(np.float64) - ref) / rms(ref)
    assert err <= 2e-7


@pytest.mark.parametrize("scale,factor", [(1, 3e3), (1, 3e4), (1, 1e6), (1, 1e9), (1, 1e12), (1, 1e30), (1e20, 1e9),
                                          (1e-4, 1e38), (1e-20, 1e38), (1e-22, 1e57)])
@pytest.mark.parametrize("wtype", TYPES)
def test_small_values_beside_large_ones(hip_available, wtype, scale, factor):
    """One large value in each super-block, where every weight is 0: the rest is
    what is left.  From 2^36 on it is what takes the products out of integers;
    the last are 0 at the large value's scale."""
    cols = 2048
    big = list(range(7, cols, 256))
    raw, W = weights(wtype, 14, 512, cols, big)
    x = np.random.default_rng(5).standard_normal(cols) * scale
    x[big] = scale * factor
    x = x.astype(np.float32)
    check(gemv(wtype, raw, 512, cols, x), W @ x.astype(np.float64))


@pytest.mark.parametrize("cols,mode", [(2048, ""), (6144, ""), (8192, ""), (2048, "norm"), (4096, "swiglu")])
@pytest.mark.parametrize("wtype", TYPES)
def test_magnitudes_all_over(hip_available, wtype, cols, mode):
    """exp(8 N(0, 1)): within a super-block values span 2^60 and more, so some
    take each way; every 50th value is 0."""
    rng = np.random.default_rng(cols)
    x = (rng.choice([-1, 1], 2 * cols) * np.exp(8 * rng.standard_normal(2 * cols)) * 1e-6).astype(np.float32)
    x[::50] = 0
    x[cols:2 * cols:3] = 1
    raw, W = weights(wtype, 15, 512, cols)
    xd = x.astype(np.float64)
    if mode == "swiglu":
        x[:cols] = np.clip(x[:cols], -60, 60)
        xd = x.astype(np.float64)
        xd = xd[:cols] / (1 + np.exp(-xd[:cols])) * xd[cols:]
        # the sigmoid's own roundings, on every x': 1e-6 of it
        y = gemv(wtype, raw, 512, cols, x, swiglu=True).astype(np.float64)
        assert np.all(np.abs(y - W @ xd) <= 2e-6 * (np.abs(W) @ np.abs(xd)))
    elif mode == "norm":
        g = rng.uniform(0.9, 1.1, cols).astype(np.float32)
        y = gemv(wtype, raw, 512, cols, x[:cols], gamma=g)
        check(y, W @ (xd[:cols] / np.sqrt(np.mean(xd[:cols] ** 2) + 1e-6) * g))
    else:
        check(gemv(wtype, raw, 512, cols, x[:cols]), W @ xd[:cols])


@pytest.mark.parametrize("scale", [1e-30, 1e-34, 1e-36])
@pytest.mark.parametrize("wtype", TYPES)
def test_tiny_values(hip_available, wtype, scale):
    raw, W = weights(wtype, 16, 512, 2048)
    x = (np.random.default_rng(6).standard_normal(2048) * scale).astype(np.float32)
    y = gemv(wtype, raw, 512, 2048, x)
    assert np.any(y != 0)
    check(y, W @ x.astype(np.float64))


@pytest.mark.parametrize("cols", [2048, 4096, 6144, 8192])
def test_q4k_sums_that_cancel(hip_available, cols):
    """Weights spread evenly about 0 (codes times 8 d less 60 d) and inputs all
    of one sign: a row's products and its minima are each about 30 times what
    is left, and both meet the same sums of x in every row.  fp32 leaves 5e-7
    and more."""
    rows = 512
    rng = np.random.default_rng(cols)
    b = rng.integers(0, 256, (rows, cols // 256, 144), dtype=np.uint8)
    d = rng.uniform(0.001, 0.002, (rows, cols // 256)).astype(np.float16)
    b[:, :, 0:2] = b[:, :, 2:4] = d[..., None].view(np.uint8)
    b[:, :, 4:16] = [8] * 4 + [60 | 3 << 6] * 4 + [8 | 12 << 4] * 4  # 8 scales of 8, 8 minima of 60
    raw = b.tobytes()
    W = O.dequant(N.W_Q4_K, raw, rows, cols).astype(np.float64)
    assert abs(W.mean()) < 0.01 * W.std()
    x = np.abs(rng.standard_normal(cols)).astype(np.float32)
    check(gemv(N.W_Q4_K, raw, rows, cols, x), W @ x.astype(np.float64))
