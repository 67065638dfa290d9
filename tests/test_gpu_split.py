"""Projections on the f16 matrix cores by the two-way split (split_gemm.h),
at the edges of its tiles, row scales and values, against float64.

Bound per element: each operand is held to 2^-23 of itself and the lo.lo
product (2^-22) is dropped, 2^-21 together, and each of the K / 4 additions
inside and between the matrix instructions rounds or truncates by at most
2^-23 of the running sum of |x w|; a value below 2^-18 of its row's largest
is held to 2^-40 of that instead.
"""
import numpy as np
import pytest

from vestra_hip import seeded

pytestmark = pytest.mark.gpu


def _bound(x, w):
    k = x.shape[1]
    ax, aw = np.abs(x).astype(np.float64), np.abs(w).astype(np.float64)
    small = 2.0 ** -39 * (ax.max(1, keepdims=True) * aw.sum(0) + ax.sum(1, keepdims=True) * aw.max(0))
    return (2.0 ** -21 + k / 4 * 2.0 ** -23) * (ax @ aw) + small


# One row; ragged rows, columns and K on every tile (64 x 32, 64 x 64, 64 x
# 128, 128 x 96, 128 x 128, 128 x 256), K of 2, 3 and an odd count of slices.
SHAPES = [(1, 64, 1), (65, 64, 33), (63, 70, 95), (97, 96, 770), (257, 101, 771), (500, 768, 768),
          (865, 768, 2304), (865, 100, 3074), (1153, 1003, 771), (1800, 416, 1500), (3460, 768, 2307)]


@pytest.mark.parametrize("m, k, n", SHAPES)
def test_split_gemm_edges_vs_float64(rt, m, k, n):
    x = seeded.normal(9000 + m, m * k).reshape(m, k)
    w = seeded.normal(9100 + n, k * n, 0.05).reshape(k, n)
    b = seeded.normal(9200, n)
    g = (0.1 + 0.9 * seeded.uniform01(9300, n)).astype(np.float32)
    ref = x.astype(np.float64) @ w.astype(np.float64)
    bound = _bound(x, w)
    xt = rt.upload_f32(x)
    got = rt.download_f32(rt.gemm_row_major_f32(xt, rt.upload_f32(w), m, k, n)).reshape(m, n)
    assert np.all(np.abs(got - ref) <= bound)
    lin = rt.prepare_linear_f32(k, n, w, b, g)
    exp = (ref + b) * g
    bound = bound * g + 2.0 ** -22 * (np.abs(ref) + np.abs(b)) * g
    assert np.all(np.abs(rt.download_f32(lin.run(xt, m)).reshape(m, n) - exp) <= bound)
    assert np.all(np.abs(rt.download_f32(lin.run_chw(xt, m)).reshape(n, m).T - exp) <= bound)
    r = seeded.normal(9400, m * n).reshape(m, n)
    rs = rt.upload_f32(r)
    lin.run_residual(xt, m, rs)
    assert np.all(np.abs(rt.download_f32(rs).reshape(m, n) - (r + exp)) <= bound + 2.0 ** -23 * np.abs(r + exp))


def test_split_gemm_row_scales(rt):
    """Rows and columns of every magnitude: zero, subnormal, tiny, huge, and
    one outlier among ordinary values."""
    m, k, n = 70, 96, 40
    x = seeded.normal(9500, m * k).reshape(m, k)
    w = seeded.normal(9600, k * n).reshape(k, n)
    x[0] = 0.0
    x[1] *= np.float32(1e-40)
    x[2] *= np.float32(1e-30)
    x[3] *= np.float32(1e30)
    x[4, 5] = 1e6
    w[:, 1] = 0.0
    w[:, 2] *= np.float32(1e-20)
    w[:, 3] *= np.float32(1e6)
    ref = x.astype(np.float64) @ w.astype(np.float64)
    for got in (rt.gemm_row_major_f32(rt.upload_f32(x), rt.upload_f32(w), m, k, n),
                rt.prepare_linear_f32(k, n, w, np.zeros(n, np.float32)).run(rt.upload_f32(x), m)):
        got = rt.download_f32(got).reshape(m, n)
        # + half a subnormal for the result's own rounding
        assert np.all(np.abs(got - ref) <= _bound(x, w) + 2.0 ** -23 * np.abs(ref) + 2.0 ** -149)


@pytest.mark.parametrize("where", ["x", "w", "both"])
def test_split_gemm_inf_and_nan(rt, where):
    """Infinities and NaNs give what the float product gives, element by
    element, and leave the other rows and columns as they are."""
    m, k, n = 70, 96, 40
    x = seeded.normal(9700, m * k).reshape(m, k)
    w = seeded.normal(9800, k * n).reshape(k, n)
    clean = x.astype(np.float64) @ w.astype(np.float64)
    bound = _bound(x, w)
    if where != "w":
        x[3, 7], x[5, 1], x[5, 2], x[9, 0] = np.inf, np.inf, -np.inf, np.nan
    if where != "x":
        w[4, 6], w[50, 8] = -np.inf, np.nan
    with np.errstate(invalid="ignore"):
        ref = x.astype(np.float64) @ w.astype(np.float64)
    fine = np.isfinite(ref)
    for got in (rt.gemm_row_major_f32(rt.upload_f32(x), rt.upload_f32(w), m, k, n),
                rt.prepare_linear_f32(k, n, w, np.zeros(n, np.float32)).run(rt.upload_f32(x), m)):
        got = rt.download_f32(got).reshape(m, n)
        assert np.array_equal(np.isnan(got), np.isnan(ref))
        assert np.array_equal(got[~fine & ~np.isnan(ref)], ref[~fine & ~np.isnan(ref)].astype(np.float32))
        assert np.all(np.abs(got[fine] - clean[fine]) <= 2 * bound[fine])
