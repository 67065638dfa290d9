"""Projections on the f16 matrix cores by the two-way split (split_gemm.h),
at the edges of its tiles, row scales and values, against float64.

Bound per element: each operand is held to 2^-23 of itself and the lo.lo
product (2^-22) is dropped, 2^-21 together, and each of the K / 4 additions
inside and between the matrix instructions rounds or truncates by at most
2^-23 of the running sum of |x w|.  A value below 2^-18 of its row's largest
is held to 2^-40 of that instead, and what that may spoil is formed again from
the floats, so the range of a row has no term.
"""
import math

import numpy as np
import pytest

from block64 import block64
from q8_compose import q8_block
from vestra_hip import da3, seeded

pytestmark = pytest.mark.gpu


def _bound(x, w):
    k = x.shape[1]
    return (2.0 ** -21 + k / 4 * 2.0 ** -23) * (np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64))


def _launches(rt, run):
    """The names of the launches that run() makes."""
    rt.profile_reset()
    rt.profile_enable(True)
    try:
        run()
        return set(rt.profile_report())
    finally:
        rt.profile_enable(False)


# One row; ragged rows, columns and K on every tile (64 x 32, 64 x 64, 64 x
# 128, 128 x 96, 128 x 128, 128 x 192, 128 x 256), K of 3, 4 and 5 slices, even and
# odd counts, and K shared out over 2, 3 and 4 workgroups.  All of them are
# shapes that the rule (split_gemm_pays) sends to the split form.
SHAPES = [(1, 97, 1), (1, 3074, 771), (65, 65, 33), (63, 70, 95), (97, 97, 770), (257, 101, 771), (500, 770, 768),
          (865, 768, 2304), (865, 100, 3074), (1153, 1003, 771), (1800, 416, 1500), (1500, 330, 3301),
          (1031, 770, 2698), (3465, 131, 1670), (3796, 97, 1547), (3460, 768, 2307), (97, 2563, 70), (257, 3074, 768),
          (300, 2402, 500), (400, 3000, 400)]


@pytest.mark.parametrize("m, k, n", SHAPES)
def test_split_gemm_edges_vs_float64(rt, m, k, n):
    """Each element within its bound, and the 2-norm error within 1e-6 (3.6e-7 at
    K = 3072, 6.2e-7 on the largest tile; an operand without its low halves
    shows 1e-4)."""
    x = seeded.normal(9000 + m, m * k).reshape(m, k)
    w = seeded.normal(9100 + n, k * n, 0.05).reshape(k, n)
    b = seeded.normal(9200, n)
    g = (0.1 + 0.9 * seeded.uniform01(9300, n)).astype(np.float32)
    r = seeded.normal(9400, m * n).reshape(m, n)
    lin = rt.prepare_linear_f32(k, n, w, b, g)
    xt, wt, rs = rt.upload_f32(x), rt.upload_f32(w), rt.upload_f32(r)
    got = {}

    def run():
        got["row_major"] = rt.download_f32(rt.gemm_row_major_f32(xt, wt, m, k, n)).reshape(m, n)
        got["linear"] = rt.download_f32(lin.run(xt, m)).reshape(m, n)
        got["chw"] = rt.download_f32(lin.run_chw(xt, m)).reshape(n, m).T
        lin.run_residual(xt, m, rs)
        got["residual"] = rt.download_f32(rs).reshape(m, n)

    assert {"split_operands", "split_rows"} <= _launches(rt, run)
    ref = x.astype(np.float64) @ w.astype(np.float64)
    bound = _bound(x, w)
    assert np.all(np.abs(got["row_major"] - ref) <= bound)
    assert np.linalg.norm(got["row_major"] - ref) <= 1e-6 * np.linalg.norm(ref)
    exp = (ref + b) * g
    bound = bound * g + 2.0 ** -22 * (np.abs(ref) + np.abs(b)) * g
    for name in ("linear", "chw"):
        assert np.all(np.abs(got[name] - exp) <= bound), name
        assert np.linalg.norm(got[name] - exp) <= 1e-6 * np.linalg.norm(exp), name
    assert np.all(np.abs(got["residual"] - (r + exp)) <= bound + 2.0 ** -23 * np.abs(r + exp))


def test_split_gemm_row_scales(rt):
    """Rows and columns of every magnitude: zero, subnormal, tiny, huge, and
    one outlier among ordinary values."""
    m, k, n = 70, 97, 40
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
    xt, wt, lin = rt.upload_f32(x), rt.upload_f32(w), rt.prepare_linear_f32(k, n, w, np.zeros(n, np.float32))
    got = []

    def run():
        got.append(rt.download_f32(rt.gemm_row_major_f32(xt, wt, m, k, n)).reshape(m, n))
        got.append(rt.download_f32(lin.run(xt, m)).reshape(m, n))

    assert {"split_operands", "split_rows"} <= _launches(rt, run)
    for a in got:
        # + the rounding of subnormal results and partial sums
        assert np.all(np.abs(a - ref) <= _bound(x, w) + 2.0 ** -23 * np.abs(ref) + k * 2.0 ** -149)


@pytest.mark.parametrize("where", ["x", "w", "both"])
def test_split_gemm_inf_and_nan(rt, where):
    """Infinities and NaNs give what the float product gives, element by
    element, and leave the other rows and columns as they are.  (A prepared
    weight that holds one has no split rows.)"""
    m, k, n = 70, 97, 40
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
    xt, wt, lin = rt.upload_f32(x), rt.upload_f32(w), rt.prepare_linear_f32(k, n, w, np.zeros(n, np.float32))
    got = []

    def run():
        got.append(rt.download_f32(rt.gemm_row_major_f32(xt, wt, m, k, n)).reshape(m, n))
        got.append(rt.download_f32(lin.run(xt, m)).reshape(m, n))

    names = _launches(rt, run)
    assert "split_operands" in names and ("split_rows" in names) == (where == "x")
    for a in got:
        assert np.array_equal(np.isnan(a), np.isnan(ref))
        assert np.array_equal(a[~fine & ~np.isnan(ref)], ref[~fine & ~np.isnan(ref)].astype(np.float32))
        assert np.all(np.abs(a[fine] - clean[fine]) <= 2 * bound[fine])


def _wide_operands(kind, m, k, n):
    """Finite operands whose large entries meet zeros or small ones."""
    x = seeded.normal(10300 + m, m * k).reshape(m, k)
    w = seeded.normal(10400 + n, k * n).reshape(k, n)
    u = seeded.uniform01(10500, m * k).reshape(m, k)
    if kind == "outlier":         # one entry of each row, of rising size, has no weight
        x[:, 7] = np.float32(10.0) ** np.linspace(4, 37, m, dtype=np.float32)
        w[7] = 0.0
    elif kind == "weight":        # the same of the columns
        w[9] = np.float32(10.0) ** np.linspace(-37, 37, n, dtype=np.float32)
        x[:, 9] = 0.0
    elif kind == "bands":         # half of the columns see the small half of each row alone
        x[:, ::2] *= np.float32(2.0 ** 45)
        w[::2, : n // 2] = 0.0
    elif kind == "spread":        # log-uniform over 2^80
        x *= np.exp2(80.0 * u - 40.0).astype(np.float32)
        w *= np.exp2(80.0 * seeded.uniform01(10600, k * n).reshape(k, n) - 40.0).astype(np.float32)
    elif kind == "one_hot":       # single entries, some of them tiny
        w[:] = 0.0
        w[(np.arange(n) * 7) % k, np.arange(n)] = 1.0
        x[u < 0.01] *= np.float32(1e-9)
    elif kind == "gelu":          # a GELU's tail: a tenth of the row far below its largest
        x = (3 * x * 0.5 * (1 + np.vectorize(math.erf)(3 * x / np.sqrt(2.0)))).astype(np.float32)
    return x, w


@pytest.mark.parametrize("kind", ["outlier", "weight", "bands", "spread", "one_hot", "gelu"])
@pytest.mark.parametrize("m, k, n", [(65, 101, 770), (97, 2563, 70), (865, 100, 3074), (1153, 1003, 768)])
def test_split_gemm_of_wide_ranges(rt, kind, m, k, n):
    """Each output is right to the rounding of its own terms |x w|, whatever
    else its row and column hold: no term for the range of either."""
    x, w = _wide_operands(kind, m, k, n)
    xt, wt = rt.upload_f32(x), rt.upload_f32(w)
    lin = rt.prepare_linear_f32(k, n, w, np.zeros(n, np.float32))
    ref = x.astype(np.float64) @ w.astype(np.float64)
    bound = (2.0 ** -21 + k / 4 * 2.0 ** -23) * (np.abs(x).astype(np.float64) @ np.abs(w)) + 2.0 ** -148
    res = rt.upload_f32(np.zeros(m * n, np.float32))
    out = {}

    def run():
        out["row_major"] = rt.download_f32(rt.gemm_row_major_f32(xt, wt, m, k, n)).reshape(m, n)
        out["linear"] = rt.download_f32(lin.run(xt, m)).reshape(m, n)
        out["chw"] = rt.download_f32(lin.run_chw(xt, m)).reshape(n, m).T
        lin.run_residual(xt, m, res)
        out["residual"] = rt.download_f32(res).reshape(m, n)
        if n % 192 == 0:
            q, kk, v = lin.run_qkv_hnd(xt, 1, m, n // 192)
            out["qkv"] = np.concatenate([rt.download_f32(t).reshape(n // 192, m, 64).transpose(1, 0, 2).reshape(m, -1)
                                         for t in (q, kk, v)], axis=1)

    assert {"split_operands", "split_rows"} <= _launches(rt, run)
    for name, got in out.items():
        over = np.abs(got - ref) / bound
        assert np.all(over <= 1.0), (name, float(over.max()), int((over > 1).sum()))


def _attention64(q, k, v):
    s = q.astype(np.float64) @ k.astype(np.float64).transpose(0, 2, 1) / np.sqrt(q.shape[2])
    p = np.exp(s - s.max(-1, keepdims=True))
    return (p / p.sum(-1, keepdims=True)) @ v.astype(np.float64)


# One key, one panel and one more (32 keys), one step and one more (128), the
# second and third step, the one-launch split's last length (64 K floats) and the
# first past it, head dims that fill no granule; scores up to 3 x the usual.  (At
# head dim 64 the shapes that attn_split_pays takes.)
@pytest.mark.parametrize("heads, tokens, hd, scale", [
    (1, 1, 60, 1.0), (3, 32, 63, 1.0), (2, 33, 60, 1.0), (13, 128, 60, 1.0), (2, 129, 64, 3.0), (1, 257, 40, 1.0),
    (2, 385, 7, 1.0), (20, 257, 64, 1.0), (13, 640, 64, 1.0), (6, 1024, 64, 3.0), (6, 1025, 64, 1.0),
    (5, 1700, 33, 1.0)])
def test_split_attention_vs_float64(rt, heads, tokens, hd, scale):
    """Relative to the largest |v| of the head: each weight p is off by the
    rounding of its exponent (2^-24 of up to 32, twice), the exponential (2^-23)
    and the score (2^-21 of sum |q k| / sqrt(hd), as a projection's), and the
    average of V by 2^-21 and one addition per eight keys in each stream."""
    n = heads * tokens * hd
    q, k, v = (seeded.normal(s + tokens, n).reshape(heads, tokens, hd) for s in (9900, 9910, 9920))
    q = q * np.float32(scale)
    q[0, 0] *= np.float32(1e-3)
    exp = _attention64(q, k, v)
    t = [rt.upload_f32(a) for a in (q, k, v)]
    score = 2.0 ** -21 * (np.abs(q).astype(np.float64) @ np.abs(k).transpose(0, 2, 1)).max() / np.sqrt(hd)
    tol = (2 * (score + 2.0 ** -18 + 2.0 ** -23) + 2.0 ** -21 + tokens / 32 * 2.0 ** -23) * np.abs(v).max()
    got = rt.download_f32(rt.attention_online_f32(*t, heads, tokens, hd)).reshape(exp.shape)
    assert np.abs(got - exp).max() <= tol
    if hd == 64:
        tm = rt.download_f32(rt.flash_attention_f32_da3_base(*t, heads, tokens, True))
        assert np.array_equal(tm.reshape(tokens, heads, hd).transpose(1, 0, 2), got)


def test_split_attention_head_scales_and_non_finite(rt):
    """Heads of different magnitude, and heads with a NaN or an infinity,
    which fall back to floats: the NaN reaches what the float attention lets
    it reach, and no other head."""
    H, T, hd = 5, 300, 64
    q, k, v = (seeded.normal(s, H * T * hd).reshape(H, T, hd) for s in (9930, 9940, 9950))
    k[1] *= np.float32(1e-20)
    v[1] *= np.float32(1e20)
    q[2] *= np.float32(1e-38)
    clean = _attention64(q, k, v)
    q[3, 5, 7] = np.nan           # one query
    v[4, 9, 3] = np.inf           # one output column
    got = rt.download_f32(rt.attention_online_f32(*(rt.upload_f32(a) for a in (q, k, v)), H, T, hd)).reshape(H, T, hd)
    vmax = np.abs(v[:3]).max(axis=(1, 2))[:, None, None]
    assert np.all(np.abs(got[:3] - clean[:3]) <= 2e-5 * vmax)
    assert np.isnan(got[3, 5]).all()
    rest = np.delete(np.arange(T), 5)
    assert np.abs(got[3, rest] - clean[3, rest]).max() <= 2e-5 * 5
    assert np.isposinf(got[4, :, 3]).all()
    cols = np.delete(np.arange(hd), 3)
    assert np.abs(got[4][:, cols] - clean[4][:, cols]).max() <= 2e-5 * 5


def _conv64(x, w, p):
    out_c, _, kh, kw = w.shape
    z = np.pad(x.astype(np.float64), ((0, 0), (p, p), (p, p)))
    oh, ow = z.shape[1] - kh + 1, z.shape[2] - kw + 1
    out = np.zeros((out_c, oh, ow))
    for ky in range(kh):
        for kx in range(kw):
            tap = z[:, ky:ky + oh, kx:kx + ow].reshape(z.shape[0], -1)
            out += (w[:, :, ky, kx].astype(np.float64) @ tap).reshape(out.shape)
    return out


@pytest.mark.parametrize("kind", ["pixel", "lowest", "channel", "region", "weight", "tiny"])
@pytest.mark.parametrize("in_c, out_c, ih, iw, k, p, relu", [
    (32, 130, 97, 143, 3, 1, False), (160, 70, 71, 65, 3, 1, True), (256, 257, 96, 93, 1, 0, False),
    (96, 130, 61, 50, 3, 0, False)])
def test_split_convolution_of_wide_ranges(rt, kind, in_c, out_c, ih, iw, k, p, relu):
    """Each output is right to the rounding of the terms in its own window,
    whatever else the image and the weight hold."""
    x = seeded.normal(10700 + ih, in_c * ih * iw).reshape(in_c, ih, iw)
    w = seeded.normal(10800 + k, out_c * in_c * k * k, 0.05).reshape(out_c, in_c, k, k)
    if kind == "pixel":       # one far pixel, each size in its own channel
        x[:, ih // 2, iw // 3] = np.float32(10.0) ** np.linspace(3, 30, in_c, dtype=np.float32)
    elif kind == "lowest":    # a mask of the type's lowest value, weightless channels under it
        x[0, :, : iw // 4] = np.finfo(np.float32).min
        w[:, 0] = 0.0
    elif kind == "channel":   # a large channel that half of the outputs do not see
        x[5] *= np.float32(1e12)
        w[: out_c // 2, 5] = 0.0
    elif kind == "region":    # a dark region
        x[:, : ih // 2] *= np.float32(1e-11)
    elif kind == "weight":    # large weights on empty channels
        w[:, 3] = np.float32(1e15)
        x[3] = 0.0
    elif kind == "tiny":      # values of every size down to a subnormal
        x *= np.exp2(-120.0 * seeded.uniform01(10900, x.size)).astype(np.float32).reshape(x.shape)
    xin = np.maximum(x, 0) if relu else x
    exp, mag = _conv64(xin, w, p), _conv64(np.abs(xin), np.abs(w), p)
    conv = rt.prepare_conv2d_f32(in_c, out_c, k, k, 1, p, w, np.zeros(out_c, np.float32))
    got = rt.download_f32((conv.run_relu_input if relu else conv.run)(rt.upload_f32(x), ih, iw)).reshape(exp.shape)
    over = np.abs(got - exp) / ((2.0 ** -21 + in_c * k * k / 4 * 2.0 ** -23) * mag + 2.0 ** -148)
    assert np.all(over <= 1.0), (float(over.max()), int((over > 1).sum()))


def _wide_attention(kind, H, T, hd):
    q, k, v = (seeded.normal(s + T, H * T * hd).reshape(H, T, hd) for s in (9860, 9870, 9880))
    if kind == "k_row":        # a key row whose huge entry meets no query
        q[:, :, 1] = 0.0
        k[:, T // 2, 1] = 1e30
    elif kind == "q_row":      # one query of another size, huge where no key has anything
        k[:, :, 2] = 0.0
        q[:, T // 3, 2] = -1e25
    elif kind == "v_row":      # a huge value row that no query attends to
        q[:, :, 0] = 30.0
        k[:, T // 2, 0] = -300.0
        v[:, T // 2] = 1e30
    elif kind == "v_dims":     # value columns of very different sizes
        v *= np.float32(10.0) ** np.linspace(-18, 18, hd, dtype=np.float32)
    elif kind == "v_rows":     # a query that attends to a tiny value row only
        q[:, 3:] *= 0.1
        q[:, :3, 0] = 30.0
        k[:, 5] *= 0.1
        k[:, 5, 0] = 30.0
        v[:, 5] *= np.float32(1e-12)
    elif kind == "sink":       # a key that takes nearly all weight and has no value
        q[:, :, 0] = 11.0
        k[:, :, 0] = 0.0
        k[:, 0] = 0.0
        k[:, 0, 0] = 1.7 * np.sqrt(hd)
        v[:, 0] = 0.0
    elif kind == "scales":     # every row of its own size
        for a in (q, k):
            a *= np.exp2(-30.0 * seeded.uniform01(9890 + T, H * T)).astype(np.float32).reshape(H, T, 1)
    return q, k, v


@pytest.mark.parametrize("kind", ["k_row", "q_row", "v_row", "v_dims", "v_rows", "sink", "scales"])
@pytest.mark.parametrize("H, T, hd", [(2, 130, 64), (6, 865, 64), (2, 1100, 40), (2, 300, 33)])
def test_split_attention_of_wide_ranges(rt, kind, H, T, hd):
    """Each output against the rounding of its own terms p |v| (as in
    test_split_attention_vs_float64, per output): rows and columns of other
    sizes take nothing from it."""
    q, k, v = _wide_attention(kind, H, T, hd)
    q64, k64, v64 = (a.astype(np.float64) for a in (q, k, v))
    s = q64 @ k64.transpose(0, 2, 1) / np.sqrt(hd)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    terms = np.abs(q64) @ np.abs(k64).transpose(0, 2, 1) / np.sqrt(hd)
    score = 2.0 ** -21 * np.where(p > 1e-12, terms, 0).max(-1)[:, :, None]
    tol = 2 * (score + 2.0 ** -18 + 2.0 ** -23) + 2.0 ** -21 + T / 32 * 2.0 ** -23
    t = [rt.upload_f32(a) for a in (q, k, v)]
    got = rt.download_f32(rt.attention_online_f32(*t, H, T, hd)).reshape(v.shape)
    over = np.abs(got - p @ v64) / (tol * (p @ np.abs(v64)) + 2.0 ** -148)
    assert np.all(over <= 1.0), (float(over.max()), int((over > 1).sum()))


# Grids of at least 128 64 x 64 tiles: ragged rows and widths, one and five
# channel slices, 1 x 1, 3 x 3 and 5 x 5 taps with and without padding, output
# channels that fill no tile.
@pytest.mark.parametrize("in_c, out_c, ih, iw, k, p, relu", [
    (32, 130, 97, 143, 3, 1, False), (160, 70, 71, 65, 3, 1, True), (256, 257, 96, 93, 1, 0, False),
    (64, 128, 70, 67, 5, 2, False), (96, 130, 61, 50, 3, 0, True)])
def test_split_convolution_vs_float64(rt, in_c, out_c, ih, iw, k, p, relu):
    x = seeded.normal(10000 + ih, in_c * ih * iw).reshape(in_c, ih, iw)
    w = seeded.normal(10100 + k, out_c * in_c * k * k, 0.05).reshape(out_c, in_c, k, k)
    b = seeded.normal(10200, out_c)
    conv = rt.prepare_conv2d_f32(in_c, out_c, k, k, 1, p, w, b)
    oh, ow = ih + 2 * p - k + 1, iw + 2 * p - k + 1

    def direct(img, wt):
        z = np.pad(img.astype(np.float64), ((0, 0), (p, p), (p, p)))
        out = np.zeros((out_c, oh, ow))
        for ky in range(k):
            for kx in range(k):
                out += np.einsum("oc,cyx->oyx", wt[:, :, ky, kx].astype(np.float64),
                                 z[:, ky:ky + oh, kx:kx + ow], optimize=True)
        return out

    xin = np.maximum(x, 0) if relu else x
    exp = direct(xin, w) + b[:, None, None]
    n = in_c * k * k
    bound = (2.0 ** -21 + n / 4 * 2.0 ** -23) * direct(np.abs(xin), np.abs(w)) + 2.0 ** -23 * np.abs(exp)
    run = conv.run_relu_input if relu else conv.run
    got = rt.download_f32(run(rt.upload_f32(x), ih, iw)).reshape(exp.shape)
    assert np.all(np.abs(got - exp) <= bound)
    # An infinity and a NaN reach what they reach in floats, and no more.
    x[1, 3, 5], x[0, ih - 1, 0] = np.inf, np.nan
    with np.errstate(invalid="ignore"):
        odd = direct(np.maximum(x, 0) if relu else x, w) + b[:, None, None]
    if relu:  # the crate's max(x, 0) of a NaN is 0
        x[0, ih - 1, 0] = 0.0
        odd = direct(np.maximum(x, 0), w) + b[:, None, None]
    got = rt.download_f32(run(rt.upload_f32(x), ih, iw)).reshape(exp.shape)
    fine = np.isfinite(odd)
    assert np.array_equal(np.isnan(got), np.isnan(odd))
    assert np.array_equal(got[~fine & ~np.isnan(odd)], odd[~fine & ~np.isnan(odd)].astype(np.float32))
    assert np.all(np.abs(got[fine] - odd[fine]) <= bound[fine])


@pytest.mark.parametrize("T, inf", [(1, None), (65, "v"), (130, "q"), (200, None), (300, "v"), (560, None)])
def test_q8_block_attention_writes_q8_rows(rt, T, inf):
    """The Q8_0 rows that the attention writes are quantize_row_q8_0 of its
    float output, bit for bit: ragged query tiles, and heads with an inf."""
    w = da3.block_weights(seed=42, layerscale=1.0)
    if inf:
        w["b_qkv"][{"q": 5, "v": 2 * 768 + 70}[inf]] = np.inf
    x = seeded.normal(9960 + T, T * 768)

    def attention(q, k, v, heads, tokens, hd):
        return rt.download_f32(rt.flash_attention_f32_da3_base(rt.upload_f32(q), rt.upload_f32(k), rt.upload_f32(v),
                                                               heads, tokens))

    def layernorm(a, rows, cols, g, b, eps):
        return rt.download_f32(rt.layernorm_f32(rt.upload_f32(a), rt.upload_f32(g), rt.upload_f32(b), rows, cols, eps))

    exp = q8_block(x, w, T, None, attention=attention, layernorm=layernorm)
    xt = rt.upload_f32(x)
    rt.vit_block_run(rt.prepare_block(w, q8_0=True), xt, 1, T)
    assert np.array_equal(rt.download_f32(xt), exp, equal_nan=True)


def _wide_block(kind):
    w = da3.block_weights(seed=61, layerscale="uniform", ln_affine=True, qk_norm=kind.startswith("late"))
    qkv, proj, fc1, fc2 = (w[n].reshape(s) for n, s in (("w_qkv", (768, 2304)), ("w_proj", (768, 768)),
                                                       ("w_fc1", (768, 3072)), ("w_fc2", (3072, 768))))
    if kind.endswith("off"):         # neurons that their bias switches off
        w["b_fc1"][:7] = -1e8
    elif kind.endswith("neuron"):    # a huge neuron that nothing reads
        w["b_fc1"][11] = 1e12
        fc2[11] = 0.0
    elif kind.endswith("value"):     # a huge value channel that nothing reads
        w["b_qkv"][2 * 768 + 70] = 1e12
        proj[70] = 0.0
    elif kind.endswith("norm"):      # a huge LayerNorm channel that nothing reads
        w["ln1_gamma"][5], w["ln2_gamma"][9] = 1e10, 1e10
        qkv[5] = 0.0
        fc1[9] = 0.0
    elif kind.endswith("weight"):    # large weights on channels that are empty
        w["ln1_gamma"][5] = w["ln1_beta"][5] = 0.0
        qkv[5] = 1e12
    elif kind.endswith("scores"):    # a huge query channel against a key channel of zero
        qkv[:, 3] *= 1e10
        qkv[:, 768 + 3] = 0.0
        w["b_qkv"][768 + 3] = 0.0
    return w


@pytest.mark.parametrize("kind", ["plain", "off", "neuron", "value", "norm", "weight", "scores", "late", "late_value",
                                  "late_neuron"])
def test_block_of_wide_weights_vs_float64(rt, kind):
    """Large channels that meet zeros leave the rest of the block as it is: the
    branches within 2e-6 of float64 (2-norm).  The split block shows 3.1e-7, and
    the fp32 matrix instructions, which the products of huge rows are formed
    again on, 1.0e-6 at fc2's K of 3072.  Only weights whose range the split
    form does not hold take the other form."""
    w = _wide_block(kind)
    T, pos = 97, da3.positions_yx(8, 12)
    x = seeded.normal(9965, T * 768)
    exp = block64(x, w, T, pos)[0]
    xt = rt.upload_f32(x)
    blk = rt.prepare_block(w)
    names = _launches(rt, lambda: rt.vit_block_run(blk, xt, 1, T, pos))
    assert ("layernorm_split" in names) == (kind in ("plain", "late", "off"))
    got = rt.download_f32(xt).astype(np.float64)
    error = np.linalg.norm(got - exp) / np.linalg.norm(exp - x)
    print(f"{kind}: {error:.2e}")
    assert error <= 2e-6


@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_block_of_non_finite_weights(rt, value):
    """Weights with an infinity or NaN keep a block on one product at a time,
    of which that one is on the fp32 matrix instructions.  It reaches its own
    output column and no other."""
    w = da3.block_weights(seed=63, layerscale="uniform")
    T = 97
    x = seeded.normal(9966, T * 768)
    exp = block64(x, w, T, None)[0].reshape(T, 768)
    w["w_fc2"].reshape(3072, 768)[5, 40] = value  # one output column of fc2
    xt, blk = rt.upload_f32(x), rt.prepare_block(w)
    names = _launches(rt, lambda: rt.vit_block_run(blk, xt, 1, T))
    assert "layernorm_split" not in names and "layernorm" in names
    got = rt.download_f32(xt).reshape(T, 768).astype(np.float64)
    assert not np.isfinite(got[:, 40]).any()
    cols = np.delete(np.arange(768), 40)
    branch = exp - x.reshape(T, 768)
    assert np.linalg.norm((got - exp)[:, cols]) <= 2e-6 * np.linalg.norm(branch[:, cols])


@pytest.mark.parametrize("value", ["", "0"])
@pytest.mark.parametrize("name, asks", [("GEMM_TAIL", "gemm"), ("GEMM_KGROUP", "gemm"), ("GEMM_TILE", "gemm"),
                                        ("GEMM_RM_DIRECT", "row_major"), ("FLASH_SPLITS", "attention"),
                                        ("FLASH_XCD", "attention"), ("CONV_DIRECT", "conv")])
def test_overrides_ask_for_the_fp32_kernels(rt, monkeypatch, name, asks, value):
    """An override of the fp32 kernels, set to anything, is obeyed by every call
    that it names: a projection, a row-major product, an attention, a
    convolution and the whole block."""
    if name == "FLASH_SPLITS" and value == "0":
        value = "1"
    m, k, n = 257, 101, 771
    x, w = rt.upload_f32(seeded.normal(1, m * k)), seeded.normal(2, k * n)
    wt, lin = rt.upload_f32(w), rt.prepare_linear_f32(k, n, w, seeded.normal(3, n))
    qkv = [rt.upload_f32(seeded.normal(s, 2 * 130 * 64)) for s in (4, 5, 6)]
    img, conv = rt.upload_f32(seeded.normal(7, 64 * 97 * 96)), rt.prepare_conv2d_f32(64, 128, 3, 3, 1, 1,
                                                                                    seeded.normal(8, 128 * 64 * 9))
    blk, x0 = rt.prepare_block(da3.block_weights(seed=62, layerscale="uniform")), seeded.normal(9, 97 * 768)

    def block():
        t = rt.upload_f32(x0)
        names = _launches(rt, lambda: rt.vit_block_run(blk, t, 1, 97))
        return names, rt.download_f32(t)

    calls = {"gemm": lambda: lin.run(x, m), "row_major": lambda: rt.gemm_row_major_f32(x, wt, m, k, n),
             "attention": lambda: rt.flash_attention_f32_da3_base(*qkv, 2, 130), "conv": lambda: conv.run(img, 97, 96)}
    split = {c: rt.download_f32(f()) for c, f in calls.items()}
    names, ref = block()
    assert "layernorm_split" in names
    monkeypatch.setenv("VESTRA_HIP_" + name, value)
    asked = {"gemm": {"gemm", "row_major", "conv"}}.get(asks, {asks})
    for c, f in calls.items():
        got = rt.download_f32(f())
        assert np.array_equal(got, split[c]) == (c not in asked), c
        assert np.linalg.norm(got - split[c]) <= 2e-6 * np.linalg.norm(split[c]), c
    names, got = block()
    assert ("layernorm_split" in names) == (asks not in ("gemm", "attention"))
    assert ("split_rows" in names) == (asks == "attention")
    assert np.linalg.norm(got - ref) <= 2e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize("m, k, n, split", [(865, 96, 3072, False), (865, 1536, 96, False), (500, 1536, 384, False),
                                            (865, 101, 3072, True), (865, 1536, 384, True), (500, 768, 768, True)])
def test_projections_take_the_faster_form(rt, m, k, n, split):
    """The shapes on both sides of the rule's lines (split_gemm_pays)."""
    lin = rt.prepare_linear_f32(k, n, seeded.normal(1, k * n), seeded.normal(2, n))
    x = rt.upload_f32(seeded.normal(3, m * k))
    assert ("split_rows" in _launches(rt, lambda: lin.run(x, m))) == split


@pytest.mark.parametrize("H, T, split", [(12, 128, False), (12, 150, True), (48, 150, False), (12, 256, False),
                                         (12, 300, True), (12, 500, False), (12, 560, True), (24, 420, True),
                                         (48, 400, False), (48, 560, True), (1, 1729, False), (4, 1300, True)])
def test_attention_takes_the_faster_form(rt, monkeypatch, H, T, split):
    """The shapes on both sides of the rule's lines (attn_split_pays): the bits
    are those of the fp32 kernels, asked for, or others; every entry point
    follows the same rule."""
    t = [rt.upload_f32(seeded.normal(s, H * T * 64)) for s in (1, 2, 3)]
    got = rt.download_f32(rt.flash_attention_f32_da3_base(*t, H, T, False))
    assert np.array_equal(rt.download_f32(rt.attention_online_f32(*t, H, T, 64)), got)
    out = rt.alloc_f32(H * T * 64)
    if 3 * H * T * 256 <= 60 << 20:  # its scratch holds the split rows
        rt.flash_attention_f32_da3_base_into(*t, H, T, False, out)
        assert np.array_equal(rt.download_f32(out), got)
    monkeypatch.setenv("VESTRA_HIP_FLASH_FUSED", "")
    asked = rt.download_f32(rt.flash_attention_f32_da3_base(*t, H, T, False))
    assert np.array_equal(asked, got) == (not split)
    assert np.linalg.norm(asked - got) <= 2e-6 * np.linalg.norm(got)
