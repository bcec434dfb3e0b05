"""The split-operand kernels (fp32 operands as three bf16 parts on the bf16
matrix cores) at the sizes where they can go wrong: tile and stage remainders,
K splits, transposed and unaligned operands, the ends of the fp32 range, and
sums that are not finite in the scaled range (formed again in fp32)."""
import ctypes
import gc

import numpy as np
import pytest

from camel_amd import _hip as H
from tests import hipkit as K
from tests.test_gpu_exact import assert_bits, exact_dense, wide, wide_pair
from tests.test_gpu_transpose import sgemm_at

pytestmark = pytest.mark.gpu

F = np.float32
EPI = H.EPI_BIAS | H.EPI_RELU

# M, N, K, transposed A: which kernel and what is ragged
SHAPES = [
    (2100, 4100, 257, False),   # 256x256 tiles, last row / column tiles 52 / 4, K % 32 = 1
    (1000, 3001, 2047, False),  # 128x128 with its two k groups, odd N and K (unaligned rows)
    (700, 1030, 2000, True),    # 128x128 with K splits, At rows of 700 floats
    (129, 4096, 2048, False),   # 128x128 with K splits, one row in the last tile row
    (8192, 512, 500, False),    # 128x128 unsplit, K % 64 = 52
    (321, 333, 8190, True),     # 128x128 with many K splits, everything odd
    (300, 3000, 800, False),    # 64x64, last row tile 44, last column tile 56, K % 64 = 32
    (67, 201, 8021, True),      # 64x64 with many K splits, everything odd
    (2662, 553, 409, False),    # 64x64, more tiles than CUs, rows unaligned
    (715, 6927, 455, False),    # 256x256 with K splits, everything odd
    (712, 5492, 466, True),     # the same transposed, K % 32 = 18
]


def run(a, b, bias, flags, trans):
    return sgemm_at(np.ascontiguousarray(a.T), b, bias, flags) if trans else K.sgemm(a, b, bias, flags)


@pytest.mark.parametrize("M,N,Kd,trans", SHAPES)
def test_exact_on_wide_operands(M, N, Kd, trans):
    for side in ("A", "B"):
        print(f"split {M}x{N}x{Kd} trans {trans} wide {side}", flush=True)
        a, b = wide_pair(0x5100 + M + Kd, (M, Kd), (Kd, N), side)
        bias = wide(0x5101 + N, (N,))
        assert_bits(run(a, b, bias, EPI, trans), exact_dense(a, b, bias, True), f"wide {side}")


@pytest.mark.parametrize("M,N,Kd,trans", SHAPES)
def test_every_bit_of_an_operand_arrives(M, N, Kd, trans):
    # One operand of random floats over 2^-90 .. 2^90, the other one 1 per
    # column (row): the product copies elements, so all 24 bits have to
    # survive the split in either operand.
    print(f"split copy {M}x{N}x{Kd}", flush=True)
    rng = np.random.default_rng(M + N)
    wide_a = (rng.uniform(-2, 2, (M, Kd)) * 2.0 ** rng.integers(-90, 90, (M, Kd))).astype(F)
    pick = rng.integers(0, Kd, N)
    b = np.zeros((Kd, N), F)
    b[pick, np.arange(N)] = 1.0
    assert_bits(run(wide_a, b, None, 0, trans) + F(0), wide_a[:, pick] + F(0), "A")
    wide_b = (rng.uniform(-2, 2, (Kd, N)) * 2.0 ** rng.integers(-90, 90, (Kd, N))).astype(F)
    pick = rng.integers(0, Kd, M)
    a = np.zeros((M, Kd), F)
    a[np.arange(M), pick] = 1.0
    assert_bits(run(a, wide_b, None, 0, trans) + F(0), wide_b[pick] + F(0), "B")


@pytest.mark.parametrize("M,N,Kd,trans", SHAPES)
def test_sums_round_once_per_stage(M, N, Kd, trans):
    # Accumulators are rounded once per 32 k: |dC| <= (K / 32 + 8) 2^-24
    # sum |a||b| -- the 8 for the 6 MFMAs of a stage, the dropped products
    # (2^-24 (1 + 2^-9) together) and the adds of k groups and splits (at most 32 more terms,
    # each a partial sum of its own K range, counted in K / 32).
    print(f"split real {M}x{N}x{Kd}", flush=True)
    rng = np.random.default_rng(M * 3 + Kd)
    a = rng.uniform(-1, 1, (M, Kd)).astype(F)
    b = rng.uniform(-1, 1, (Kd, N)).astype(F)
    got = run(a, b, None, 0, trans).astype(np.float64)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    bound = (Kd / 32 + 8) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64))
    assert np.all(np.abs(got - a64 @ b64) <= bound)


# (Of larger operands a few values, below 2^-16, are not scaled exactly: 27 of 3e6
# at 715 x 6927 x 455, enough to change a bit of one sum in 4e6.)
@pytest.mark.parametrize("M,N,Kd,trans", SHAPES[:9])
def test_operands_outside_the_exact_range(M, N, Kd, trans):
    # Values whose parts would leave the bf16 range unscaled, and values near the
    # fp32 maximum, whose scaled parts do leave it and whose outputs are formed
    # again in fp32: both to the fp32 kernels' bound.  Scaling by a power of two
    # is exact, so a scaled A and a scaled B give the same bits.
    print(f"split range {M}x{N}x{Kd}", flush=True)
    rng = np.random.default_rng(M + 7 * Kd)
    a = rng.uniform(-1, 1, (M, Kd)).astype(F)
    b = rng.uniform(-1, 1, (Kd, N)).astype(F)
    tiny = run(a * F(2.0 ** -110), b, None, 0, trans)
    tiny_b = run(a, b * F(2.0 ** -110), None, 0, trans)
    assert_bits(tiny, tiny_b, "scale of A against scale of B")
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    bound = 1e-5 * np.sqrt(Kd) * (np.abs(a64) @ np.abs(b64))
    assert np.all(np.abs(tiny.astype(np.float64) * 2.0 ** 110 - a64 @ b64) <= bound)
    # a few tiny elements among ordinary ones
    few = a.copy()
    few[::97, ::31] *= F(2.0 ** -120)
    got = run(few, b, None, 0, trans).astype(np.float64)
    assert np.all(np.abs(got - few.astype(np.float64) @ b64) <= bound)
    # the fp32 maximum against small factors: finite results
    big = a.copy()
    big[0, 0] = big[M - 1, Kd - 1] = np.finfo(F).max
    small = b * F(2.0 ** -20)
    got = run(big, small, None, 0, trans).astype(np.float64)
    ref = big.astype(np.float64) @ small.astype(np.float64)
    lim = 1e-5 * np.sqrt(Kd) * (np.abs(big.astype(np.float64)) @ np.abs(small.astype(np.float64)))
    assert np.all(np.abs(got - ref) <= lim)


def ulps(got, exact):
    return np.abs(got - exact) / np.spacing(np.abs(exact).astype(F)).astype(np.float64)


@pytest.mark.parametrize("M,N,Kd,trans", SHAPES)
def test_sums_of_one_term(M, N, Kd, trans):
    # One product per output.  Of x, y in [1, 2): |mid| <= 2^-8, |lo| <= 2^-17, so
    # the three dropped part products are at most 2^-24 (1 + 2^-9), half a unit
    # of the last place; the sum's cut to 24 bits is one unit, or half a unit
    # where hi hi is added rounded (64x64 tiles); the cuts of the five small
    # products, whose sum is below 2^-6, are 5 2^-30 2^(23) = 0.04 units.
    print(f"split one term {M}x{N}x{Kd}", flush=True)
    rng = np.random.default_rng(M + 3 * N)
    pick = rng.integers(0, Kd, N)
    a = rng.uniform(-2, 2, (M, Kd)).astype(F)
    b = np.zeros((Kd, N), F)
    w = b[pick, np.arange(N)] = rng.uniform(-2, 2, N).astype(F)
    got = run(a, b, None, 0, trans)
    err = ulps(got, a[:, pick].astype(np.float64) * w.astype(np.float64))
    tiles64 = (M, N, Kd, trans) in SHAPES[6:9]
    print(f"largest error {err.max():.3f} units of the last place", flush=True)
    assert err.max() <= (1.05 if tiles64 else 1.55)


@pytest.mark.parametrize("M,N,Kd,trans", SHAPES)
def test_subnormal_operands_arrive(M, N, Kd, trans):
    # One operand is a 1 (or 2^100) per column or row, the other one ordinary
    # values with subnormal ones among them, down to the last bit of fp32: the
    # product copies them, scaled.
    print(f"split subnormal {M}x{N}x{Kd}", flush=True)
    rng = np.random.default_rng(M + 5 * N)

    def values(shape):
        v = rng.uniform(-1, 1, shape).astype(F)
        low = rng.random(shape) < 0.25
        v[low] = (rng.uniform(-1, 1, low.sum()) * 2.0 ** rng.integers(-149, -133, low.sum())).astype(F)
        return v

    for factor in (F(1), F(2.0 ** 100)):
        a, pick = values((M, Kd)), rng.integers(0, Kd, N)
        b = np.zeros((Kd, N), F)
        b[pick, np.arange(N)] = factor
        assert_bits(run(a, b, None, 0, trans) + F(0), a[:, pick] * factor + F(0), f"A x {factor}")
        b, pick = values((Kd, N)), rng.integers(0, Kd, M)
        a = np.zeros((M, Kd), F)
        a[np.arange(M), pick] = factor
        assert_bits(run(a, b, None, 0, trans) + F(0), b[pick] * factor + F(0), f"B x {factor}")


@pytest.mark.parametrize("M,N,Kd,trans", SHAPES)
def test_outputs_depend_on_their_own_row_and_column(M, N, Kd, trans):
    # A special value in one row of A and one column of B changes no bit
    # elsewhere.
    print(f"split own {M}x{N}x{Kd}", flush=True)
    rng = np.random.default_rng(M + 11 * N)
    a = rng.uniform(-1, 1, (M, Kd)).astype(F)
    b = rng.uniform(-1, 1, (Kd, N)).astype(F)
    base = run(a, b, None, 0, trans)
    rest = np.ix_(np.arange(M) != 1, np.arange(N) != N - 2)
    for value in (1e-33, 1e-42, 1e32, np.finfo(F).max, np.inf, np.nan):
        a2, b2 = a.copy(), b.copy()
        a2[1, Kd - 1] = b2[0, N - 2] = value
        assert_bits(run(a2, b2, None, 0, trans)[rest], base[rest], f"{value}")


@pytest.mark.parametrize("M,N,Kd,trans", SHAPES)
def test_sums_beyond_the_scaled_range(M, N, Kd, trans):
    # Sums past 2^80, the fp32 maximum once scaled, are formed in fp32, to the
    # fp32 kernels' bound; those below stay as they are.
    print(f"split large {M}x{N}x{Kd}", flush=True)
    rng = np.random.default_rng(M + 17 * Kd)
    a = rng.uniform(-1, 1, (M, Kd)).astype(F)
    b = rng.uniform(-1, 1, (Kd, N)).astype(F)
    base = run(a, b, None, 0, trans)
    big = np.arange(M) % 3 == 0
    a[big] *= F(2.0 ** 50)
    got = run(a, b * F(2.0 ** 45), None, 0, trans)
    assert_bits(got[~big], base[~big] * F(2.0 ** 45), "small rows")
    a64, b64 = a.astype(np.float64), b.astype(np.float64) * 2.0 ** 45
    bound = 1e-5 * np.sqrt(Kd) * (np.abs(a64[big]) @ np.abs(b64))
    assert np.all(np.abs(got[big] - a64[big] @ b64) <= bound)


@pytest.mark.parametrize("M,N,Kd,trans", SHAPES[:4] + SHAPES[6:8] + SHAPES[9:])
def test_special_values_propagate(M, N, Kd, trans):
    print(f"split special {M}x{N}x{Kd}", flush=True)
    rng = np.random.default_rng(M + 13 * Kd)
    a = rng.uniform(-1, 1, (M, Kd)).astype(F)
    b = rng.uniform(-1, 1, (Kd, N)).astype(F)
    for arr in (a, b):
        flat = arr.reshape(-1)
        at = rng.choice(flat.size, size=3, replace=False)
        flat[at] = (np.inf, -np.inf, np.nan)
    b[5, :8] = 0.0
    a[3, 5] = np.inf
    with np.errstate(invalid="ignore"):
        ref = a.astype(np.float64) @ b.astype(np.float64)
    got = run(a, b, None, 0, trans)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isposinf(got), np.isposinf(ref))
    assert np.array_equal(np.isneginf(got), np.isneginf(ref))


# ---- convolutions ------------------------------------------------------------

# N, C, H, W, Co, KH, KW, stride, pad: which kernel and what is ragged
CONVS = [
    (8, 32, 56, 56, 64, 3, 3, 1, 1),     # patch kernel, tiles within images (the last of 64 pixels)
    (16, 64, 28, 28, 200, 3, 3, 1, 1),   # patch, tiles across images, Co % 128 = 72
    (45, 31, 17, 19, 130, 3, 2, 1, 2),   # patch, 31 of 32 channels, odd everything
    (8, 32, 120, 120, 20, 5, 5, 1, 0),   # 32-channel runs, patch too long: im2col loads
    (5, 13, 33, 31, 47, 5, 5, 2, 2),     # im2col loads, channels padded to 16, K splits
    (2, 100, 9, 7, 130, 1, 1, 1, 0),     # one tap, K % 32 = 8: stage below k = 0
    (1, 256, 7, 7, 96, 3, 3, 1, 1),      # many K splits of one tile of 49 pixels
    (4, 32, 20, 18, 64, 3, 1, 1, 1),     # kernels of width 1: a tap is a row (few stages: fp32 kernels)
    (4, 128, 20, 18, 64, 3, 1, 1, 1),
    (3, 40, 21, 17, 70, 2, 1, 2, 0),
    (2, 64, 15, 13, 130, 7, 1, 1, 0),
    (2, 64, 19, 16, 130, 3, 1, 2, 1),    # strided and padded
    (2, 64, 16, 19, 130, 1, 3, 2, 1),
    (16, 32, 44, 40, 64, 5, 1, 1, 1),    # (patch)
    (2, 32, 11, 25, 48, 1, 5, 1, 2),     # and of height 1 (fp32 kernels)
    (2, 80, 11, 25, 48, 1, 5, 1, 2),
    (2, 64, 13, 15, 64, 1, 1, 1, 0),     # few stages and tiles: fp32 kernels, NHWC order
    (2, 32, 21, 20, 64, 3, 3, 1, 1),
    (1, 64, 17, 9, 100, 1, 1, 2, 0),     # beyond 64 channels
    (1, 10, 31, 29, 40, 3, 3, 2, 1),     # gathered columns
]


def conv(x, w, bias, geom, flags, pool=False, layout=0):
    N, C, H_, W_, Co, KH, KW, st, pad = geom
    OH, OW = (H_ + 2 * pad - KH) // st + 1, (W_ + 2 * pad - KW) // st + 1
    shape = (N, Co, OH // 2, OW // 2) if pool else (N, Co, OH, OW)
    if layout == H.CONV_X_NCHW4:
        x = x.reshape(N, C // 4, 4, H_, W_).transpose(0, 1, 3, 4, 2)
    elif layout == H.CONV_X_NHWC:
        x = x.transpose(0, 2, 3, 1)
    dx, dw = K.dev(x), K.dev(w)
    db = K.dev(bias) if bias is not None else None
    dy = K.empty(int(np.prod(shape)) * 4)
    H.call("camel_hip_conv2d_pool2" if pool else "camel_hip_conv2d", K.P(dx.ptr), K.P(dw.ptr),
           K.P(db.ptr) if db is not None else None, K.P(dy.ptr), *geom, flags | layout)
    return K.host(dy, F, shape)


def pooled(y):
    n, c, h, w = y.shape
    y = y[:, :, :h // 2 * 2, :w // 2 * 2].reshape(n, c, h // 2, 2, w // 2, 2)
    out = y[:, :, :, 0, :, 0]
    for dy, dx in ((0, 1), (1, 0), (1, 1)):
        out = np.where(y[:, :, :, dy, :, dx] > out, y[:, :, :, dy, :, dx], out)
    return out


@pytest.mark.parametrize("geom", CONVS)
def test_conv_exact_on_wide_operands(geom):
    from tests.test_gpu_exact import exact_conv, ternary
    N, C, H_, W_, Co, KH, KW, st, pad = geom
    print(f"split conv {geom}", flush=True)
    for side in ("x", "w"):
        if side == "x":
            x = wide(0x5200 + C, (N, C, H_, W_), -1023, 1023)
            w = ternary(0x5201 + Co, (Co, C * KH * KW), 1).reshape(Co, C, KH, KW)
        else:
            x = ternary(0x5202 + C, (N, C, H_, W_), 1)
            w = wide(0x5203 + Co, (Co, C, KH, KW), -1023, 1023)
        bias = wide(0x5204, (Co,))
        want = exact_conv(x, w, bias, st, pad, True)
        assert_bits(conv(x, w, bias, geom, EPI), want, f"wide {side}")
        if want.shape[2] >= 2 and want.shape[3] >= 2:
            assert_bits(conv(x, w, bias, geom, EPI, pool=True), pooled(want), f"wide {side}, pooled")


@pytest.mark.parametrize("geom", CONVS)
def test_conv_layouts_pool_and_special_values(geom):
    # Random floats with a few special and out-of-range values: the layouts and
    # the pooled form agree bit for bit (non-finite sums are formed again one
    # by one, whatever the tile), and non-finite outputs sit where the fp64
    # convolution has them.
    N, C, H_, W_, Co, KH, KW, st, pad = geom
    print(f"split conv special {geom}", flush=True)
    rng = np.random.default_rng(C + Co)
    x = rng.uniform(-1, 1, (N, C, H_, W_)).astype(F)
    w = rng.uniform(-1, 1, (Co, C, KH, KW)).astype(F)
    bias = rng.uniform(-1, 1, Co).astype(F)
    x[0, 0, 0, 0], x[-1, -1, -1, -1], x[0, C // 2, H_ // 2, W_ // 2] = np.inf, np.nan, -np.inf
    y = conv(x, w, bias, geom, H.EPI_BIAS)
    if C % 4 == 0:
        for layout in (H.CONV_X_NHWC, H.CONV_X_NCHW4):
            np.testing.assert_array_equal(conv(x, w, bias, geom, H.EPI_BIAS, layout=layout), y)
    if min(y.shape[2:]) >= 2:
        np.testing.assert_array_equal(conv(x, w, bias, geom, H.EPI_BIAS, pool=True), pooled(y))
    # the non-finite outputs: the windows that hold a special value
    xf = np.where(np.isfinite(x), 0, 1).astype(F)
    touched = conv(xf, np.ones_like(w), None, geom, 0) > 0
    assert np.array_equal(~np.isfinite(y), touched)
    # values whose parts would leave the bf16 range unscaled
    x = np.where(np.isfinite(x), x, 0).astype(F)
    base = conv(x, w, None, geom, 0)
    tiny = conv(x * F(2.0 ** -112), w, None, geom, 0).astype(np.float64) * 2.0 ** 112
    bound = 1e-5 * np.sqrt(C * KH * KW) * conv(np.abs(x), np.abs(w), None, geom, 0)
    assert np.all(np.abs(tiny - base) <= bound)


@pytest.mark.parametrize("geom", CONVS)
def test_conv_forms_agree_on_tiny_values(geom):
    N, C, H_, W_, Co, KH, KW, st, pad = geom
    # Inputs and weights with values far below the others, subnormal ones among
    # them: every layout and the pooled form give the same bits, and a kernel
    # that copies one tap of one channel copies subnormal inputs.
    print(f"split conv tiny {geom}", flush=True)
    rng = np.random.default_rng(C + 3 * Co)
    x = rng.uniform(-1, 1, (N, C, H_, W_)).astype(F)
    w = rng.uniform(-1, 1, (Co, C, KH, KW)).astype(F)
    for arr in (x, w):
        v = arr.reshape(-1)
        at = rng.choice(v.size, size=max(1, v.size // 3000), replace=False)
        v[at] = (rng.uniform(-1, 1, at.size) * 2.0 ** rng.integers(-149, -90, at.size)).astype(F)
    y = conv(x, w, None, geom, 0)
    if C % 4 == 0:
        for layout in (H.CONV_X_NHWC, H.CONV_X_NCHW4):
            np.testing.assert_array_equal(conv(x, w, None, geom, 0, layout=layout), y)
    if min(y.shape[2:]) >= 2:
        np.testing.assert_array_equal(conv(x, w, None, geom, 0, pool=True), pooled(y))
    xs = (rng.uniform(-1, 1, x.shape) * 2.0 ** -138).astype(F)
    ws = np.zeros_like(w)
    ws[:, 0, 0, 0] = 1.0
    got = conv(xs, ws, None, geom, 0)
    OH, OW = got.shape[2:]
    xp = np.zeros((N, H_ + 2 * pad, W_ + 2 * pad), F)
    xp[:, pad:pad + H_, pad:pad + W_] = xs[:, 0]
    want = xp[:, 0:st * (OH - 1) + 1:st, 0:st * (OW - 1) + 1:st]
    np.testing.assert_array_equal(got, np.broadcast_to(want[:, None], got.shape))


@pytest.mark.parametrize("tiny", ["x", "w2", "one pixel"])
def test_conv_pair_equals_its_calls_on_tiny_values(tiny):
    from tests.test_gpu_fusion import _pair_fused, _pair_unfused
    print(f"split pair tiny {tiny}", flush=True)
    rng = np.random.default_rng(0x5400)
    x = rng.uniform(-1, 1, (3, 1, 28, 28)).astype(F)
    w1 = rng.uniform(-1, 1, (32, 1, 3, 3)).astype(F)
    w2 = rng.uniform(-1, 1, (64, 32, 3, 3)).astype(F)
    if tiny == "x":
        x[:, :, 4:12, 5:14] *= F(2.0 ** -120)
    elif tiny == "w2":
        w2[3, 5, 1, 1], w2[40, 7, 0, 2] = 1e-40, 1e-33
    else:
        x[...] = 0
        x[1, 0, 14, 14] = 1e-38
    want = _pair_unfused(x, w1, None, w2, None, 0, 0)
    assert want.any()
    np.testing.assert_array_equal(_pair_fused(x, w1, None, w2, None, 0, 0), want)


@pytest.mark.parametrize("geom", CONVS)
def test_conv_sums_of_one_term(geom):
    # As test_sums_of_one_term: a kernel of one tap of one channel, a weight of
    # its own per output channel.
    N, C, H_, W_, Co, KH, KW, st, pad = geom
    print(f"split conv one term {geom}", flush=True)
    rng = np.random.default_rng(C + 5 * Co)
    x = rng.uniform(-2, 2, (N, C, H_, W_)).astype(F)
    w = np.zeros((Co, C, KH, KW), F)
    one = w[:, C - 1, KH - 1, KW - 1] = rng.uniform(-2, 2, Co).astype(F)
    got = conv(x, w, None, geom, 0)
    OH, OW = got.shape[2:]
    xp = np.zeros((N, H_ + 2 * pad, W_ + 2 * pad))
    xp[:, pad:pad + H_, pad:pad + W_] = x[:, C - 1]
    px = xp[:, KH - 1:KH + st * (OH - 1):st, KW - 1:KW + st * (OW - 1):st]
    exact = px[:, None] * one.astype(np.float64)[None, :, None, None]
    assert ulps(got, exact).max() <= 1.55


GATHERED = [
    (1, 12, 31, 33, 33, 3, 3, 2, 1),
    (4, 6, 24, 23, 40, 3, 3, 1, 1),      # another geometry: offsets of its own
    (2, 100, 9, 7, 40, 1, 1, 1, 0),      # one tap
    (2, 20, 11, 13, 33, 3, 1, 1, 1),     # kernels of width and height 1
    (2, 20, 11, 13, 33, 1, 3, 1, 0),
    (1, 3, 20, 19, 130, 7, 7, 1, 3),     # more than 32 taps, more than 64 channels
    (1, 4, 70, 72, 20, 61, 67, 1, 0),    # the longest sum
]


def test_gathered_convs_of_several_geometries_in_turn():
    # Small layers and many-tap ones that gather their columns: exact whatever
    # geometry ran before, and nothing of a call stays allocated after it.
    from tests.test_gpu_exact import exact_conv, ternary
    cases = []
    for n, geom in enumerate(GATHERED):
        N, C, H_, W_, Co, KH, KW, st, pad = geom
        x = ternary(0x5300 + n, (N, C, H_, W_), 1)
        w = ternary(0x5320 + n, (Co, C * KH * KW), 1).reshape(Co, C, KH, KW)
        cases.append((geom, x, w, exact_conv(x, w, None, st, pad)))
    used = ctypes.c_size_t()
    H.call("camel_hip_pool_stats", ctypes.byref(used), None)
    before = used.value
    for geom, x, w, want in cases + cases[::-1] + cases:
        print(f"gathered conv {geom}", flush=True)
        assert_bits(conv(x, w, None, geom, 0), want, f"{geom}")
    gc.collect()
    H.call("camel_hip_pool_stats", ctypes.byref(used), None)
    assert used.value == before
