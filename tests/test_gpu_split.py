"""The split-operand kernels (fp32 operands as three bf16 parts on the bf16
matrix cores) at the sizes where they can go wrong: tile and stage remainders,
K splits, transposed and unaligned operands, and operands outside the exact
range of the split (tiles computed again in fp32)."""
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
    (1000, 3001, 2047, False),  # 256x256, K splits, odd N and K (unaligned rows)
    (700, 1030, 2000, True),    # At rows of 700 floats, K splits
    (129, 4096, 2048, False),   # 128x128, two k groups, one row in the last tile row
    (8192, 512, 500, False),    # 128x128 unsplit, K % 64 = 52
    (321, 333, 8190, True),     # 128x128 with many K splits, everything odd
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
    # (2^-25 each) and the adds of k groups and splits (at most 32 more terms,
    # each a partial sum of its own K range, counted in K / 32).
    print(f"split real {M}x{N}x{Kd}", flush=True)
    rng = np.random.default_rng(M * 3 + Kd)
    a = rng.uniform(-1, 1, (M, Kd)).astype(F)
    b = rng.uniform(-1, 1, (Kd, N)).astype(F)
    got = run(a, b, None, 0, trans).astype(np.float64)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    bound = (Kd / 32 + 8) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64))
    assert np.all(np.abs(got - a64 @ b64) <= bound)


@pytest.mark.parametrize("M,N,Kd,trans", SHAPES)
def test_operands_outside_the_exact_range(M, N, Kd, trans):
    # Values below 2^-100 lose their last part in bf16 and values near the
    # fp32 maximum round to infinity there: their tiles run in fp32, to the
    # fp32 kernels' bound.  Scaling by a power of two is exact, so a scaled A
    # and a scaled B give the same bits.
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


@pytest.mark.parametrize("M,N,Kd,trans", SHAPES[:4])
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
