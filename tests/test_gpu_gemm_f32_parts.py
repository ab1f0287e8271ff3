"""The fp32 GEMM on bf16 parts (m > 16, any alignment): every element within 2 gamma_K of the
float64 product, at the edges of its chunks, tiles and K splits."""

import ctypes as C

import numpy as np
import pytest

from hip_helpers import Epilogue, assert_gamma_bound, check, dev, lib, same_bits

pytestmark = pytest.mark.gpu


def run(a, b, epi=None, skip=0, c=None):
    """C of accel_hip_matmul_fused with A and B starting `skip` floats into their buffers."""
    (m, k), n = a.shape, b.shape[1]
    ad = dev(np.concatenate([np.zeros(skip, np.float32), a.ravel()]))
    bd = dev(np.concatenate([np.zeros(skip, np.float32), b.ravel()]))
    cd = c if c is not None else dev(np.full((m, n), 3.0, np.float32))
    check(lib().accel_hip_matmul_fused(ad.at(skip), bd.at(skip), cd.ptr, m, k, n, C.byref(epi) if epi else None))
    return cd.numpy()


# k around a chunk and the two-chunk splits, n and m around both tiles; the last three fill 128
# tiles without a split, with two and with a ragged k.
SHAPES = [(17, 32, 1), (33, 33, 3), (64, 63, 64), (65, 64, 65), (127, 65, 129), (129, 95, 127), (40, 1003, 200),
          (33, 4095, 65), (1100, 500, 4100), (700, 1000, 1100), (333, 1999, 3001)]


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_gemm_f32_parts_bound_and_integer_sums(m, k, n):
    r = np.random.default_rng(m * 131 + k + n)
    print(f"gemm f32 {m}x{k}x{n}", flush=True)
    a = r.standard_normal((m, k)).astype(np.float32)
    b = (r.standard_normal((k, n)) * 0.05).astype(np.float32)
    for skip in (0, 1):
        assert_gamma_bound(run(a, b, skip=skip), a, b)
    # Small integers: every order of summation is exact, so an element taken twice or left out
    # shows. The residual is C itself.
    a = r.integers(-8, 9, size=(m, k)).astype(np.float32)
    b = r.integers(-8, 9, size=(k, n)).astype(np.float32)
    res = r.integers(-99, 100, size=(m, n)).astype(np.float32)
    c = dev(res)
    got = run(a, b, Epilogue(alpha=1.0, beta=1.0, residual=c.ptr), c=c)
    same_bits(got, (a.astype(np.float64) @ b + res).astype(np.float32))


@pytest.mark.parametrize("m,k,n", [(70, 101, 75), (1100, 101, 4100)])
def test_gemm_f32_parts_values_beyond_the_bf16_parts(m, k, n):
    """Rows and columns with an infinity, a NaN, a value above the largest bf16 or only values below
    2^-110 come out as fp32 products do; the others are untouched by them."""
    r = np.random.default_rng(11)
    a = r.standard_normal((m, k)).astype(np.float32)
    b = (r.standard_normal((k, n)) * 0.05).astype(np.float32)
    a[3, k - 1] = np.inf
    a[17, 0] = np.nan
    a[40] = 0
    a[40, 50] = np.float32(3.399e38)
    b[50] = np.where(r.random(n) < 0.5, 1, 0)
    a[41] = r.integers(1, 1 << 20, size=k) * np.float32(2.0 ** -140)
    b[20, 7] = -np.inf
    a[40, 20] = 1
    got = run(a, b)
    cols = [j for j in range(n) if j != 7]
    rest = [i for i in range(m) if i not in (3, 17, 41)]
    assert_gamma_bound(got[np.ix_(rest, cols)], a[rest], b[:, cols])
    last = b[k - 1, cols].astype(np.float64)
    same_bits(got[3, cols], np.where(last > 0, np.inf, np.where(last < 0, -np.inf, np.nan)).astype(np.float32))
    assert np.isnan(got[17]).all()
    same_bits(got[rest, 7], np.where(a[rest, 20] > 0, -np.inf, np.inf).astype(np.float32))
    up = np.float64(2.0 ** 100)  # exact scaling, so the bound's absolute term does not hide the row
    assert_gamma_bound(got[[41]][:, cols].astype(np.float64) * up, a[[41]].astype(np.float64) * up, b[:, cols])


@pytest.mark.parametrize("m,k,n", [(70, 101, 75), (1100, 101, 4100)])
@pytest.mark.parametrize("tiny,huge", [(-118, 60), (-126, 70), (-136, 100), (-145, 20), (-145, 127), (-70, -70)])
def test_gemm_f32_parts_values_below_the_parts(m, k, n, tiny, huge):
    """Values of 2^tiny (some or all bits below what the parts hold) in a row of A and a column of B
    against values of 2^huge in the other operand: within the bound of the exact product."""
    r = np.random.default_rng(1000 + tiny * 7 + huge)

    def values(count, exponent):
        return np.ldexp(r.uniform(1, 2, count) * r.choice([-1, 1], count), exponent).astype(np.float32)

    a = r.standard_normal((m, k)).astype(np.float32)
    b = (r.standard_normal((k, n)) * 0.05).astype(np.float32)
    a[5], b[:, 9] = values(k, tiny), values(k, huge)
    a[66], b[:, 70] = values(k, huge), values(k, tiny)
    a[66, 30:] = 0  # the sums stay below the fp32 limit
    b[30:, 9] = 0
    got = run(a, b).astype(np.float64)
    # Scaled (exactly) so that the bound's absolute term, 1e-30 > 2^-100, is k roundings of subnormal
    # products, 2^-150 each, and hides no more.
    up = np.float64(2.0 ** 43)
    rest = [i for i in range(m) if i not in (5, 66)]
    cols = [j for j in range(n) if j not in (9, 70)]
    for i, j in (([5], [9]), ([66], [70]), ([5], cols), (rest, [70]), (rest, cols)):
        assert_gamma_bound(got[np.ix_(i, j)] * up, a[i].astype(np.float64) * up, b[:, j])


@pytest.mark.parametrize("m,k,n", [(70, 101, 75), (1100, 101, 4100)])
@pytest.mark.parametrize("tiny,huge", [(-116, 56), (-122, 66), (-126, 70), (-130, 100)])
@pytest.mark.parametrize("side", ["a", "b"])
def test_gemm_f32_parts_tiny_operand_against_huge_ones(m, k, n, tiny, huge, side):
    """A row of A (a column of B) whose low bits the parts lose, where no sum is small: the other
    operand is of 2^huge throughout."""
    r = np.random.default_rng(1000 + tiny * 7 + huge)

    def values(shape, exponent):
        return np.ldexp(r.uniform(1, 2, shape) * r.choice([-1, 1], shape), exponent).astype(np.float32)

    a = values((m, k), 0 if side == "a" else huge)
    b = values((k, n), huge if side == "a" else 0)
    if side == "a":
        a[60] = values(k, tiny)
    else:
        b[:, 60] = values(k, tiny)
    assert_gamma_bound(run(a, b), a, b)
