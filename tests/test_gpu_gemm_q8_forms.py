"""The int8-weight GEMM (m > 16) in its general forms: zero points, a per-row scale, a k of no whole
chunks of 32, an n of no whole octets, operands aligned to their elements only."""

import ctypes as C

import numpy as np
import pytest

from hip_helpers import Epilogue, assert_gamma_bound, check, dev, lib, quant_plane, same_bits

pytestmark = pytest.mark.gpu

AXIS = {"col": 1, "row": 0, "tensor": -1}


def weight(r, k, n, mode, zero, unit_scale=False):
    count = {"col": n, "row": k, "tensor": 1}[mode]
    q = r.integers(-128, 128, size=(k, n), dtype=np.int8)
    s = np.ones(count, np.float32) if unit_scale else r.uniform(1e-3, 1e-2, count).astype(np.float32)
    z = r.integers(-128, 128, size=count, dtype=np.int8) if zero else None
    return q, s, z


def dequant(q, s, z, mode):
    shape = {"col": (1, -1), "row": (-1, 1), "tensor": (1, 1)}[mode]
    w = q.astype(np.float32) - (0 if z is None else z.astype(np.float32).reshape(shape))
    return (w * s.reshape(shape)).astype(np.float32)


def run(a, q, s, z, mode, skip=0, epi=None, c=None):
    """C, with A starting `skip` floats and q `skip` matrices of n bytes into their buffers."""
    (m, k), n = a.shape, q.shape[1]
    ad = dev(np.concatenate([np.zeros(skip, np.float32), a.ravel()]))
    qd = dev(np.concatenate([np.zeros(skip * n, np.int8), q.ravel()]))
    sd, zd = dev(s), dev(z) if z is not None else None
    # The offset of a per-row plane must be a multiple of the matrix, so only the others are moved.
    rows = k + (skip if mode != "row" else 0)
    if mode == "row":
        qd, skip_q = dev(q), 0
    else:
        skip_q = skip * n
    plane = quant_plane(qd, sd, zd, [rows, n], AXIS[mode], skip_q)
    cd = c if c is not None else dev(np.full((m, n), 3.0, np.float32))
    check(lib().accel_hip_matmul_quantized_fused(ad.at(skip), None, None, C.byref(plane), cd.ptr, m, k, n,
                                                 C.byref(epi) if epi else None))
    return cd.numpy()


# k around a chunk and the three-chunk splits, n around an octet and both tiles, m around the tiles;
# 333 x 1601 x 1030 and 700 x 1000 x 1100 take 128 tiles, the others 64, most with a split K.
SHAPES = [(17, 32, 8), (33, 33, 9), (64, 63, 63), (65, 65, 65), (127, 95, 129), (129, 97, 127), (20, 127, 200),
          (17, 4095, 15), (333, 1601, 1030), (700, 1000, 1100)]
FORMS = [("col", True), ("col", False), ("tensor", True), ("row", False), ("row", True)]


@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("mode,zero", FORMS)
def test_gemm_q8_forms_bound_and_integer_sums(m, k, n, mode, zero):
    r = np.random.default_rng(m * 7919 + k + n)
    print(f"gemm q8 {m}x{k}x{n} {mode} zero {zero}", flush=True)
    q, s, z = weight(r, k, n, mode, zero)
    a = r.standard_normal((m, k)).astype(np.float32)
    for skip in (0, 1):
        assert_gamma_bound(run(a, q, s, z, mode, skip), a, dequant(q, s, z, mode))
    # Small integers with scale 1: every order of summation is exact, so an element taken twice or
    # left out shows. The residual is C itself.
    q, s, z = weight(r, k, n, mode, zero, unit_scale=True)
    a = r.integers(-4, 5, size=(m, k)).astype(np.float32)
    res = r.integers(-99, 100, size=(m, n)).astype(np.float32)
    c = dev(res)
    got = run(a, q, s, z, mode, epi=Epilogue(alpha=1.0, beta=1.0, residual=c.ptr), c=c)
    same_bits(got, (a.astype(np.float64) @ dequant(q, s, z, mode).astype(np.float64) + res).astype(np.float32))


@pytest.mark.parametrize("mode,zero", FORMS)
def test_gemm_q8_forms_values_beyond_the_bf16_parts(mode, zero):
    """Rows with an infinity, a NaN, a value above the largest bf16 and only values below 2^-110 come
    out as fp32 products do; the other rows are untouched by them."""
    m, k, n = 70, 101, 75
    r = np.random.default_rng(5)
    q, s, z = weight(r, k, n, mode, zero, unit_scale=True)
    a = r.standard_normal((m, k)).astype(np.float32)
    a[3, k - 1] = np.inf
    a[17, 0] = np.nan
    a[40] = 0
    a[40, 50] = np.float32(3.399e38)
    q[50] = np.where(r.random(n) < 0.5, 1, 0) + (0 if z is None else z.reshape(-1)[50 % z.size] if mode != "col" else z)
    a[41] = r.integers(1, 1 << 20, size=k) * np.float32(2.0 ** -140)
    w = dequant(q, s, z, mode)
    got = run(a, q, s, z, mode)
    rest = [i for i in range(m) if i not in (3, 17, 41)]
    assert_gamma_bound(got[rest], a[rest], w)
    last = w[k - 1].astype(np.float64)
    same_bits(got[3], np.where(last > 0, np.inf, np.where(last < 0, -np.inf, np.nan)).astype(np.float32))
    assert np.isnan(got[17]).all()
    up = np.float64(2.0 ** 100)  # exact scaling, so the bound's absolute term does not hide the row
    assert_gamma_bound(got[[41]].astype(np.float64) * up, a[[41]].astype(np.float64) * up, w)


@pytest.mark.parametrize("m,k,n", [(70, 101, 75), (700, 1000, 1100)])
@pytest.mark.parametrize("mode,zero", FORMS)
def test_gemm_q8_forms_activations_below_the_parts(m, k, n, mode, zero):
    """A row whose activations are all below the smallest bf16 gives their product with the weights
    (2^100 scales, so that the results are far from the fp32 minimum), not zero; zero rows stay zero."""
    r = np.random.default_rng(6)
    q, s, z = weight(r, k, n, mode, zero)
    s *= np.float32(2.0 ** (100 if mode != "row" else 10))
    a = r.standard_normal((m, k)).astype(np.float32)
    a[5] = r.integers(1, 16, size=k) * np.float32(2.0 ** -140)
    a[68] = 0
    w = dequant(q, s, z, mode).astype(np.float64)
    got = run(a, q, s, z, mode).astype(np.float64)
    up = np.float64(2.0 ** 43)  # exact: the bound's absolute term stays below what subnormal sums round
    assert_gamma_bound(got * up, a.astype(np.float64) * up, w)
    assert not got[68].any()


# The plain form (128 and 64 tiles), the small kernel (k <= 768 and k = 1536), the image and wide
# kernels, the group-interleaved GEMV and the in-place GEMV on the same kind of plane.
PLAIN_SHAPES = [(333, 1024, 2048), (100, 2048, 1024), (40, 576, 192), (40, 1536, 256), (2100, 96, 2056), (700, 96, 6000),
                (5, 4096, 8192), (16, 4096, 8192), (9, 1024, 512)]


@pytest.mark.parametrize("m,k,n", PLAIN_SHAPES)
def test_q8_plain_planes_not_finite_activations(m, k, n):
    """Whole chunks, no zero points: rows with an infinity, a NaN and a value above the largest bf16
    come out as fp32 products do, whichever kernel the size picks; the other rows are untouched."""
    r = np.random.default_rng(5)
    q, s, _ = weight(r, k, n, "col", False, unit_scale=True)
    a = r.standard_normal((m, k)).astype(np.float32)
    a[1, k - 1] = np.inf
    a[2, 0] = np.nan
    a[3] = 0
    a[3, 50] = np.float32(-3.399e38)
    q[50] = np.where(r.random(n) < 0.5, 1, 0)
    q[k - 1, :8] = 0
    print(f"q8 {m}x{k}x{n}", flush=True)
    got = run(a, q, s, None, "col")
    rest = [0] + list(range(4, m))
    assert_gamma_bound(got[rest], a[rest], q)
    same_bits(got[3], (a[3, 50] * q[50].astype(np.float32)) + np.float32(0))
    last = q[k - 1].astype(np.float64)
    same_bits(got[1], np.where(last > 0, np.inf, np.where(last < 0, -np.inf, np.nan)).astype(np.float32))
    assert np.isnan(got[2]).all()
