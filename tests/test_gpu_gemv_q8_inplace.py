"""The int8 GEMV that reads W in place (gemv_q8_inplace.hip): every plane form, ragged sizes and
alignments, each run width (1, 2, 4 and 8 columns a lane) and splits of K, against float64."""

import ctypes as C

import numpy as np
import pytest

from hip_helpers import DeviceArray, Epilogue, assert_gamma_bound, check, dev, lib, quant_plane, same_bits
from test_gpu_gemm_q8_forms import FORMS, dequant, run, weight

pytestmark = pytest.mark.gpu

# k around a 32-row block, the 8 waves of a workgroup and the splits (of 512 or 256 rows); n around
# a run and a group of each width: below 4 Mi elements 1 or 2 columns a lane, 2051 x 2049 4 columns
# in 7 splits, 4100 x 4097 4 columns with two workgroups a CU, 2047 x 14345 8 columns.
SHAPES = [(5, 1, 1), (7, 31, 2), (16, 32, 3), (9, 33, 33), (5, 257, 31), (16, 1023, 65), (12, 1025, 129),
          (6, 2051, 2049), (16, 4100, 4097), (3, 2047, 14345), (13, 2047, 14345)]


@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("mode,zero", [("col", False)] + FORMS)
def test_gemv_q8_in_place_bound_and_integer_sums(m, k, n, mode, zero):
    r = np.random.default_rng(m * 7919 + k + n)
    print(f"gemv q8 {m}x{k}x{n} {mode} zero {zero}", flush=True)
    q, s, z = weight(r, k, n, mode, zero)
    a = r.standard_normal((m, k)).astype(np.float32)
    large = k * n > 1 << 24
    for skip in (1,) if large else (0, 1):
        assert_gamma_bound(run(a, q, s, z, mode, skip), a, dequant(q, s, z, mode))
    # Small integers with scale 1: every order of summation is exact, so an element taken twice or
    # left out shows. The residual is C itself.
    q, s, z = weight(r, k, n, mode, zero, unit_scale=True)
    a = r.integers(-2, 3, size=(m, k)).astype(np.float32)
    res = r.integers(-99, 100, size=(m, n)).astype(np.float32)
    c = dev(res)
    got = run(a, q, s, z, mode, epi=Epilogue(alpha=1.0, beta=1.0, residual=c.ptr), c=c)
    same_bits(got, a @ dequant(q, s, z, mode) + res)


@pytest.mark.parametrize("mode,zero", [("col", False)] + FORMS)
def test_gemv_q8_in_place_values_beyond_the_bf16_parts(mode, zero):
    """Rows with an infinity, a NaN, a value above the largest bf16 and only values below 2^-110 come
    out as fp32 products do; the other rows are untouched by them."""
    m, k, n = 9, 1101, 75
    r = np.random.default_rng(5)
    q, s, z = weight(r, k, n, mode, zero, unit_scale=True)
    a = r.standard_normal((m, k)).astype(np.float32)
    a[1, k - 1] = np.inf
    a[3, 0] = np.nan
    a[4] = 0
    a[4, 50] = np.float32(3.399e38)
    q[50] = np.where(r.random(n) < 0.5, 1, 0) + (0 if z is None else z.reshape(-1)[50 % z.size] if mode != "col" else z)
    a[6] = r.integers(1, 1 << 20, size=k) * np.float32(2.0 ** -140)
    w = dequant(q, s, z, mode)
    got = run(a, q, s, z, mode)
    rest = [i for i in range(m) if i not in (1, 3, 6)]
    assert_gamma_bound(got[rest], a[rest], w)
    last = w[k - 1].astype(np.float64)
    same_bits(got[1], np.where(last > 0, np.inf, np.where(last < 0, -np.inf, np.nan)).astype(np.float32))
    assert np.isnan(got[3]).all()
    up = np.float64(2.0 ** 100)  # exact scaling, so the bound's absolute term does not hide the row
    assert_gamma_bound(got[[6]].astype(np.float64) * up, a[[6]].astype(np.float64) * up, w)


@pytest.mark.parametrize("m,k,n", [(7, 33, 2), (9, 1101, 75), (16, 2051, 2049), (13, 2047, 14345)])
@pytest.mark.parametrize("mode,zero", [("col", False)] + FORMS)
def test_gemv_q8_in_place_activations_below_the_parts(m, k, n, mode, zero):
    """A row whose activations are all below the smallest bf16 gives their product with the weights
    (2^100 scales, so that the results are far from the fp32 minimum), not zero; zero rows stay zero,
    and an infinite last row scale reaches the rows that have an activation there."""
    r = np.random.default_rng(6)
    q, s, z = weight(r, k, n, mode, zero)
    s *= np.float32(2.0 ** (100 if mode != "row" else 10))
    a = r.standard_normal((m, k)).astype(np.float32)
    a[5] = r.integers(1, 16, size=k) * np.float32(2.0 ** -140)
    a[2] = 0
    w = dequant(q, s, z, mode).astype(np.float64)
    got = run(a, q, s, z, mode).astype(np.float64)
    up = np.float64(2.0 ** 43)  # exact: the bound's absolute term stays below what subnormal sums round
    assert_gamma_bound(got * up, a.astype(np.float64) * up, w)
    assert not got[2].any()
    if mode == "row":
        s[-1] = np.inf
        with np.errstate(invalid="ignore"):
            sign = np.sign(a[:, -1:] * (q[-1].astype(np.float32) - (z[-1].astype(np.float32) if zero else 0)))
        same_bits(run(a, q, s, z, mode), np.where(sign == 0, np.nan, np.copysign(np.inf, sign)).astype(np.float32))


@pytest.mark.parametrize("m,zero", [(8, True), (8, False), (4, False)])
def test_gemv_q8_in_place_in_a_capture(m, zero):
    """No staged copy is needed: captured before any other use of the weight, replayed with the
    activations changed in between, each replay within the bound of the exact product. (Four rows of
    a plane without zero points take the column tiles where there are some, outside a capture.)"""
    k, n = 2048, 4096
    r = np.random.default_rng(7)
    q, s, z = weight(r, k, n, "col", zero)
    qd, warm, sd, zd = dev(q), dev(q), dev(s), dev(z) if zero else None
    plane = quant_plane(qd, sd, zd, [k, n], 1)
    wplane = quant_plane(warm, sd, zd, [k, n], 1)  # another weight sizes the workspaces
    ad, cd = dev(r.standard_normal((m, k)).astype(np.float32)), dev(np.zeros((m, n), np.float32))
    args = (m, k, n, None)
    # (rows of eight: the workspaces they take cover four)
    a8, c8 = dev(np.zeros((8, k), np.float32)), dev(np.zeros((8, n), np.float32))
    check(lib().accel_hip_matmul_quantized_fused(a8.ptr, None, None, C.byref(wplane), c8.ptr, 8, k, n, None))
    check(lib().accel_hip_synchronize())
    graph = C.c_void_p()
    check(lib().accel_hip_capture_begin())
    check(lib().accel_hip_matmul_quantized_fused(ad.ptr, None, None, C.byref(plane), cd.ptr, *args))
    check(lib().accel_hip_capture_end(C.byref(graph)))
    try:
        for _ in range(3):
            a = r.standard_normal((m, k)).astype(np.float32)
            ad.upload(a)
            check(lib().accel_hip_graph_launch(graph, 2))
            assert_gamma_bound(cd.numpy(), a, dequant(q, s, z, "col"))
    finally:
        lib().accel_hip_graph_destroy(graph)


def test_gemv_q8_in_place_more_columns_than_one_grid_dimension():
    """2^30 and a few columns: more threads than one dimension of a grid holds. Integer products, so
    the compared spans are exact: the ends, the last whole group and where the second row of workgroups
    starts."""
    m, k, n = 3, 1, (1 << 30) + 1043
    r = np.random.default_rng(1)
    q = np.frombuffer(r.bytes(n), np.int8)
    qd, sd = dev(q), dev(np.ones(1, np.float32))
    a = np.array([[1], [-2], [3]], np.float32)
    ad, cd = dev(a), DeviceArray((m, n))
    plane = quant_plane(qd, sd, None, [k, n], -1)
    check(lib().accel_hip_matmul_quantized(ad.ptr, None, None, C.byref(plane), cd.ptr, m, k, n))
    span = 2048
    for row in range(m):
        for start in (0, (1 << 29) - 1024, (1 << 29) + (1 << 27) - 1024, (1 << 30) - 1024, n - span):
            got = np.empty(span, np.float32)
            check(lib().accel_hip_peek(got.ctypes.data, cd.at(row * n + start), got.nbytes))
            same_bits(got, a[row, 0] * q[start:start + span].astype(np.float32) + np.float32(0))
