"""The fp32-weight GEMV (m <= 16, accel_hip_matmul and its fused form): every element within
2 gamma_K of the float64 product, at the edges of its batches, column runs and K splits."""

import ctypes as C

import numpy as np
import pytest

from hip_helpers import Epilogue, assert_gamma_bound, check, dev, lib, same_bits

pytestmark = pytest.mark.gpu


def run(a, b, epi=None, a_skip=0, b_skip=0, c=None):
    """C of accel_hip_matmul_fused with A and B starting a_skip / b_skip floats into their buffers."""
    (m, k), n = a.shape, b.shape[1]
    ad = dev(np.concatenate([np.zeros(a_skip, np.float32), a.ravel()]))
    bd = dev(np.concatenate([np.zeros(b_skip, np.float32), b.ravel()]))
    cd = c if c is not None else dev(np.full((m, n), 3.0, np.float32))
    check(lib().accel_hip_matmul_fused(ad.at(a_skip), bd.at(b_skip), cd.ptr, m, k, n, C.byref(epi) if epi else None))
    return cd.numpy()


# k around the 4-row step, the 16- and 32-row batches and the 8 waves; n around a run and a column
# group; 1536 and 4096 split K; 1600 x 4100 and 4096 x 4099 take runs of 2 and 4 columns, ragged.
SHAPES = [(1, 1, 4), (2, 3, 5), (16, 31, 17), (3, 33, 63), (15, 255, 65), (1, 257, 1003), (5, 576, 960), (1, 1536, 576),
          (16, 4096, 256), (7, 1600, 4100), (16, 4096, 4099), (1, 4093, 4096)]


@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("skip", [0, 1])
def test_gemv_f32_bound(m, k, n, skip):
    r = np.random.default_rng(m * 131 + k + n)
    a = r.standard_normal((m, k)).astype(np.float32)
    b = (r.standard_normal((k, n)) * 0.05).astype(np.float32)
    print(f"gemv f32 {m}x{k}x{n} skip {skip}", flush=True)
    assert_gamma_bound(run(a, b, a_skip=skip, b_skip=skip), a, b)


@pytest.mark.parametrize("m,k,n", [(1, 37, 131), (16, 1536, 576), (4, 4096, 4099)])
def test_gemv_f32_integer_sums_and_in_place_residual(m, k, n):
    """Small integers: any order of summation is exact, so a row or column taken twice or left out
    shows. The residual is C itself: each element is read and written by one thread only."""
    r = np.random.default_rng(k)
    a = r.integers(-8, 9, size=(m, k)).astype(np.float32)
    b = r.integers(-8, 9, size=(k, n)).astype(np.float32)
    res = r.integers(-100, 101, size=(m, n)).astype(np.float32)
    want = (a.astype(np.int64) @ b.astype(np.int64) + res.astype(np.int64)).astype(np.float32)
    c = dev(res)
    epi = Epilogue(alpha=1.0, beta=1.0, residual=c.ptr)
    for _ in range(2):  # the arrival counters are left zero
        c.upload(res)
        same_bits(run(a, b, epi, c=c), want)


def test_gemv_f32_non_finite_values_stay_in_their_rows():
    m, k, n = 3, 1539, 70
    r = np.random.default_rng(9)
    a = r.standard_normal((m, k)).astype(np.float32)
    b = (r.standard_normal((k, n)) * 0.05).astype(np.float32)
    a[1, k - 1] = np.inf
    got = run(a, b)
    assert_gamma_bound(got[[0, 2]], a[[0, 2]], b)
    same_bits(got[1], np.where(b[k - 1] > 0, np.inf, -np.inf).astype(np.float32))
