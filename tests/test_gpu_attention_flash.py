"""Attention of several rows with head_dim 64 or 128 on the matrix cores (AttentionFlashKernel),
against the same causal softmax in float64: row blocks and key ranges whole and partial, one or
several key ranges per row block, a key that only later rows see holding no finite value."""

import ctypes as C
import os

import numpy as np
import pytest

from hip_helpers import check, dev, lib

pytestmark = pytest.mark.gpu


def run(q, k, v, position):
    seq, heads, dim = q.shape
    out = dev(np.full(q.shape, 3.0, np.float32))
    scores = dev(np.zeros(k.shape[0], np.float32))
    qd, kd, vd = dev(q), dev(k), dev(v)
    check(lib().accel_hip_attention(qd.buffer, kd.buffer, vd.buffer, scores.buffer, out.buffer, seq, position, heads,
                                    k.shape[1], dim))
    return out.numpy()


def want(q, k, v, position):
    seq, heads, dim = q.shape
    group = heads // k.shape[1]
    out = np.empty(q.shape)
    for s in range(seq):
        for h in range(heads):
            kk, vv = (x[:position + s + 1, h // group].astype(np.float64) for x in (k, v))
            p = kk @ q[s, h].astype(np.float64) / np.sqrt(dim)
            e = np.exp(p - p.max())
            out[s, h] = e @ vv / e.sum()
    return out


def inputs(seq, position, heads, kv_heads, dim):
    r = np.random.default_rng(seq * 31 + position + dim)
    rows = seq + position
    return [r.standard_normal(s).astype(np.float32) for s in ((seq, heads, dim), (rows, kv_heads, dim),
                                                              (rows, kv_heads, dim))]


# (2, 0): fewer keys than one wave's step. (40, 700) and (5, 2100): the key range in several parts,
# the last ones short. (300, 0, 64 heads): more workgroups than CUs. 65537
# heads: more than a grid's second dimension holds.
@pytest.mark.parametrize("seq,position,heads,kv_heads,dim", [
    (2, 0, 3, 1, 64), (5, 0, 2, 2, 128), (16, 0, 4, 2, 64), (17, 3, 9, 3, 64), (33, 64, 3, 3, 128), (65, 1, 4, 1, 64),
    (40, 700, 6, 2, 64), (5, 2100, 4, 4, 128), (300, 0, 64, 8, 64), (3, 131, 32, 8, 128), (2, 1, 65537, 65537, 64)])
def test_attention_flash_against_float64(seq, position, heads, kv_heads, dim):
    q, k, v = inputs(seq, position, heads, kv_heads, dim)
    print(f"attention {seq} rows from {position}, {heads}/{kv_heads} heads of {dim}", flush=True)
    got = run(q, k, v, position)
    if heads > 65535:  # the first and the last heads are enough of them
        some = np.r_[0:20, heads - 20:heads]
        got, q, k, v = got[:, some], q[:, some], k[:, some], v[:, some]
    np.testing.assert_allclose(got, want(q, k, v, position), rtol=1e-5, atol=2e-6)


@pytest.mark.parametrize("position", [0, 900])
@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_attention_flash_masked_values_are_not_read(position, value):
    """Rows before a non-finite value's position keep their results; the rows that see it do not
    stay finite in that column, and only there."""
    q, k, v = inputs(21, position, 3, 1, 64)
    v[position + 9, 0, 7] = value
    got, exact = run(q, k, v, position), want(q, k, v, position)
    np.testing.assert_allclose(got[:9], exact[:9], rtol=1e-5, atol=2e-6)
    others = np.arange(64) != 7
    np.testing.assert_allclose(got[9:, :, others], exact[9:, :, others], rtol=1e-5, atol=2e-6)
    assert not np.isfinite(got[9:, :, 7]).any()


def test_attention_flash_takes_no_score_scratch():
    """4096 rows from position 16384, 32 heads: the kernel that keeps scores in memory would take 10.7
    GB for them. Only a few rows are compared (float64)."""
    hip = C.CDLL(os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "lib", "libamdhip64.so"))

    def free_bytes():
        check(lib().accel_hip_synchronize())
        free, total = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    seq, position, heads, dim = 4096, 16384, 32, 64
    r = np.random.default_rng(3)
    q = r.standard_normal((seq, heads, dim), dtype=np.float32)
    k, v = (r.standard_normal((seq + position, 1, dim), dtype=np.float32) for _ in range(2))
    out, scores = dev(np.zeros(q.shape, np.float32)), dev(np.zeros(len(k), np.float32))
    qd, kd, vd = dev(q), dev(k), dev(v)
    before = free_bytes()
    check(lib().accel_hip_attention(qd.buffer, kd.buffer, vd.buffer, scores.buffer, out.buffer, seq, position, heads, 1,
                                    dim))
    assert before - free_bytes() < 1 << 30
    got = out.numpy()
    for s in (0, 2049, seq - 1):
        exact = want(q[s:s + 1, :2], k[:position + s + 1], v[:position + s + 1], position + s)
        np.testing.assert_allclose(got[s, :2], exact[0], rtol=1e-5, atol=2e-6)
