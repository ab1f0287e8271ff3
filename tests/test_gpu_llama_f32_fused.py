"""The fp32 decode row's RMSNorm and SiLU * up inside the fp32 GEMVs (fuse bit 0) against the separate
passes, at the sizes where the GEMV changes form: one workgroup over all of K, K in splits, a K of no
whole batch, 1, 2 and 4 columns a lane, an unaligned row."""

import numpy as np
import pytest

from test_gpu_llama import Engine, _decode_row_logits

pytestmark = pytest.mark.gpu


def _weights(cfg, seed):
    r = np.random.default_rng(seed)
    H, I, V = cfg["hidden"], cfg["intermediate"], cfg["vocab"]
    kv = cfg["kv_heads"] * (H // cfg["heads"])
    mat = lambda o, i: (r.standard_normal((o, i)) * i ** -0.5).astype(np.float32)
    norm = lambda: r.normal(1.0, 0.1, H).astype(np.float32)
    out = [(1, -1, mat(V, H)), (3, -1, mat(V, H)), (2, -1, norm())]
    for layer in range(cfg["layers"]):
        out += [(4, layer, norm()), (5, layer, norm())]
        out += [(kind, layer, mat(o, i)) for kind, o, i in
                ((6, H, H), (7, kv, H), (8, kv, H), (9, H, H), (10, I, H), (11, I, H), (12, H, I))]
    return out


# (hidden, heads, kv_heads, intermediate): 576 whole and a ragged 1537 in splits; 66, with K's last
# batch short; 1024 x 5000 (two and four columns a lane, the norm over a split K); a hidden above
# the prologue's longest row, which keeps the separate passes, and an intermediate above it.
SIZES = [(576, 9, 3, 1536), (66, 3, 1, 1537), (1024, 16, 4, 5000), (4100, 82, 1, 64), (64, 1, 1, 4097)]


@pytest.mark.parametrize("hidden,heads,kv_heads,inter", SIZES)
def test_fp32_decode_row_fused_matches_separate_passes(hidden, heads, kv_heads, inter):
    cfg = dict(vocab=515, hidden=hidden, layers=2, heads=heads, kv_heads=kv_heads, intermediate=inter, context=32,
               eps=1e-5, rope_theta=10000.0)
    print(f"hidden {hidden} intermediate {inter}", flush=True)
    eng = Engine(cfg, _weights(cfg, hidden))
    try:
        prompt = np.random.default_rng(1).integers(0, cfg["vocab"], size=9).astype(np.int32)
        want = _decode_row_logits(eng, cfg, prompt, 6)
        got = _decode_row_logits(eng, cfg, prompt, 7)
        assert np.isfinite(got).all()
        # Two fp32 evaluations of about ten chained products of K <= 5000 terms: each within
        # sqrt(K) * 2^-24 = 4e-6 of its row's rms, a few of them added, on logits of rms 1.
        np.testing.assert_allclose(got, want, rtol=1e-4, atol=1e-4)
    finally:
        eng.close()
