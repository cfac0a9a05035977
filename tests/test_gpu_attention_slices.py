"""Split decode attention at the edges of its slices: one, two and four positions per slot, one or two
steps or a loop of them, a slot with no position, empty slices, every number of position slots in a
wave (head_dim 128, 64, 32 and 16) and every group size, against float64. Scores, weights and sums are
fp32: a sum over `seq` weights in any order is within seq * 2^-24, and a weight 2^x carries a few
2^-24 times its exponent's magnitude, so 2e-6 covers both at these lengths."""
from __future__ import annotations

import numpy as np
import pytest

import l0llm_amd as l0

pytestmark = pytest.mark.gpu


def _reference(q, k, v, hd, nh, nkv, seq):
    out = np.empty((nh, hd))
    q, k, v = q.astype(np.float64).reshape(nh, hd), k.astype(np.float64).reshape(-1, nkv, hd), v.astype(np.float64).reshape(-1, nkv, hd)
    for h in range(nh):
        s = k[:seq, h // (nh // nkv)] @ q[h] / np.sqrt(hd)
        p = np.exp(s - s.max())
        out[h] = (p / p.sum()) @ v[:seq, h // (nh // nkv)]
    return out.reshape(-1)


@pytest.mark.parametrize("cache", [l0.F16, l0.F32])
@pytest.mark.parametrize("hd,nh,nkv", [(128, 32, 8), (64, 14, 2), (64, 8, 8), (32, 8, 4), (16, 4, 2), (128, 7, 1)])
@pytest.mark.parametrize("seq,cap", [(1, 1), (15, 16), (17, 17), (33, 64), (64, 64), (65, 128), (128, 128), (129, 129),
                                     (64, 130), (200, 1000), (1000, 1000), (2049, 2049), (4097, 4100)])
def test_slices_match_reference(device, suite, cache, hd, nh, nkv, seq, cap):
    rng = np.random.default_rng(seq * 7 + cap + hd + nh)
    dt = np.float32 if cache == l0.F32 else np.float16
    k = rng.normal(0, 1, (cap, nkv * hd)).astype(dt)
    v = rng.normal(0, 1, (cap, nkv * hd)).astype(dt)
    k[seq:] = np.nan  # never read
    v[seq:] = np.nan
    q = rng.normal(0, 1, nh * hd).astype(np.float32)
    up = lambda a: device.alloc_shared(np.ascontiguousarray(a if a.dtype == np.float32 else a.view(np.uint16)))
    qb, kb, vb, ob = up(q), up(k), up(v), device.alloc(nh * hd * 4)
    suite.attention_execute(qb, kb, vb, ob, hd, nh, nkv, seq, cap, cache_dtype=cache)
    got = ob.read().astype(np.float64)
    for b in (qb, kb, vb, ob):
        b.free()
    want = _reference(q, k, v, hd, nh, nkv, seq)
    assert np.linalg.norm(got - want) <= 2e-6 * np.linalg.norm(want)
