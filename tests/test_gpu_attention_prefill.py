"""Causal prefill attention at the edges of its tiles, for both caches, against float64: one token, a last
block of query vectors that is partly empty, chunks that start inside, at and just past a step of 16 or 64
positions, tokens of one block on both sides of it, group sizes that do not divide the block, large groups.
fp32 cache: fp32 operands and sums, 2e-6 as the decode kernel's. fp16 cache: the scaled q and the weights
are rounded to fp16 (2^-12 relative at most each; the scores' error, |q k| 2^-12 over random signs, moves
a weight by about as much), which 1e-3 in the 2-norm covers."""
from __future__ import annotations

import numpy as np
import pytest

import l0llm_amd as l0

pytestmark = pytest.mark.gpu


def _reference(q, k, v, hd, nh, nkv, pos0, tokens):
    q, k, v = q.astype(np.float64).reshape(tokens, nh, hd), k.astype(np.float64).reshape(-1, nkv, hd), v.astype(np.float64).reshape(-1, nkv, hd)
    out = np.empty((tokens, nh, hd))
    n = pos0 + tokens
    see = np.arange(n)[None, :] <= pos0 + np.arange(tokens)[:, None]
    for h in range(nh):
        s = np.where(see, q[:, h] @ k[:n, h // (nh // nkv)].T / np.sqrt(hd), -np.inf)
        p = np.exp(s - s.max(axis=1, keepdims=True))
        out[:, h] = (p / p.sum(axis=1, keepdims=True)) @ v[:n, h // (nh // nkv)]
    return out.reshape(tokens, nh * hd)


@pytest.mark.parametrize("cache", [l0.F16, l0.F32])
@pytest.mark.parametrize("hd,nh,nkv", [(128, 8, 2), (64, 14, 2), (64, 3, 3), (128, 16, 1), (64, 20, 1)])
@pytest.mark.parametrize("pos0,tokens", [(0, 1), (0, 2), (15, 1), (16, 3), (1, 15), (0, 17), (63, 2), (64, 33), (37, 100), (130, 65), (0, 300)])
def test_prefill_matches_reference(device, suite, cache, hd, nh, nkv, pos0, tokens):
    rng = np.random.default_rng(pos0 * 1000 + tokens + hd + nh)
    n, cap = pos0 + tokens, pos0 + tokens + 5
    dt = np.float32 if cache == l0.F32 else np.float16
    k = rng.normal(0, 1, (cap, nkv * hd)).astype(dt)
    v = rng.normal(0, 1, (cap, nkv * hd)).astype(dt)
    k[n:] = np.nan  # never read
    v[n:] = np.nan
    q = rng.normal(0, 1, (tokens, nh * hd)).astype(np.float32)
    up = lambda a: device.alloc_shared(np.ascontiguousarray(a if a.dtype == np.float32 else a.view(np.uint16)))
    qb, kb, vb, ob = up(q), up(k), up(v), device.alloc((tokens * nh * hd + 16) * 4)
    ob.zero()
    suite.attention_execute_prefill(qb, kb, vb, ob, hd, nh, nkv, pos0, tokens, cap, cache_dtype=cache)
    raw = ob.read().astype(np.float64)
    for b in (qb, kb, vb, ob):
        b.free()
    assert not np.any(raw[tokens * nh * hd:])
    got, want = raw[: tokens * nh * hd].reshape(tokens, nh * hd), _reference(q, k, v, hd, nh, nkv, pos0, tokens)
    assert np.linalg.norm(got - want) <= (2e-6 if cache == l0.F32 else 1e-3) * np.linalg.norm(want)
