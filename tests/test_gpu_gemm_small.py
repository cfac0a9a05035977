"""GEMM shapes with few blocks, on the tiles of 64 x 64 and 128 x 64 that take K whole, at the edges of
their ranges (row counts around 64, 128 and 256, ragged columns, block counts on both sides of the rules),
against float64 products of the stored operands: 16-bit operands multiply exactly in fp32, so the result
carries the fp32 summation error only, within K * 2^-24 of sum |x w|."""
from __future__ import annotations

import numpy as np
import pytest

import l0llm_amd as l0
from tests.helpers import dequant, stored

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", [l0.I8PC, l0.F16, l0.BF16])
@pytest.mark.parametrize("m,n,k", [(65, 64, 512), (66, 900, 896), (127, 8200, 576), (128, 8192, 1024), (129, 8190, 640), (129, 2052, 2048),
                                   (255, 1150, 896), (256, 896, 896), (300, 2044, 2048), (511, 3070, 2048), (1000, 1028, 576)])
def test_few_block_shapes_match_reference(device, suite, storage, m, n, k):
    rng = np.random.default_rng(m + n + k + storage)
    st, ws, s = stored(storage, rng.normal(0, 0.02, (n, k)).astype(np.float32))
    x = rng.normal(0, 1, (m, k)).astype(np.float32)
    if storage == l0.BF16:
        xs = (x.view(np.uint32) >> 16).astype(np.uint16)
        x = (xs.astype(np.uint32) << 16).view(np.float32)
    else:
        xs = x.astype(np.float16).view(np.uint16)
        x = xs.view(np.float16).astype(np.float32)
    up = lambda a: device.alloc_shared(np.ascontiguousarray(a))
    xb, wb, sb, yb = up(xs), up(ws), up(s) if s is not None else None, device.alloc((m * n + 16) * 4)
    yb.zero()
    if storage == l0.I8PC:
        suite.gemm_nk_i8pc(m, n, k, xb, wb, sb, yb, l0.F32)
    else:
        suite.gemm_nk(storage, m, n, k, xb, wb, yb, l0.F32)
    raw = yb.read().astype(np.float64)
    for b in (xb, wb, sb, yb):
        if b is not None:
            b.free()
    assert not np.any(raw[m * n:])
    w, xd = dequant(st, ws, s), x.astype(np.float64)
    want = xd @ w.T
    bound = k * 2.0**-24 * (np.abs(xd) @ np.abs(w).T) + 1e-30
    assert np.all(np.abs(raw[: m * n].reshape(m, n) - want) <= bound)
