"""Several fp32 activation rows through int8, fp16 and bf16 weights on the matrix cores, against the
oracle. Activations and weights enter the products with all their bits, so the results carry fp32
summation error only: a sum of K terms in any order is within K * 2^-24 of sum |x w| (2^-24 the fp32
rounding; the bound per element below), and far closer in the 2-norm."""
from __future__ import annotations

import numpy as np
import pytest

import l0llm_amd as l0
from tests.helpers import dequant, stored

pytestmark = pytest.mark.gpu


def _run(device, suite, storage, x, ws, s, n, y_dtype=l0.F32):
    rows, k = x.shape
    up = lambda a: device.alloc_shared(np.ascontiguousarray(a))
    wb, xb = up(ws), up(x)
    sb = up(s) if s is not None else None
    yb = device.alloc(rows * n * (4 if y_dtype == l0.F32 else 2) + 64)
    yb.zero()
    suite.gemv_nk(storage, rows, n, k, xb, l0.F32, wb, sb, yb, y_dtype)
    raw = yb.read(np.float32 if y_dtype == l0.F32 else np.float16).astype(np.float64)
    for b in (wb, xb, yb, sb):
        if b is not None:
            b.free()
    assert not np.any(raw[rows * n:]), "wrote past the output"
    return raw[: rows * n].reshape(rows, n)


def _check(got, x, storage, ws, s):
    w = dequant(storage, ws, s)
    want = x.astype(np.float64) @ w.T
    bound = x.shape[1] * 2.0**-24 * (np.abs(x.astype(np.float64)) @ np.abs(w).T) + 1e-30
    assert np.all(np.abs(got - want) <= bound)
    assert np.linalg.norm(got - want) <= 5e-7 * np.linalg.norm(want)


# rows: the edges of the 16-row groups and of the 64-row launches; n: 16-, 32- and 64-column blocks
# with whole and ragged last blocks (the block width follows the count); k: whole steps of 64, a step
# of which one or two 16-byte chunks are inside, fewer steps than waves.
@pytest.mark.parametrize("storage", [l0.I8PC, l0.F16, l0.BF16])
@pytest.mark.parametrize("rows,n,k", [
    (2, 1, 16), (2, 512, 64), (3, 37, 80), (15, 4096, 96), (16, 8190, 512), (17, 8191, 144), (31, 6145, 1040),
    (32, 9728, 208), (33, 100, 4864), (47, 6200, 528), (48, 33, 1024), (49, 8200, 272), (63, 6150, 560), (64, 16, 2048),
    (65, 70, 640), (130, 8192, 128)])
def test_rows_match_reference(device, suite, storage, rows, n, k):
    rng = np.random.default_rng(rows * 131 + n + k + storage)
    w = rng.normal(0, 0.02, (n, k)).astype(np.float32)
    x = rng.normal(0, 1, (rows, k)).astype(np.float32)
    st, ws, s = stored(storage, w)
    _check(_run(device, suite, storage, x, ws, s, n), x, st, ws, s)


@pytest.mark.parametrize("storage", [l0.I8PC, l0.F16, l0.BF16])
def test_rows_keep_all_bits_of_wide_ranging_activations(device, suite, storage):
    """Activations over 60 powers of two, an outlier under zero weights, fp16 subnormal weights and
    the int8 extremes: every element's own bits count, whatever stands beside it."""
    rng = np.random.default_rng(5 + storage)
    rows, n, k = 21, 200, 320
    x = (rng.normal(0, 1, (rows, k)) * 2.0 ** rng.integers(-30, 30, (rows, 1))).astype(np.float32)
    x[:, 0] = np.float32(1e30)
    if storage == l0.I8PC:
        st, ws = l0.I8PC, rng.integers(-128, 128, (n, k)).astype(np.int8)
        s = rng.uniform(1e-3, 1e-2, n).astype(np.float16).view(np.uint16)
        ws[:, 0] = 0
    else:
        w = rng.normal(0, 1e-6 if storage == l0.F16 else 0.02, (n, k)).astype(np.float32)
        w[:, 0] = 0
        st, ws, s = stored(storage, w)
    _check(_run(device, suite, storage, x, ws, s, n), x, st, ws, s)


@pytest.mark.parametrize("storage", [l0.I8PC, l0.F16, l0.BF16])
def test_rows_infinities_and_nan_stay_in_their_row(device, suite, storage):
    rng = np.random.default_rng(9)
    rows, n, k = 18, 96, 128
    w = np.abs(rng.normal(0, 0.02, (n, k))).astype(np.float32) + np.float32(0.01)
    x = rng.normal(0, 1, (rows, k)).astype(np.float32)
    st, ws, s = stored(storage, w)
    clean = _run(device, suite, storage, x, ws, s, n)
    x[3, 5], x[7, 100], x[17, 0], x[9, 64] = np.inf, np.nan, -np.inf, np.float32(3.4e38)
    got = _run(device, suite, storage, x, ws, s, n)
    assert np.all(got[3] == np.inf) and np.all(np.isnan(got[7])) and np.all(got[17] == -np.inf)
    if storage != l0.I8PC:  # an infinite weight: its output alone, for every row whose product is one
        big = ws.copy()
        big[11, 2] = 0x7C00 if storage == l0.F16 else 0x7F80
        inf = _run(device, suite, storage, np.abs(x[:3]) + 1, big, s, n)
        assert np.all(inf[:, 11] == np.inf) and np.all(np.isfinite(np.delete(inf, 11, axis=1)))
    others = [r for r in range(rows) if r not in (3, 7, 9, 17)]
    np.testing.assert_array_equal(got[others], clean[others])
    if storage != l0.I8PC:  # 3.4e38 has an fp32 product with weights below 1, as it had before its split
        assert np.all(np.isfinite(got[9]))


def test_rows_half_output_and_residual_free_store(device, suite):
    rng = np.random.default_rng(3)
    rows, n, k = 20, 515, 256
    w = rng.normal(0, 0.02, (n, k)).astype(np.float32)
    x = rng.normal(0, 1, (rows, k)).astype(np.float32)
    st, ws, s = stored(l0.F16, w)
    got = _run(device, suite, l0.F16, x, ws, s, n, l0.F16)
    want = x.astype(np.float64) @ dequant(st, ws, s).T
    assert np.all(np.abs(got - want) <= 2.0**-11 * np.abs(want) + 1e-6)  # one fp16 rounding


def test_rows_record_and_replay(device, suite):
    """A recorded multi-row call needs no memory of its own: it replays on new inputs."""
    rng = np.random.default_rng(4)
    rows, n, k = 13, 1152, 896
    w = rng.normal(0, 0.02, (n, k)).astype(np.float32)
    st, ws, s = stored(l0.I8PC, w)
    up = lambda a: device.alloc_shared(np.ascontiguousarray(a))
    x = rng.normal(0, 1, (rows, k)).astype(np.float32)
    wb, sb, xb, yb = up(ws), up(s), up(x), device.alloc(rows * n * 4)
    device.begin_recording()
    suite.gemv_nk(l0.I8PC, rows, n, k, xb, l0.F32, wb, sb, yb, l0.F32)
    device.end_recording()
    for i in range(3):
        x = rng.normal(0, 1, (rows, k)).astype(np.float32)
        xb.write(x)
        device.replay_recording()
        device.synchronize()
        _check(yb.read(np.float32, rows * n).reshape(rows, n).astype(np.float64), x, st, ws, s)
    for b in (wb, sb, xb, yb):
        b.free()
