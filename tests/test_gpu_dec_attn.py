"""The decoder's chunk attention (k_dec_attn_mfma, k_dec.hip) against float64: 34 tokens, 12 heads of
64, o = (softmax(q k^T / 8) - softmax(qd kd^T / 8)) v, fp16 out.

Tolerance: the output's fp16 rounding, and fp32 arithmetic in the probabilities: a score is off by
at most 64 roundings of its absolute sum, an exponential and the sums by a few tens more.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import randn, rng

pytestmark = pytest.mark.gpu

S, H, D = 34, 12, 64


def _run(hip, x, nch):
    from aria_amd.device import DeviceArray
    f = hip.lib().aria_k_dec_attn
    f.restype, f.argtypes = C.c_int, [C.c_void_p, C.c_void_p, C.c_int, C.c_void_p]
    dx = DeviceArray.from_host(x)
    dy = DeviceArray.from_host(np.full((nch * S + 2, H * D), 7, np.float16))
    st = hip.lib().aria_hip_default_stream()
    assert f(dy.p, dx.p, nch, st) == 0
    hip.check(hip.lib().aria_hip_stream_sync(st))
    y = dy.to_host()
    assert np.all(y[nch * S:] == 7)   # nothing past the chunks' rows
    return y[:nch * S].reshape(nch, S, H, D).transpose(0, 2, 1, 3).astype(np.float64)


def _want(x, nch):
    q, k, v, qd, kd = x.astype(np.float64).reshape(nch, S, 5, H, D).transpose(2, 0, 3, 1, 4)

    def probs(q, k):
        s = q @ k.swapaxes(-1, -2) / 8
        e = np.exp(s - s.max(-1, keepdims=True))
        mag = (np.abs(q) @ np.abs(k).swapaxes(-1, -2) / 8).max(-1, keepdims=True)
        return e / e.sum(-1, keepdims=True), 2 * 2.0 ** -24 * (64 * mag + 64)
    p0, e0 = probs(q, k)
    p1, e1 = probs(qd, kd)
    want = (p0 - p1) @ v
    a = np.abs(v)
    return want, e0 * (p0 @ a) + e1 * (p1 @ a) + 2.0 ** -11 * np.abs(want) + 2.0 ** -25


@pytest.mark.parametrize("nch,scale", [(1, 1.0), (2, 3.0), (5, 0.1), (23, 1.0)])
def test_chunks(hip, nch, scale):
    x = randn(rng(nch), (nch * S, 5 * H * D), scale)
    want, tol = _want(x, nch)
    got = _run(hip, x, nch)
    assert np.all(np.abs(got - want) <= tol), np.max(np.abs(got - want) / tol)


@pytest.mark.parametrize("row", [0, 17, 32, 33])
def test_non_finite_values(hip, row):
    """inf in v makes its dim NaN (inf - inf), NaN in k or a large score its head; other heads and
    chunks are untouched. The rows past the chunk that the padding repeats add nothing."""
    x = randn(rng(3), (3 * S, 5 * H * D))
    clean = _run(hip, x, 3)
    for sec, bad in ((2, np.inf), (1, np.nan), (4, np.nan), (4, -np.inf)):
        y = x.copy()
        h, d = 5, 9
        y[S + row, sec * H * D + h * D + d] = bad
        got = _run(hip, y, 3)
        other = np.ones((3, H), bool)
        other[1, h] = False
        assert np.array_equal(got[other], clean[other])
        if sec == 2:
            assert np.isnan(got[1, h, :, d]).all()
            keep = np.arange(D) != d
            assert np.array_equal(got[1, h][:, keep], clean[1, h][:, keep])
        elif np.isnan(bad):
            assert np.isnan(got[1, h]).all()
        else:   # score -inf (weight zero) where qd is positive, +inf (NaN) where it is negative
            qd = y[S:2 * S, 3 * H * D + h * D + d]
            assert np.isnan(got[1, h][qd < 0]).all() and np.isfinite(got[1, h][qd > 0]).all()
