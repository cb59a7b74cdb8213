"""The decoder's mapping convolution on split operands (k_dec_split, k_dec_split_w, k_dec_map in
k_dec.hip) against a float64 convolution of the same fp32 values.

Bound: the three bf16 parts hold all 24 bits of a value, each rounded to the nearest, and the three
part products left out are together at most 2^-24 (1 + 2^-10) of each product. The sums round in fp32:
144 additions of the large part and 720 of the small parts (2^-7 of it), each by at most 2^-24 of the
running sum, which is at most the sum of absolute products. Hence
|error| <= (2^-24 + 152 * 2^-24) sum |x w| + 2^-23 |result|.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import randn, rng

pytestmark = pytest.mark.gpu


def _run(hip, seq, W, b, T, form):
    from aria_amd.device import DeviceArray
    L = hip.lib()
    for name, args in (("aria_k_dec_split", [C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_void_p]),
                       ("aria_k_dec_split_w", [C.c_void_p, C.c_void_p, C.c_void_p]),
                       ("aria_k_dec_map", [C.c_void_p] * 4 + [C.c_int, C.c_int, C.c_void_p])):
        getattr(L, name).restype, getattr(L, name).argtypes = C.c_int, args
    st = L.aria_hip_default_stream()
    Lt, Lout = 16 * T, 16 * (T + T % 2)
    dseq, dW, db = DeviceArray.from_host(seq), DeviceArray.from_host(W), DeviceArray.from_host(b)
    xs, ws = DeviceArray((Lt + 2) * 4608, np.uint8), DeviceArray(512 * 72 * 192, np.uint8)
    da = DeviceArray.from_host(np.full((2, Lt * 256), np.nan, np.float32))
    hip.check(L.aria_k_dec_split_w(ws.p, dW.p, st))
    hip.check(L.aria_k_dec_split(xs.p, dseq.p, Lt, Lout, st))
    hip.check(L.aria_k_dec_map(da.p, xs.p, ws.p, db.p, Lt, form, st))
    hip.check(L.aria_hip_stream_sync(st))
    return da.to_host()


def _columns(seq, T):
    """the convolution's input rows [16 T, 768, 3] in float64"""
    Lt, Lout = 16 * T, 16 * (T + T % 2)
    pos = np.arange(Lout)
    f = np.zeros((Lout + 2, 768))
    f[1:-1] = seq[(pos // 16) * 17 + 1 + pos % 16]
    return np.stack([f[j:j + Lt] for j in range(3)], axis=2)


def _audio(y, T):
    return y.reshape(16 * T, 2, 256).transpose(1, 0, 2).reshape(2, 4096 * T)


@pytest.mark.parametrize("form", [0, 1, 2, 3])
@pytest.mark.parametrize("T", [1, 2, 5, 13])   # one tile with rows to spare, ragged tiles, odd T (a pad frame)
def test_map_matches_float64(hip, T, form):
    r = rng(60 + T)
    seq = randn(r, (17 * (T + T % 2), 768))
    seq *= 10.0 ** r.uniform(-3, 2, (seq.shape[0], 1)).astype(np.float32)   # rows of very different scale
    W, b = randn(r, (512, 2304), 0.02), randn(r, 512, 0.05)
    x = _columns(seq, T).reshape(16 * T, -1)
    w = W.astype(np.float64)
    want = _audio(x @ w.T + b, T)
    bound = _audio((2.0 ** -24 + 152 * 2.0 ** -24) * (np.abs(x) @ np.abs(w).T), T) + 2.0 ** -23 * np.abs(want) + 1e-12
    got = _run(hip, seq, W, b, T, form)
    assert np.all(np.abs(got - want) <= bound), np.max(np.abs(got - want) / bound)
    assert np.array_equal(_run(hip, seq, W, b, T, form), got)


def _low_ones(r, shape, sign):
    """values whose low 16 mantissa bits are all ones, or one bit around half of them: the remainders of
    the parts are as large as they get"""
    m = r.integers(0, 128, shape, np.uint32) << np.uint32(16) | r.choice(np.array([0xFFFF, 0x7FFF, 0x8001, 0xFF7F], np.uint32), shape)
    v = (m | np.uint32(127 << 23)).view(np.float32)
    return v if sign is None else v * r.choice(np.array(sign, np.float32), shape)


@pytest.mark.parametrize("form", [1, 2, 3])
@pytest.mark.parametrize("T", [1, 12])
def test_map_one_product(hip, T, form):
    """Every output is a single product, so nothing averages out: the products left out (2^-24 of it),
    the five small ones' roundings (2^-24 of 2^-7 of it each) and the final sum's."""
    r = rng(80 + T)
    seq = np.zeros((17 * (T + T % 2), 768), np.float32)
    seq[np.arange(seq.shape[0]), r.integers(0, 768, seq.shape[0])] = _low_ones(r, seq.shape[0], (1, -1))
    W = np.zeros((512, 768, 3), np.float32)
    W[:, :, 1] = _low_ones(r, (512, 768), (1, -1))   # the middle tap: one feature row an output
    W = W.reshape(512, 2304)
    b = np.zeros(512, np.float32)
    want = _audio(_columns(seq, T).reshape(16 * T, -1) @ W.astype(np.float64).T, T)
    got = _run(hip, seq, W, b, T, form)
    assert np.all(want != 0)
    assert np.max(np.abs(got / want - 1)) <= 2.1 * 2.0 ** -24


@pytest.mark.parametrize("form", [1, 2, 3])
def test_map_products_of_one_sign(hip, form):
    """All products positive, low mantissa bits all ones: what is left out of them adds up."""
    T = 5
    r = rng(90)
    seq = _low_ones(r, (17 * (T + T % 2), 768), None)
    W, b = _low_ones(r, (512, 2304), None), np.zeros(512, np.float32)
    x, w = _columns(seq, T).reshape(16 * T, -1), W.astype(np.float64)
    want = _audio(x @ w.T, T)
    got = _run(hip, seq, W, b, T, form)
    bound = (153 * 2.0 ** -24 + 2.0 ** -23) * want
    assert np.all(np.abs(got - want) <= bound), np.max(np.abs(got - want) / bound)


@pytest.mark.parametrize("form", [1, 2, 3])
def test_map_keeps_the_class_of_non_finite_values(hip, form):
    """infinities, NaN and values near the largest float come out as in an fp32 product"""
    T = 4
    r = rng(71)
    seq = randn(r, (17 * T, 768))
    W, b = np.abs(randn(r, (512, 2304), 0.02)) + 1e-3, randn(r, 512, 0.05)
    seq[5, 3], seq[25, 9], seq[45, 100], seq[60, 7] = np.inf, np.nan, -np.inf, 3.3e38
    with np.errstate(invalid="ignore", over="ignore"):
        want = _audio(_columns(seq, T).reshape(16 * T, -1) @ W.astype(np.float64).T + b, T).astype(np.float32)
    got = _run(hip, seq, W, b, T, form)
    assert np.isinf(want).any() and np.isnan(want).any() and np.nanmax(np.abs(want[np.isfinite(want)])) > 1e35
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    fin = np.isfinite(want)
    assert np.allclose(got[fin], want[fin], rtol=1e-4, atol=1e-3)
