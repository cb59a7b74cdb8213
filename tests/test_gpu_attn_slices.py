"""The attention's four-slice form (k_attn.hip: few queries, the keys shared by four slices of one,
two or three query waves) against float64 softmax(q k^T / 8) v of the same fp16 operands.

Tolerance: the probabilities are rounded to fp16 (2^-11 of each, or 2^-25 where they are subnormal;
the largest is at least 1) and divided by the sum of the rounded ones, so both roundings count once
in the product and once in the sum; the fp32 scores and exponentials add under 1e-4 of a
probability, the fp16 output 2^-11 of the value.
"""
from __future__ import annotations

import numpy as np
import pytest

from conftest import randn, rng

pytestmark = pytest.mark.gpu


def _run(hip, q, k, v, H, out_f16):
    from aria_amd.device import DeviceArray
    BH, Nq, _ = q.shape
    dq, dk, dv = (DeviceArray.from_host(a) for a in (q, k, v))
    do = DeviceArray.from_host(np.full((BH // H, Nq, H * 64), np.nan, np.float16 if out_f16 else np.float32))
    hip.check(hip.lib().aria_hip_flash_attention_dev(dq.p, dk.p, dv.p, do.p, int(out_f16), BH // H, H, Nq, k.shape[1], 64,
                                                     None))
    hip.check(hip.lib().aria_hip_stream_sync(None))
    return do.to_host().reshape(BH // H, Nq, H, 64).transpose(0, 2, 1, 3).reshape(BH, Nq, 64).astype(np.float64)


def _check(got, q, k, v, out_f16):
    q, k, v = (a.astype(np.float64) for a in (q, k, v))
    s = q @ k.transpose(0, 2, 1) / 8
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    want = p @ v
    tol = (2.0 ** -10 + 1e-4) * (p @ np.abs(v)) + 2 * k.shape[1] * 2.0 ** -25 * np.abs(v).max()
    tol += 2.0 ** -11 * np.abs(want) if out_f16 else 0
    assert np.all(np.abs(got - want) <= tol), np.max(np.abs(got - want) / tol)


# one query wave per slice (a workgroup per 32 queries fits the CUs), two (per 64) and, on 512 and
# 1000 keys, three (per 96)
@pytest.mark.parametrize("BH,H,Nq", [(64, 16, 257), (64, 16, 384), (2, 1, 1), (4, 2, 31), (2, 2, 33), (16, 16, 172), (64, 16, 130), (64, 16, 255)])
@pytest.mark.parametrize("Nk", [65, 128, 129, 172, 256, 257, 512, 513, 1000])
def test_lengths(hip, BH, H, Nq, Nk):
    r = rng(BH + Nq + Nk)
    q, k, v = (randn(r, (BH, n, 64)).astype(np.float16) for n in (Nq, Nk, Nk))
    for out_f16 in (0, 1):
        _check(_run(hip, q, k, v, H, out_f16), q, k, v, out_f16)


@pytest.mark.parametrize("BH,Nq,Nk", [(4, 40, 256), (64, 130, 256), (64, 300, 512)])
def test_slices_of_keys_that_score_minus_infinity(hip, BH, Nq, Nk):
    """The second slice's keys all score -inf: weight zero, as if they were not there. All keys so:
    not a number."""
    r = rng(7)
    q, k, v = (randn(r, (BH, n, 64)).astype(np.float16) for n in (Nq, Nk, Nk))
    q[:, :, 0] = np.abs(q[:, :, 0]) + np.float16(0.5)
    k[:, Nk // 4:Nk // 2, 0] = -np.inf
    left = np.r_[0:Nk // 4, Nk // 2:Nk]
    _check(_run(hip, q, k, v, 4, 0), q, k[:, left], v[:, left], 0)
    k[:, :, 0] = -np.inf
    assert np.isnan(_run(hip, q, k, v, 4, 0)).all()
