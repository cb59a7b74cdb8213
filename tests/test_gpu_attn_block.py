"""A block's self-attention (aria_k_flash_attn_pf): how a launch is shared out (CPU), and that weights to
prefetch change none of its bits. Tolerance: test_gpu_attn_slices.py's.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import randn, rng
from test_gpu_attn_slices import _check


class Spans(C.Structure):
    """aria_prefetch_set (aria_amd/csrc/aria_hip_kernels.h)"""
    _fields_ = [("p", C.c_void_p * 12), ("bytes", C.c_size_t * 12), ("n", C.c_int)]


@pytest.mark.gpu
@pytest.mark.parametrize("BH,N", [(16, 172), (16, 480), (16, 564), (32, 450), (32, 710), (16, 1296), (32, 1296)])
def test_block_attention_same_bits_with_and_without_spans(hip, BH, N):
    """A block's self-attention by itself (nothing to prefetch) and inside a step (the next block's
    weights to prefetch) sums in the same order."""
    from aria_amd.device import DeviceArray
    L = hip.lib()
    f = L.aria_k_flash_attn_pf
    f.restype, f.argtypes = C.c_int, [C.c_void_p] * 4 + [C.c_int] * 5 + [C.POINTER(Spans), C.c_void_p]
    r = rng(N)
    q, k, v = (randn(r, (BH, N, 64)).astype(np.float16) for _ in range(3))
    dq, dk, dv = (DeviceArray.from_host(a) for a in (q, k, v))
    w = DeviceArray.from_host(np.zeros(1 << 20, np.uint8))
    st, outs = L.aria_hip_default_stream(), []
    for n in (0, 2):
        pf = Spans()
        pf.n = n
        for i in range(n):
            pf.p[i], pf.bytes[i] = w.p, w.nbytes
        do = DeviceArray.from_host(np.full((BH // 16, N, 1024), np.nan, np.float32))
        hip.check(f(dq.p, dk.p, dv.p, do.p, 0, BH, 16, N, N, C.byref(pf), st))
        hip.check(L.aria_hip_stream_sync(st))
        outs.append(do.to_host())
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    _check(outs[0].reshape(BH // 16, N, 16, 64).transpose(0, 2, 1, 3).reshape(BH, N, 64).astype(np.float64), q, k, v, 0)


def test_plan():
    """Over sizes: the form is the same with and without spans to prefetch, every query and head has a
    workgroup, prefetch workgroups only fill idle CUs, and the four-slice forms have them too where
    many are idle."""
    import aria_amd
    try:
        f = aria_amd.lib().aria_k_flash_attn_plan
    except (aria_amd.HipError, OSError) as e:
        pytest.skip(f"library not built: {e}")
    f.restype, f.argtypes = None, [C.c_int] * 6 + [C.POINTER(C.c_int * 4)]

    def plan(*a):
        o = (C.c_int * 4)()
        f(*a, C.byref(o))
        return list(o)

    r = np.random.default_rng(4)
    seen = set()
    for _ in range(20000):
        BH, Nq, Nk = 16 * int(r.integers(1, 5)), int(2 ** r.uniform(0, 12)), int(2 ** r.uniform(0, 12))
        a, b, c = plan(BH, Nq, Nk, 1, 0, 256), plan(BH, Nq, Nk, 1, 1, 256), plan(BH, Nq, Nk, 0, 0, 256)
        assert a[:3] == b[:3] and a[3] == c[3] == 0
        for ks, qw, T, npw in (a, b, c):
            assert T == BH * -(-Nq // (32 * qw)) and qw <= {1: 4, 2: 6, 4: 3}[ks]
            idle = 256 - -(-T // 8) * 8
            assert npw == 0 or (npw == idle >= (96 if ks == 4 else 8) and Nk > 448)
        seen |= {("block", *b[:2], b[3] > 0), ("plain", *c[:2], False)}
    assert {("plain", 4, 3, False), ("plain", 4, 1, False), ("block", 2, 6, True), ("block", 4, 2, False),
            ("block", 4, 2, True)} <= seen
    assert not any(s[:3] == ("block", 4, 3) for s in seen)
