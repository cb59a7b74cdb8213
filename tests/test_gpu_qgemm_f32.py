"""fp32 activations straight into the K-split GEMM kernel (k_qgemm_ks.hip): every tile and weight type
at ragged edges against float64 of the fp16-rounded activations, the entry points that choose between
it and the fp16 staging pass, and the rule that chooses.

Tolerances: test_gpu_qgemm_ks.py's (the operands are the same, fp32 accumulation in another order).
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import randn, rng
from test_gpu_epilogue import Epi, _launcher
from test_gpu_qgemm_ks import F16, KS, Q4, Q8, Op


def _f32(op, r):
    """The op's activations as fp32 values that round to its fp16 ones (moved by under half an ulp)."""
    x16 = op.dx.to_host().astype(np.float32)
    return (x16 * (1 + r.uniform(-0.99, 0.99, x16.shape) * 2.0 ** -12)).astype(np.float32), x16


@pytest.mark.gpu
@pytest.mark.parametrize("wt", [Q8, Q4, F16])
@pytest.mark.parametrize("cfg", range(3))
def test_every_tile(hip, port, cfg, wt):
    from aria_amd.device import DeviceArray
    r = rng(40 + cfg)
    for M, K, N in ((1, 64, 4), (33, 256, 100), (97, 1152, 196), (64, 2048, 64)):
        op = Op(hip, port, wt, M, K, N, 700 + 10 * cfg + wt)
        x, x16 = _f32(op, r)
        assert np.array_equal(x.astype(np.float16).astype(np.float32), x16)
        dx, dy = DeviceArray.from_host(x), DeviceArray.from_host(np.full((M, N), np.nan, np.float32))
        st = hip.lib().aria_hip_default_stream()
        e = Epi()
        e.mode, e.rows_per_batch = 2, M
        y0 = randn(r, (M, N))
        for epi in (None, C.byref(e)):
            if epi:
                dy = DeviceArray.from_host(y0)
            assert _launcher(hip)(dy.p, 0, dx.p, 0, wt, op.dq.p, op.ds.p if op.ds else None, op.db.p, M, K, N, KS + cfg, 0,
                                  epi, st) == 0
            hip.check(hip.lib().aria_hip_stream_sync(st))
            want = op.want + (y0 if epi else 0)
            bound = op.bound + (2.0 ** -23 * np.abs(y0) if epi else 0)
            y = dy.to_host()
            assert np.all(np.abs(y - want) <= bound), (M, K, N, np.max(np.abs(y - want) / bound))


@pytest.mark.gpu
@pytest.mark.parametrize("wt", [Q8, Q4, F16])
def test_entry_points(hip, port, wt):
    """Either side of the rule's lines (tiles in one round, K, an output over the activations): the
    allocating and the allocation-free entry agree in every bit, and with float64."""
    from aria_amd.device import DeviceArray
    L = hip.lib()
    r = rng(60 + wt)
    for M, K, N in ((256, 1024, 1024), (257, 1024, 1024), (1024, 256, 1024), (1025, 256, 1024), (40, 2048, 64),
                    (40, 2112, 64), (40, 96, 64), (64, 512, 512)):
        op = Op(hip, port, wt, M, K, N, 800 + wt)
        x, _ = _f32(op, r)
        for half in (0, 1):
            outs = []
            for fn in ("aria_hip_qlinear_dev", "aria_hip_qlinear_noalloc_dev"):
                for over in (False, True) if K == N and not half else (False,):
                    dx = DeviceArray.from_host(x)
                    dy = dx if over else DeviceArray((M, N), np.float16 if half else np.float32)
                    hip.check(getattr(L, fn)(dy.p, half, dx.p, 0, wt, op.dq.p, op.ds.p if op.ds else None, op.db.p, M, K,
                                             N, None))
                    hip.check(L.aria_hip_stream_sync(None))
                    outs.append((over, dy.to_host()))
            for over, y in outs:
                bound = op.bound + (2.0 ** -11 * np.abs(op.want) if half else 0)
                assert np.all(np.abs(y - op.want) <= bound), (M, K, N, over)
                ref = next(o for v, o in outs if v == over)
                assert np.array_equal(y, ref), (M, K, N, over)


def test_rule():
    """Over sizes, alignments and overlaps: direct only where the kernel takes the call (whole
    K-tiles, 16-byte rows and operands), in one round of tiles, and never onto its own input."""
    import aria_amd
    try:
        f = aria_amd.lib().aria_k_qgemm_f32_direct
    except (aria_amd.HipError, OSError) as e:
        pytest.skip(f"library not built: {e}")
    f.restype = C.c_int
    f.argtypes = [C.c_void_p, C.c_int] + [C.c_void_p, C.c_int] + [C.c_void_p] * 3 + [C.c_int] * 3
    base = 1 << 40   # addresses only compared
    x, y, q, s, b = (base + (i << 36) for i in range(5))
    seen = set()
    r = np.random.default_rng(5)
    for _ in range(20000):
        M, K, N = int(2 ** r.uniform(0, 13)), int(r.choice((32, 64, 96, 1024, 2048, 2112, 4096))), int(2 ** r.uniform(0, 13))
        wt, half = int(r.integers(3)), int(r.integers(2))
        off = [int(o) for o in r.choice((0, 0, 0, 0, 0, 0, 4, 8), 5)]
        d = f(y + off[0], half, x + off[1], wt, q + off[2], s + off[3], b + off[4], M, K, N)
        tiles = min(-(-M // 32) * -(-N // 32), -(-M // 32) * -(-N // 64), -(-M // 64) * -(-N // 64))
        ok = tiles <= 256 and K % 64 == 0 and K <= 2048 and N % 4 == 0 and not any(off[:3]) and not off[4] and (
            wt == F16 or not off[3])
        assert d == ok, (wt, M, K, N, off)
        seen.add(ok)
        if ok:   # an output whose last byte is x's first, and one that starts in x's last row
            ny = M * N * (2 if half else 4)
            assert not f(x, half, x, wt, q, s, b, M, K, N)
            assert not f(x + 16 * ((M * K * 4 - 4) // 16), half, x, wt, q, s, b, M, K, N)
            assert f(x + M * K * 4, half, x, wt, q, s, b, M, K, N)
            assert f(x - (ny + 15) // 16 * 16, half, x, wt, q, s, b, M, K, N)
    assert seen == {True, False}
