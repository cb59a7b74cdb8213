"""The K-split GEMM kernel (k_qgemm_ks.hip): every configuration and weight type against float64
at ragged edges, its fused epilogues against the other GEMM kernels', and the rule that picks it.

Tolerances: the operands are the values the kernel multiplies (fp16 activations, Q8 and fp16
weights exact), so only the fp32 accumulation differs from float64: K products round by at most
K 2^-24 of their absolute sum. A Q4 weight is also rounded to fp16 (2^-11 of it) from
n step + (min - 1024 step), each operation rounded in fp32 at magnitude up to 1040 step. W8A8 sums are
exact integers; three fp32 roundings remain.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from conftest import randn, rng
from test_gpu_epilogue import Epi, _launcher, _rope_tables

Q8, Q4, F16, I8 = 0, 1, 2, 3
KS = 100           # aria_k_qgemm_e tiles / aria_k_gemm_i8_t fm: KS + configuration
KS_FN = (1, 2, 2, 2, 2)


def _i8_launcher(hip):
    f = hip.lib().aria_k_gemm_i8_t
    f.restype = C.c_int
    f.argtypes = [C.c_void_p, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p,
                  C.c_int, C.c_int, C.c_int, C.c_int, C.c_int, C.POINTER(Epi), C.c_void_p]
    return f


class Op:
    """One product's device operands and its float64 value."""

    def __init__(self, hip, port, wt, M, K, N, seed):
        from aria_amd.device import DeviceArray
        r = rng(seed)
        x = randn(r, (M, K)); W = randn(r, (N, K), 0.05); b = randn(r, N)
        self.hip, self.wt, self.M, self.K, self.N = hip, wt, M, K, N
        x16 = x.astype(np.float16)
        x64 = x16.astype(np.float64)
        self.ds = self.dsx = None
        rounding = np.zeros((N, K))
        if wt == F16:
            q = W.astype(np.float16)
            w64 = q.astype(np.float64)
        elif wt == Q4:
            q, s = port.q4_quant(W)
            w64 = port.q4_dequant(q, s, K).astype(np.float64)
            step = np.repeat(s.reshape(N, -1, 2)[:, :, 1].astype(np.float64), 32, axis=1)[:, :K]
            rounding = 2.0 ** -11 * np.abs(w64) + 2 * 1040 * step * 2.0 ** -24
        else:
            q, s = port.q8_quant(W)
            w64 = q.astype(np.float64) * s.astype(np.float64)[:, None]
        if wt != F16:
            self.ds = DeviceArray.from_host(s)
        if wt == I8:
            amax = np.abs(x).max(axis=1)
            inv = (np.float32(127) / amax)[:, None]
            xq = np.clip(np.rint(x * inv), -127, 127).astype(np.int8)
            sx = (amax / np.float32(127)).astype(np.float32)
            self.dx, self.dsx = DeviceArray.from_host(xq), DeviceArray.from_host(sx)
            x64 = xq.astype(np.float64) * sx.astype(np.float64)[:, None]
        else:
            self.dx = DeviceArray.from_host(x16)
        self.dq, self.db = DeviceArray.from_host(q), DeviceArray.from_host(b)
        self.want = x64 @ w64.T + b.astype(np.float64)
        self.bound = K * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T) + 4 * 2.0 ** -24 * np.abs(self.want) + 1e-7
        self.bound += np.abs(x64) @ rounding.T

    def run(self, tiles, dy=None, epi=None, gelu=0, y_f16=0):
        st = self.hip.lib().aria_hip_default_stream()
        e = C.byref(epi) if epi is not None else None
        y = dy.p if dy is not None else None
        if self.wt == I8:
            rc = _i8_launcher(self.hip)(y, y_f16, self.dx.p, self.dsx.p, self.dq.p, self.ds.p, self.db.p, self.M, self.K,
                                        self.N, tiles, gelu, e, st)
        else:
            rc = _launcher(self.hip)(y, y_f16, self.dx.p, 1, self.wt, self.dq.p, self.ds.p if self.ds else None,
                                     self.db.p, self.M, self.K, self.N, tiles, gelu, e, st)
        if rc == 0:
            self.hip.check(self.hip.lib().aria_hip_stream_sync(st))
        return rc


@pytest.mark.gpu
@pytest.mark.parametrize("wt", [Q8, Q4, F16, I8])
@pytest.mark.parametrize("cfg", range(5))
def test_every_configuration(hip, port, cfg, wt):
    """One row, fewer K-tiles than waves, ragged M and N, a K that leaves waves uneven shares."""
    from aria_amd.device import DeviceArray
    for M, K, N in ((1, 128, 32), (33, 256, 100), (97, 1152, 196), (64, 4096, 64)):
        op = Op(hip, port, wt, M, K, N, 900 + 10 * cfg + wt)
        dy = DeviceArray.from_host(np.full((M, N), np.nan, np.float32))
        assert op.run(KS + cfg, dy) == 0
        y = dy.to_host()
        assert np.all(np.abs(y - op.want) <= op.bound), (M, K, N, np.max(np.abs(y - op.want) / op.bound))
        for _ in range(3):   # a fixed order of summation: the same bits every time
            assert op.run(KS + cfg, dy) == 0
            assert np.array_equal(dy.to_host().view(np.uint32), y.view(np.uint32))


def _near(a, b, half):
    """The same sums in another fp32 order, then perhaps one fp16 rounding."""
    a, b = a.astype(np.float64), b.astype(np.float64)
    tol = 2e-5 * np.max(np.abs(b)) + (2.0 ** -10 * np.abs(b) if half else 0.0)
    return np.all(np.abs(a - b) <= tol)


@pytest.mark.gpu
@pytest.mark.parametrize("wt", [Q8, Q4, F16, I8])
def test_epilogues_match_the_other_kernels(hip, port, wt):
    """STORE (fp32, fp16, GELU), GLU, GATE_RES (a tile over three sequences), ADD, HEADS with RoPE."""
    from aria_amd.device import DeviceArray
    # the large-tile kernel's 64 x 256 (the same Q4 unpack), the LDS-operand kernel's 128 x 128,
    # k_gemm_i8's 64 x 256
    other = {Q8: 15, Q4: 15, F16: 2, I8: 2}[wt]
    heads, S = 2, 45
    M, K, N = 3 * S, 384, 3 * heads * 64
    op = Op(hip, port, wt, M, K, N, 970 + wt)
    r = rng(980)
    y0, add2 = randn(r, (M, N)), DeviceArray.from_host(randn(r, (M, N)))
    gate, gate2 = DeviceArray.from_host(randn(r, (1, N))), DeviceArray.from_host(randn(r, (3, N)))
    cos_t, sin_t = (DeviceArray.from_host(t) for t in _rope_tables(S, 32))
    nw = DeviceArray.from_host((1 + 0.1 * randn(r, 64)).astype(np.float32))

    def res(cfg, mode, shape, dtype, init=None, gelu=0):
        dy = DeviceArray.from_host(init if init is not None else np.zeros(shape, dtype))
        e = Epi()
        e.mode, e.rows_per_batch = mode, S
        if mode == 1:
            e.gate, e.gate2, e.gate2_bs = gate.p, gate2.p, N
        if mode == 2:
            e.add2 = add2.p
        outs = [dy]
        if mode == 3:
            outs = [DeviceArray((3, heads, S, 64), np.float16) for _ in range(3)]
            e.heads, e.nsec, e.rot, e.eps, e.cos_t, e.sin_t = heads, 3, 32, 1e-6, cos_t.p, sin_t.p
            for i in range(3):
                e.kind[i], e.dst[i] = i, outs[i].p
            e.w[0], e.w[1] = nw.p, None
        assert op.run(cfg, dy, e, gelu, int(dtype == np.float16)) == 0
        return [o.to_host() for o in outs]

    for cfg in range(5):
        for mode, shape, dtype, init, gelu in ((0, (M, N), np.float32, None, 0), (0, (M, N), np.float16, None, 1),
                                               (4, (M, N // 2), np.float16, None, 0), (4, (M, N // 2), np.float32, None, 0),
                                               (1, (M, N), np.float32, y0, 0), (2, (M, N), np.float32, y0, 0),
                                               (3, (M, N), np.float32, None, 0)):
            if mode == 3 and KS_FN[cfg] != 2:   # a head's 64 columns must sit in one tile
                dy = DeviceArray((M, N))
                e = Epi()
                e.mode, e.rows_per_batch, e.heads, e.nsec = 3, S, heads, 3
                for i in range(3):
                    e.dst[i] = dy.p
                assert op.run(KS + cfg, dy, e) != 0
                continue
            a = res(KS + cfg, mode, shape, dtype, init, gelu)
            b = res(other, mode, shape, dtype, init, gelu)
            for u, v in zip(a, b):
                assert _near(u, v, u.dtype == np.float16), (wt, cfg, mode, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("cfg", range(5))
def test_decoder_epilogues(hip, cfg):
    import test_gpu_epilogue as E
    for rot in (0, 8, 32):
        E.test_dyt_rope_epilogue(hip, rot, KS + cfg)
    E.test_add_dyt_epilogue(hip, KS + cfg)


def test_pick_names_a_kernel_that_takes_the_shape():
    """qgemm_pick over every weight type, with and without HEADS: a K-split configuration that
    exists (two 32-column blocks for HEADS), or a large-tile one whose K halves are whole."""
    import aria_amd
    try:
        L = aria_amd.lib()
    except (aria_amd.HipError, OSError) as e:
        pytest.skip(f"library not built: {e}")
    pick = L._Z10qgemm_pickibiiii
    pick.restype = C.c_int
    pick.argtypes = [C.c_int, C.c_bool, C.c_int, C.c_int, C.c_int, C.c_int]
    r = np.random.default_rng(3)
    seen = set()
    for _ in range(20000):
        wt, heads = int(r.integers(4)), bool(r.integers(2))
        unit = 128 if wt == I8 else 64
        M, K, N = int(2 ** r.uniform(0, 15)), unit * int(r.integers(1, 65)), 64 * int(r.integers(1, 130))
        even = (K // unit) % 2 == 0
        if wt == F16:
            cur = -1 if heads else int(r.integers(5))
        elif wt == I8:
            cur = (5 if N <= 1024 and even else 1) if heads else (4 if N <= 1024 and even else 2)
        else:
            cur = (6 if N <= 1024 and even else 8) if heads else (5 if N <= 1024 and even else 1)
        c = pick(wt, heads, M, N, K, cur)
        seen.add((wt, heads, c))
        if c >= KS:
            assert c - KS < len(KS_FN) and (not heads or KS_FN[c - KS] == 2)
        elif c != cur:
            assert wt != F16
            halves = (4, 5) if wt == I8 else (5, 6)
            assert c not in halves or even
            assert not heads or c in ((1, 5) if wt == I8 else (6, 8))
    assert {c for _, _, c in seen} >= {KS + i for i in range(5)}


@pytest.mark.gpu
@pytest.mark.parametrize("wt", [Q8, Q4, F16])
def test_in_place(hip, port, wt):
    """fp16 activations overwritten by the output (K = N, one column tile): as with an output of its own."""
    from aria_amd.device import DeviceArray
    L = hip.lib()
    for M, K in ((33, 64), (172, 128), (1000, 64), (2592, 128)):
        op = Op(hip, port, wt, M, K, K, 900 + wt)
        x = op.dx.to_host()
        for fn in ("aria_hip_qlinear_dev", "aria_hip_qlinear_noalloc_dev"):
            d = DeviceArray.from_host(x)
            hip.check(getattr(L, fn)(d.p, 1, d.p, 1, wt, op.dq.p, op.ds.p if op.ds else None, op.db.p, M, K, K, None))
            hip.check(L.aria_hip_stream_sync(None))
            bound = op.bound + 2.0 ** -11 * np.abs(op.want) + 2.0 ** -25
            assert np.all(np.abs(d.to_host() - op.want) <= bound), (M, K, fn)


def test_route_keeps_whole_rows_in_place():
    """An output that overlaps fp16 activations never takes the K-split kernel's narrow tiles, which
    others take at these sizes; one that only touches them does."""
    import aria_amd
    try:
        f = aria_amd.lib().aria_k_qgemm_route
    except (aria_amd.HipError, OSError) as e:
        pytest.skip(f"library not built: {e}")
    f.restype = C.c_int
    f.argtypes = [C.c_void_p, C.c_int] + [C.c_void_p, C.c_int] + [C.c_void_p] * 3 + [C.c_int] * 3
    base = 1 << 40   # addresses only compared
    x, y, q, s, b = (base + (i << 36) for i in range(5))
    for wt in (Q8, Q4, F16):
        for K in (64, 128):
            for M in (1, 33, 172, 710, 2592):
                assert f(y, 1, x, wt, q, s, b, M, K, K) >= KS
                assert f(x + 2 * M * K, 1, x, wt, q, s, b, M, K, K) >= KS
                assert f(x - 2 * M * K, 1, x, wt, q, s, b, M, K, K) >= KS
                for o in (0, 16, -16, 2 * M * K - 16, 16 - 2 * M * K):
                    assert 0 <= f(x + o, 1, x, wt, q, s, b, M, K, K) < KS, (wt, K, M, o)


# (weight type, HEADS, M, K, N, the configuration that the pick starts from, those measured within 9 % of the
# fastest): a wide output of few products, more rows than 2592, HEADS at another width, and the DiT's
MEASURED = ((Q4, 0, 8192, 128, 16384, 4, (1, 3, 4, 7)), (Q8, 0, 5184, 128, 16384, 4, (3, 4, 7)),
            (Q4, 0, 12000, 256, 4096, 7, (0, 1, 3, 4, 7)), (Q8, 0, 2592, 128, 16384, 4, (0, 1, 3, 4)),
            (Q4, 0, 1836, 256, 4096, 7, (1, 7, 8)), (Q8, 0, 3500, 4096, 1024, 5, (1, 2, 6)),
            (Q8, 0, 5184, 1024, 256, 5, (0, 5)), (I8, 0, 8192, 1024, 8192, 3, (3,)), (I8, 0, 5184, 1024, 4096, 6, (3, 6)),
            (I8, 0, 8192, 1536, 6144, 3, (3,)), (I8, 0, 8192, 4096, 1024, 4, (1, 2)), (F16, 1, 1836, 2048, 2048, -1, (-1,)),
            (Q8, 0, 172, 4096, 1024, 5, (KS,)), (Q4, 0, 710, 4096, 1024, 5, (KS + 2,)), (Q8, 0, 2592, 1024, 4096, 7, (3, 7)),
            (F16, 1, 172, 1024, 3072, -1, (KS + 2, KS + 4)))


@pytest.mark.parametrize("wt,heads,M,K,N,cur,fast", MEASURED)
def test_pick_is_among_the_fastest_measured(wt, heads, M, K, N, cur, fast):
    import aria_amd
    try:
        pick = aria_amd.lib()._Z10qgemm_pickibiiii
    except (aria_amd.HipError, OSError) as e:
        pytest.skip(f"library not built: {e}")
    pick.restype, pick.argtypes = C.c_int, [C.c_int, C.c_bool] + [C.c_int] * 4
    assert pick(wt, bool(heads), M, N, K, cur) in fast
