"""The denoise step around its blocks (aria_hip_dit.c step_compute): the residual pre and post
convolutions, the io projections and the memory tokens, at channel counts that take the fused
residual (multiples of 32) and one that does not, with and without memory tokens, one and two
sequences, odd lengths.

Oracle: the same step with every projection outside the blocks in float64 on the fp16-rounded
weights, and the blocks through aria_hip_dit_block_forward_dev. Gate: the full-DiT one of
test_gpu_dit.py (the io GEMMs round their activations to fp16, 2^-11 of a value; a row or a sequence
in the wrong place is off by O(1)).
"""
from __future__ import annotations

import numpy as np
import pytest

from conftest import assert_close, randn, rng
from test_gpu_dit import ATOL, RTOL, inputs, make_dit

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("io_ch,n_mem,B,T", [(64, 3, 1, 21), (64, 3, 2, 37), (256, 64, 1, 33), (256, 64, 2, 45),
                                             (32, 5, 2, 1), (96, 0, 2, 19), (16, 3, 2, 21)])
def test_step_io(hip, port, io_ch, n_mem, B, T):
    from aria_amd.device import DeviceArray
    from aria_amd.dit import DitBlock, random_dit
    ed, H, rot, n_cond, inner = 128, 2, 32, 9, 256
    M = random_dit(rng(io_ch + n_mem + T), 2, ed, inner, io_ch, n_mem)
    r = rng(T)
    for k in ("preprocess", "postprocess"):   # a residual that would be missed
        M[k] = randn(r, (io_ch, io_ch), 0.5 * io_ch ** -0.5)
    w = {k: M[k].astype(np.float16).astype(np.float64) for k in ("preprocess", "postprocess", "project_in", "project_out")}
    S = n_mem + T
    c, s = port.rope_freqs(S, rot, 10000.0)
    dit = make_dit(M, 4, H, rot)
    _, ced, _ = inputs(2, B, io_ch, T, n_cond, ed)
    dit.set_request(T, list(ced), c, s)
    dctx, dc, dsn = DeviceArray.from_host(ced.reshape(B * n_cond, ed)), DeviceArray.from_host(c), DeviceArray.from_host(s)
    blocks = [DitBlock(b, ed, H, inner, ed, precision=4) for b in M["blocks"]]
    for k in range(3):   # the step again with other inputs: the io buffers are used over, the last ones by a replay
        x, _, g = inputs(500 + k, B, io_ch, T, n_cond, ed)
        h = x.astype(np.float64).transpose(0, 2, 1)
        h = (h + h @ w["preprocess"].T) @ w["project_in"].T
        seq = np.concatenate([np.broadcast_to(M["memory_tokens"].astype(np.float64), (B, n_mem, ed)), h], 1)
        dx, dg = DeviceArray.from_host(seq.reshape(B * S, ed).astype(np.float32)), DeviceArray.from_host(g)
        for b in blocks:
            dk, dv = b.cross_kv(dctx, B, n_cond)
            b.forward(dx, B, S, dg, dk, dv, n_cond, dc, dsn, rot)
        hip.check(hip.lib().aria_hip_stream_sync(None))
        o = dx.to_host().reshape(B, S, ed)[:, n_mem:].astype(np.float64) @ w["project_out"].T
        want = (o + o @ w["postprocess"].T).transpose(0, 2, 1)
        got = dit.step(x, g)
        assert_close(got, want, ATOL, RTOL, f"step {k}")
        gate = ATOL + RTOL * np.abs(want).max()
        assert np.abs(o.transpose(0, 2, 1) - want).max() > 10 * gate   # a lost residual shows
    for b in blocks:
        b.free()
    dit.free()
