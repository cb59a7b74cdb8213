"""The workloads this framework is timed on: what a program that generates audio with the SA3 DiT
and the small-music decoder has it do, called through the public entry points of ``aria_amd``.

Sizes are the DiT's and the decoder's own. small-music: model width 1024, 16 heads of 64, FFN
4096, 20 blocks, 256 latent channels, 64 memory tokens, 32 rotated dims; a latent frame lasts
4096 samples at 44.1 kHz, so 10 s are T = 108 frames (a sequence of 64 + 108 tokens) and 60 s are
T = 646; a guided request (CFG) runs two sequences. The benchmark's own shapes are two sequences
of 216 or 1296 tokens with 256 context tokens of width 768.

Inputs are torch tensors (or the host arrays that a host entry point takes) drawn from the seed;
work runs on the library's own streams. ``exact`` restates each path in float64 torch.
"""
import math
import types

import numpy as np
import torch

import aria_amd
from aria_amd import check, dec, dit
from aria_amd.device import DeviceArray

DIM, HEADS, INNER, DEPTH, IO, N_MEM, ROT = 1024, 16, 4096, 20, 256, 64, 32
PRECISION = {"q4": dit.Q4, "q8": dit.Q8, "f16": dit.F16, "auto": dit.AUTO}
WTYPE = {"q8": 0, "q4": 1, "f16": 2}
# the projections of a block, (K, N): sa_to_out / ca_to_q / ca_to_out, sa_to_qkv, the GELU and
# the GLU ff_in, ff_out
PROJECTIONS = ((1024, 1024), (1024, 3072), (1024, 4096), (1024, 8192), (4096, 1024))


def listed():
    return [
        # LayerNorm -> adaLN modulate -> GELU -> residual as one op, the benchmark's smallest shape:
        # one launch of a few microseconds
        {"name": "chain_216", "kind": "chain", "B": 2, "S": 216, "dim": 1024},
        # softmax over materialised scores, the benchmark's largest memory-bound op
        {"name": "softmax_1296", "kind": "softmax", "rows": 2 * 16 * 1296, "cols": 1296},
        # the dequantize-on-use GEMM with fp32 activations as aria_linear_q8 takes them, full size
        {"name": "linear_q8_2592", "kind": "linear", "wtype": "q8", "x": "f32", "y": "f32", "M": 2592, "K": 1024,
         "N": 4096, "bias": False},
        # the same on Q4 weights at the FFN's second projection, one 60 s sequence
        {"name": "linear_q4_710", "kind": "linear", "wtype": "q4", "x": "f16", "y": "f32", "M": 710, "K": 4096,
         "N": 1024, "bias": True},
        # W8A8 (quantise the rows, int8 GEMM) at the qkv projection of a guided 10 s request
        {"name": "linear_q8a8_344", "kind": "linear", "wtype": "q8a8", "x": "f32", "y": "f32", "M": 344, "K": 1024,
         "N": 3072, "bias": False},
        # self-attention of a guided 60 s request
        {"name": "attention_710", "kind": "attention", "B": 2, "Nq": 710, "Nk": 710, "out": "f16"},
        # one block as the benchmark runs it: q4, GELU FFN, two sequences of 1296 tokens
        {"name": "block_q4_1296", "kind": "block", "precision": "q4", "ffn": "gelu", "B": 2, "S": 1296, "Sc": 256,
         "ctx": 768},
        # one block of the model itself (GLU FFN, Q8 weights) on a guided 10 s request
        {"name": "block_q8_172", "kind": "block", "precision": "q8", "ffn": "glu", "B": 2, "S": 172, "Sc": 256,
         "ctx": 1024},
        # a whole denoise step of a 10 s request as the sampler's host loop calls it: latent and
        # conditioning from host memory, velocity back
        {"name": "step_q4_10s", "kind": "step", "precision": "q4", "B": 1, "T": 108, "Sc": 256, "io": "host"},
        # a whole denoise step of a guided 60 s request with the latent kept on the device, at the
        # precision the model picks by itself (W8A8)
        {"name": "step_auto_60s", "kind": "step", "precision": "auto", "B": 2, "T": 646, "Sc": 256, "io": "device"},
        # latent to stereo audio, 10 s and 60 s
        {"name": "decode_10s", "kind": "decode", "T": 108},
        {"name": "decode_60s", "kind": "decode", "T": 646},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("chain", "softmax", "linear", "linear", "attention", "block", "block", "step", "step", "decode"))
    if kind == "chain":
        return {"kind": kind, "B": rng.choice((1, 2)), "S": _log_int(rng, 24, 1296), "dim": rng.choice((512, 768, 1024, 2048))}
    if kind == "softmax":
        n = _log_int(rng, 40, 1296)
        return {"kind": kind, "rows": 16 * rng.choice((1, 2)) * n, "cols": n}
    if kind == "linear":
        wt = rng.choice(("q8", "q4", "f16", "q8a8"))
        K, N = rng.choice(PROJECTIONS)
        x = rng.choice(("f32", "f16"))
        # the W8A8 entry writes fp32
        y = "f32" if wt == "q8a8" else rng.choice(("f32", "f16"))
        return {"kind": kind, "wtype": wt, "x": x, "y": y, "M": _log_int(rng, 40, 2592), "K": K, "N": N,
                "bias": rng.random() < 0.5}
    if kind == "attention":
        nq = _log_int(rng, 72, 1296)
        return {"kind": kind, "B": rng.choice((1, 2)), "Nq": nq, "Nk": nq if rng.random() < 0.6 else rng.randint(16, 257),
                "out": rng.choice(("f16", "f32"))}
    if kind == "block":
        return {"kind": kind, "precision": rng.choice(("q4", "q8", "f16", "auto")), "ffn": rng.choice(("gelu", "glu")),
                "B": rng.choice((1, 2)), "S": _log_int(rng, 86, 1296), "Sc": rng.randint(16, 257), "ctx": rng.choice((768, 1024))}
    if kind == "step":
        return {"kind": kind, "precision": rng.choice(("q4", "q8", "f16", "auto")), "B": rng.choice((1, 2)),
                "T": _log_int(rng, 22, 646), "Sc": rng.randint(16, 257), "io": rng.choice(("host", "device"))}
    return {"kind": kind, "T": _log_int(rng, 5, 646)}


# ---- inputs ----

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, sigma=1.0, mean=0.0):
    return torch.randn(*shape, generator=g, device="cuda").mul_(sigma).add_(mean)


def _buf(t):
    """A tensor as the package's wrappers take device memory."""
    return types.SimpleNamespace(p=t.data_ptr(), t=t)


def _view(owner, ptr, shape):
    """A device buffer of the handle ``owner`` as a tensor over the same memory. The tensor keeps
    the handle, whose end frees that memory."""
    holder = types.SimpleNamespace(owner=owner, __cuda_array_interface__={
        "shape": tuple(shape), "typestr": "<f4", "data": (int(ptr), False), "version": 2, "strides": None})
    t = torch.as_tensor(holder, device="cuda")
    t.owner = owner
    return t


def _block_weights(g, dim, inner, ctx, glu):
    """One block's fp32 weights: projections N(0, 0.02), norm gains around 1."""
    def n(*shape):
        return _randn(g, *shape, sigma=0.02)
    w = {k: 1 + n(dim) for k in ("pre_norm", "cross_norm", "ff_norm")}
    w.update({k: 1 + n(64) for k in ("sa_q_norm", "sa_k_norm", "ca_q_norm", "ca_k_norm")})
    w.update(sa_to_qkv=n(3 * dim, dim), sa_to_out=n(dim, dim), ca_to_q=n(dim, dim), ca_to_kv=n(2 * dim, ctx),
             ca_to_out=n(dim, dim), ff_in_w=n((2 if glu else 1) * inner, dim), ff_in_b=n((2 if glu else 1) * inner),
             ff_out_w=n(dim, inner), ff_out_b=n(dim), to_scale_shift_gate=n(6 * dim))
    return w


def _rope_tables(S, rot):
    inv = 10000.0 ** (-torch.arange(0, rot, 2, dtype=torch.float64) / rot)
    a = torch.arange(S, dtype=torch.float64)[:, None] * inv[None, :]
    return a.cos().float(), a.sin().float()


def _block_inputs(case, seed):
    g = _gen(seed)
    B, S, Sc = case["B"], case["S"], case["Sc"]
    w = _block_weights(g, DIM, INNER, case["ctx"], case["ffn"] == "glu")
    x = _randn(g, B * S, DIM)
    ctx = _randn(g, B * Sc, case["ctx"])
    gcond = _randn(g, B, 6 * DIM, sigma=0.1)
    return w, x, ctx, gcond


DISTINCT = 4   # block weight sets of a 20-block model: block i holds set i % 4


def _step_inputs(case, seed):
    g = _gen(seed)
    B, T, Sc = case["B"], case["T"], case["Sc"]
    m = {"preprocess": _randn(g, IO, IO, sigma=0.02), "postprocess": _randn(g, IO, IO, sigma=0.02),
         "project_in": _randn(g, DIM, IO, sigma=0.06), "project_out": _randn(g, IO, DIM, sigma=0.03),
         "memory_tokens": _randn(g, N_MEM, DIM)}
    sets = [_block_weights(g, DIM, INNER, DIM, True) for _ in range(DISTINCT)]
    x = _randn(g, B, IO, T)
    ced = _randn(g, B, Sc, DIM)
    gcond = _randn(g, B, 6 * DIM, sigma=0.1)
    return m, sets, x, ced, gcond


D_DIM, D_INNER, D_QKV, D_CHUNK, D_HEADS = 768, 2304, 3840, 34, 12


def _decoder_inputs(case, seed):
    """A checkpoint's tensors under the reference's names, activations O(1) throughout, and a latent."""
    g = _gen(seed)
    pfx = "pretransform.model."
    t = {pfx + "bottleneck.running_std": torch.full((1,), 0.9, device="cuda"),
         pfx + "decoder.layers.1.weight": _randn(g, D_DIM, 256, sigma=1 / 16.0),
         pfx + "decoder.layers.1.bias": _randn(g, D_DIM, sigma=0.05),
         pfx + "decoder.layers.3.new_tokens": _randn(g, D_DIM, sigma=0.5),
         pfx + "decoder.layers.3.mapping.weight_g": torch.rand(512, 1, 1, generator=g, device="cuda") + 0.5,
         pfx + "decoder.layers.3.mapping.weight_v": _randn(g, 512, D_DIM, 3),
         pfx + "decoder.layers.3.mapping.bias": _randn(g, 512, sigma=0.05)}
    for i in range(6):
        p = pfx + "decoder.layers.3.transformers.%d." % i
        for n, width, gain in (("pre_norm", D_DIM, 1.0), ("ff_norm", D_DIM, 1.0), ("self_attn.q_norm", 64, 2.0),
                               ("self_attn.k_norm", 64, 2.0)):
            t[p + n + ".alpha"] = torch.rand(1, generator=g, device="cuda") + 0.5
            t[p + n + ".gamma"] = _randn(g, width, sigma=0.1 * gain, mean=gain)
            t[p + n + ".beta"] = _randn(g, width, sigma=0.05)
        t[p + "self_attn.to_qkv.weight"] = _randn(g, D_QKV, D_DIM, sigma=D_DIM ** -0.5)
        t[p + "self_attn.to_out.weight"] = _randn(g, D_DIM, D_DIM, sigma=0.5 * D_DIM ** -0.5)
        t[p + "ff.ff.0.proj.weight"] = _randn(g, 2 * D_INNER, D_DIM, sigma=D_DIM ** -0.5)
        t[p + "ff.ff.0.proj.bias"] = _randn(g, 2 * D_INNER, sigma=0.05)
        t[p + "ff.ff.2.weight"] = _randn(g, D_DIM, D_INNER, sigma=0.5 * D_INNER ** -0.5)
        t[p + "ff.ff.2.bias"] = _randn(g, D_DIM, sigma=0.05)
    return t, _randn(g, 256, case["T"])


def _linear_inputs(case, seed):
    g = _gen(seed)
    x = _randn(g, case["M"], case["K"])
    w = _randn(g, case["N"], case["K"], sigma=0.02)
    b = _randn(g, case["N"], sigma=0.02) if case["bias"] else None
    return (x.half() if case["x"] == "f16" else x), w, b


def _chain_inputs(case, seed):
    g = _gen(seed)
    B, S, dim = case["B"], case["S"], case["dim"]
    return (_randn(g, B, S, dim), _randn(g, dim, sigma=0.1, mean=1.0), _randn(g, dim, sigma=0.1),
            _randn(g, B, dim, sigma=0.1), _randn(g, B, dim, sigma=0.1))


def _attention_inputs(case, seed):
    """q and k as the head preparation leaves them: RMS-normalised rows with gains around 1."""
    g = _gen(seed)
    BH = case["B"] * HEADS
    q = torch.nn.functional.normalize(_randn(g, BH, case["Nq"], 64), dim=-1).mul_(8.0)
    k = torch.nn.functional.normalize(_randn(g, BH, case["Nk"], 64), dim=-1).mul_(8.0)
    return q.half(), k.half(), _randn(g, BH, case["Nk"], 64).half()


def _host(d):
    return {k: v.cpu().numpy() for k, v in d.items()}


# ---- the program: prepare once, run many times ----

def prepare(case, seed):
    L = aria_amd.lib()
    check(L.aria_hip_init(), "aria_hip_init")
    kind = case["kind"]
    s = types.SimpleNamespace(kind=kind, case=case, L=L)
    if kind == "chain":
        s.x, s.g, s.b, s.sc, s.sh = _chain_inputs(case, seed)
        s.y = torch.empty_like(s.x)
    elif kind == "softmax":
        s.x = _randn(_gen(seed), case["rows"], case["cols"], sigma=2.0)
    elif kind == "linear":
        s.x, w, s.bias = _linear_inputs(case, seed)
        M, K, N = case["M"], case["K"], case["N"]
        s.y = torch.empty(M, N, device="cuda", dtype=torch.float16 if case["y"] == "f16" else torch.float32)
        s.scale = None
        torch.cuda.synchronize()
        if case["wtype"] == "f16":
            s.q = w.half()
        elif case["wtype"] == "q4":
            s.q = torch.empty(N, K // 2, device="cuda", dtype=torch.uint8)
            s.scale = torch.empty(N, K // 32, 2, device="cuda")
            check(L.aria_hip_q4_quant_dev(s.q.data_ptr(), s.scale.data_ptr(), w.data_ptr(), N, K, None), "pack")
        else:
            s.q = torch.empty(N, K, device="cuda", dtype=torch.int8)
            s.scale = torch.empty(N, device="cuda")
            check(L.aria_hip_q8_quant_dev(s.q.data_ptr(), s.scale.data_ptr(), w.data_ptr(), N, K, None), "pack")
        check(L.aria_hip_stream_sync(None), "pack")
        if case["wtype"] == "q8a8":
            s.ws = torch.empty(int(L.aria_hip_q8a8_ws_bytes(M, K)), device="cuda", dtype=torch.uint8)
    elif kind == "attention":
        s.q, s.k, s.v = _attention_inputs(case, seed)
        s.y = torch.empty(case["B"], case["Nq"], HEADS * 64, device="cuda",
                          dtype=torch.float16 if case["out"] == "f16" else torch.float32)
    elif kind == "block":
        w, x, ctx, gcond = _block_inputs(case, seed)
        B, S, Sc = case["B"], case["S"], case["Sc"]
        precision = dit.Q8A8 if case["precision"] == "auto" else PRECISION[case["precision"]]
        s.block = dit.DitBlock(_host(w), DIM, HEADS, INNER, case["ctx"], dit.FFN_GLU if case["ffn"] == "glu" else dit.FFN_GELU,
                               precision)
        s.x, s.g = _buf(x), _buf(gcond)
        s.cos, s.sin = (_buf(t.cuda()) for t in _rope_tables(S, ROT))
        torch.cuda.synchronize()
        s.k, s.v = s.block.cross_kv(_buf(ctx), B, Sc)
        check(L.aria_hip_stream_sync(None), "cross_kv")
        s.ws = s.block.workspace(B, S, Sc)
    elif kind == "step":
        m, sets, x, ced, gcond = _step_inputs(case, seed)
        sets = [_host(w) for w in sets]
        model = dict(_host(m), blocks=[sets[i % DISTINCT] for i in range(DEPTH)])
        s.dit = dit.Dit(model, DEPTH, DIM, HEADS, INNER, IO, N_MEM, ROT, precision=PRECISION[case["precision"]])
        cos, sin = _rope_tables(N_MEM + case["T"], ROT)
        s.dit.set_request(case["T"], list(ced.cpu().numpy()), cos.numpy(), sin.numpy())
        s.x, s.g = x.cpu().numpy(), gcond.cpu().numpy()
        if case["io"] == "device":
            dx, dv, dg = s.dit.device_buffers()
            L.aria_cuda_memcpy_h2d(dx, s.x.ctypes.data, s.x.nbytes)
            L.aria_cuda_memcpy_h2d(dg, s.g.ctypes.data, s.g.nbytes)
            s.out = _view(s.dit, dv, s.x.shape)
    else:
        t, s.latent = _decoder_inputs(case, seed)
        s.dec = dec.Decoder.from_tensors(_host(t))
        s.audio = torch.empty(2, case["T"] * 4096, device="cuda")
    torch.cuda.synchronize()
    return s


def run(s):
    c, L = s.case, s.L
    if s.kind == "chain":
        check(L.aria_hip_ln_mod_gelu_res_dev(s.y.data_ptr(), s.x.data_ptr(), s.g.data_ptr(), s.b.data_ptr(), s.sc.data_ptr(),
                                             s.sh.data_ptr(), c["B"] * c["S"], c["dim"], c["S"], 1e-6, None), "chain")
        return s.y
    if s.kind == "softmax":   # in place: a second pass takes the softmax of the first one's rows
        check(L.aria_hip_softmax_dev(s.x.data_ptr(), c["rows"], c["cols"], None, None), "softmax")
        return s.x
    if s.kind == "linear":
        b = s.bias.data_ptr() if s.bias is not None else None
        if c["wtype"] == "q8a8":
            check(L.aria_hip_linear_q8a8_dev(s.y.data_ptr(), s.x.data_ptr(), int(c["x"] == "f16"), s.q.data_ptr(),
                                             s.scale.data_ptr(), b, c["M"], c["K"], c["N"], s.ws.data_ptr(), None), "linear")
        else:
            check(L.aria_hip_qlinear_dev(s.y.data_ptr(), int(c["y"] == "f16"), s.x.data_ptr(), int(c["x"] == "f16"),
                                         WTYPE[c["wtype"]], s.q.data_ptr(), s.scale.data_ptr() if s.scale is not None else None,
                                         b, c["M"], c["K"], c["N"], None), "linear")
        return s.y
    if s.kind == "attention":
        check(L.aria_hip_flash_attention_dev(s.q.data_ptr(), s.k.data_ptr(), s.v.data_ptr(), s.y.data_ptr(),
                                             int(c["out"] == "f16"), c["B"], HEADS, c["Nq"], c["Nk"], 64, None), "attention")
        return s.y
    if s.kind == "block":   # in place on the residual stream
        s.block.forward(s.x, c["B"], c["S"], s.g, s.k, s.v, c["Sc"], s.cos, s.sin, ROT, ws=s.ws)
        return s.x.t
    if s.kind == "step":
        if c["io"] == "host":
            return s.dit.step(s.x, s.g)
        s.dit.run()
        return s.out
    s.dec.forward_dev(s.audio.data_ptr(), s.latent.data_ptr(), c["T"])
    return s.audio


# ---- what a pass cannot do without ----

def _weight_bytes(wtype, K, N):
    return {"q8": N * K + 4 * N, "q8a8": N * K + 4 * N, "q4": N * K // 2 + N * K // 4, "f16": 2 * N * K}[wtype]


def _block_work(precision, glu, B, S, Sc):
    at = "f16" if precision == "f16" else "q8"
    ff = "q4" if precision == "q4" else at
    M, n_in = B * S, (2 if glu else 1) * INNER
    projections = [(at, DIM, 3 * DIM)] + [(at, DIM, DIM)] * 3 + [(ff, DIM, n_in), (ff, INNER, DIM)]
    weights = sum(_weight_bytes(t, K, N) for t, K, N in projections)
    flops = sum(2 * M * K * N for _, K, N in projections) + 4 * M * (S + Sc) * DIM
    return weights, flops, 2 * 2 * B * Sc * DIM   # ... and the context's K and V, fp16


def work(case):
    kind = case["kind"]
    if kind == "chain":
        n = case["B"] * case["S"] * case["dim"]
        return {"bytes": 8 * n + 8 * case["dim"] * (1 + case["B"]), "flops": 0}
    if kind == "softmax":
        return {"bytes": 8 * case["rows"] * case["cols"], "flops": 0}
    if kind == "linear":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": M * K * (2 if case["x"] == "f16" else 4) + _weight_bytes(case["wtype"], K, N) +
                M * N * (2 if case["y"] == "f16" else 4), "flops": 2 * M * K * N}
    if kind == "attention":
        BH, nq, nk = case["B"] * HEADS, case["Nq"], case["Nk"]
        return {"bytes": BH * 64 * (2 * nq + 4 * nk + (2 if case["out"] == "f16" else 4) * nq), "flops": 4 * BH * nq * nk * 64}
    if kind == "block":
        weights, flops, kv = _block_work(case["precision"], case["ffn"] == "glu", case["B"], case["S"], case["Sc"])
        return {"bytes": weights + kv + 8 * case["B"] * case["S"] * DIM, "flops": flops}
    if kind == "step":
        B, T, S = case["B"], case["T"], N_MEM + case["T"]
        weights, flops, kv = _block_work(case["precision"], True, B, S, case["Sc"])
        return {"bytes": DEPTH * (weights + kv) + 8 * B * IO * T + 4 * IO * (IO + DIM),
                "flops": DEPTH * flops + 4 * B * T * IO * (IO + DIM)}
    T = case["T"]
    L = 17 * (T + T % 2)
    per_row = 2 * D_DIM * (D_QKV + D_DIM + 3 * D_INNER) + 8 * D_CHUNK * D_DIM
    return {"bytes": 6 * 2 * D_DIM * (D_QKV + D_DIM + 3 * D_INNER) + 4 * 512 * 3 * D_DIM + 4 * 256 * T + 4 * 8192 * T,
            "flops": 3 * (2 * L + D_CHUNK) * per_row + 2 * 16 * T * 512 * 3 * D_DIM + 2 * T * 256 * D_DIM}


def tolerance(case):
    """About four times the distance from ``exact`` that was measured over these ranges."""
    kind = case["kind"]
    if kind in ("chain", "softmax"):
        return {"rel": 4e-7, "max": 4e-5}     # fp32 throughout
    if kind == "linear":
        if case["y"] == "f16":
            return {"rel": 1.5e-3}
        if case["wtype"] == "q8a8":
            return {"rel": 4e-7}              # exact integer sums, a few fp32 roundings
        # fp32 sums of fp16 products; fp32 activations and Q4 weights are rounded to fp16 first
        return {"rel": 1.2e-3} if case["x"] == "f32" or case["wtype"] == "q4" else {"rel": 2e-6}
    if kind == "attention":
        return {"rel": 1.2e-3}                # fp16 probabilities
    if kind == "block":
        # W8A8: a rounding difference can move an activation by a whole int8 step
        return {"rel": 1.2e-2} if case["precision"] == "auto" else {"rel": 5e-4}
    if kind == "step":
        return {"rel": 3e-2} if case["precision"] == "auto" else {"rel": 3e-3}   # the same over 20 blocks
    return {"rel": 6e-4}


# ---- the same in float64 ----

def _div(a, b):
    """a / b rounded once: torch multiplies by the reciprocal where one side is a Python number."""
    like = a if torch.is_tensor(a) else b
    a, b = (t if torch.is_tensor(t) else torch.full_like(like, t) for t in (a, b))
    return a / b


def _q8(w):
    """Per-row symmetric int8 as a value: the packed format's own fp32 rule, then 64 bits."""
    s = _div(w.abs().amax(-1, keepdim=True), 127.0)
    return torch.clamp(torch.round(w * _div(1.0, s)), -127, 127).double() * s.double()


def _q4(w):
    b = w.reshape(w.shape[0], -1, 32)
    mn = b.amin(-1, keepdim=True)
    s = _div(b.amax(-1, keepdim=True) - mn, 15.0)
    return (torch.clamp(torch.round((b - mn) * _div(1.0, s)), 0, 15).double() * s.double() + mn.double()).reshape(w.shape)


def _rows_q8(x):
    a = x.abs().amax(-1, keepdim=True)
    return torch.clamp(torch.round(x * _div(127.0, a)), -127, 127).double() * _div(a, 127.0).double()


def _weight(wtype, w):
    return {"q8": _q8, "q8a8": _q8, "q4": _q4, "f16": lambda v: v.half().double()}[wtype](w)


def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _silu(x):
    return x * torch.sigmoid(x)


def _rope(x, cos, sin):
    """Rotate-half on the first 2 * cos.shape[1] dims of x [..., S, 64]."""
    h = cos.shape[1]
    a, b = x[..., :h], x[..., h:2 * h]
    return torch.cat((a * cos - b * sin, b * cos + a * sin, x[..., 2 * h:]), -1)


def _attend(q, k, v):
    p = torch.softmax(torch.matmul(q, k.transpose(-1, -2).contiguous()) * 0.125, -1)
    return torch.matmul(p, v)


def _exact_block(w, wt, glu, x, k, v, gcond, cos, sin, quantised):
    """One sequence [S, dim] through the block; ``wt`` its projections in 64 bits."""
    def lin(name, h, b=None):
        y = (_rows_q8(h) if quantised else h) @ wt[name].T
        return y if b is None else y + b.double()

    def split(t):
        return t.reshape(t.shape[0], -1, 64).transpose(0, 1).contiguous()

    mod = (w["to_scale_shift_gate"].double() + gcond.double()).reshape(6, -1)
    h = _rms(x, w["pre_norm"], 1e-5) * (1 + mod[0]) + mod[1]
    q, kk, vv = (split(t) for t in lin("sa_to_qkv", h).chunk(3, -1))
    q, kk = _rope(_rms(q, w["sa_q_norm"], 1e-6), cos, sin), _rope(_rms(kk, w["sa_k_norm"], 1e-6), cos, sin)
    o = _attend(q, kk, vv).transpose(0, 1).reshape(x.shape)
    x = x + lin("sa_to_out", o) * torch.sigmoid(1 - mod[2])
    q = _rms(split(lin("ca_to_q", _rms(x, w["cross_norm"], 1e-5))), w["ca_q_norm"], 1e-6)
    x = x + lin("ca_to_out", _attend(q, k, v).transpose(0, 1).reshape(x.shape))
    h = lin("ff_in_w", _rms(x, w["ff_norm"], 1e-5) * (1 + mod[3]) + mod[4], w["ff_in_b"])
    if glu:
        val, gate = h.chunk(2, -1)
        h = _silu(gate) * val
    else:
        h = _gelu(h)
    return x + lin("ff_out_w", h, w["ff_out_b"]) * torch.sigmoid(1 - mod[5])


def _exact_weights(w, precision):
    at = "f16" if precision == "f16" else "q8"
    ff = "q4" if precision == "q4" else at
    return {n: _weight(ff if n.startswith("ff") else at, w[n]) for n in
            ("sa_to_qkv", "sa_to_out", "ca_to_q", "ca_to_out", "ff_in_w", "ff_out_w")}


def _exact_cross(w, ctx):
    kv = ctx.double() @ w["ca_to_kv"].half().double().T
    k, v = (t.reshape(t.shape[0], -1, 64).transpose(0, 1).contiguous() for t in kv.chunk(2, -1))
    return _rms(k, w["ca_k_norm"], 1e-6), v


def _exact_decode(case, seed):
    t, latent = _decoder_inputs(case, seed)
    pfx = "pretransform.model."
    T = case["T"]
    Tp = T + T % 2
    L = 17 * Tp
    cos, sin = (c.double().cuda() for c in _rope_tables(D_CHUNK, 32))

    def half(name):
        return t[name].half().double()

    def dyt(x, name):
        return torch.tanh(t[name + ".alpha"].double() * x) * t[name + ".gamma"].double() + t[name + ".beta"].double()

    def block(x, i):
        p = pfx + "decoder.layers.3.transformers.%d." % i
        n = x.shape[0] // D_CHUNK
        qkv = dyt(x, p + "pre_norm") @ half(p + "self_attn.to_qkv.weight").T
        q, k, v, qd, kd = (a.contiguous() for a in qkv.reshape(n, D_CHUNK, 5, D_HEADS, 64).permute(2, 0, 3, 1, 4))
        q, qd = (_rope(dyt(a, p + "self_attn.q_norm"), cos, sin) for a in (q, qd))
        k, kd = (_rope(dyt(a, p + "self_attn.k_norm"), cos, sin) for a in (k, kd))
        m = (_attend(q, k, v) - _attend(qd, kd, v)).transpose(1, 2).reshape(x.shape)
        x = x + m @ half(p + "self_attn.to_out.weight").T
        h = dyt(x, p + "ff_norm") @ half(p + "ff.ff.0.proj.weight").T + t[p + "ff.ff.0.proj.bias"].double()
        val, gate = h.chunk(2, -1)
        return x + (val * _silu(gate)) @ half(p + "ff.ff.2.weight").T + t[p + "ff.ff.2.bias"].double()

    x = (latent.double() * t[pfx + "bottleneck.running_std"].double()).T @ half(pfx + "decoder.layers.1.weight").T
    x = x + t[pfx + "decoder.layers.1.bias"].double()
    seq = t[pfx + "decoder.layers.3.new_tokens"].double().repeat(L, 1)
    seq[0::17] = 0
    seq[0:17 * T:17] = x
    for i in range(3):
        seq = block(seq, i)
    seq = torch.cat((seq[:17], seq, seq[-17:]))
    for i in range(3, 6):
        seq = block(seq, i)
    seq = seq[17:17 + L].reshape(Tp, 17, D_DIM)[:, 1:].reshape(16 * Tp, D_DIM)
    zero = torch.zeros(1, D_DIM, device="cuda", dtype=torch.float64)
    seq = torch.cat((zero, seq, zero))
    v = t[pfx + "decoder.layers.3.mapping.weight_v"].reshape(512, -1)
    gain = (t[pfx + "decoder.layers.3.mapping.weight_g"].reshape(512, 1).double() / v.double().square().sum(1, keepdim=True).sqrt())
    w = (v * gain.float()).double().reshape(512, D_DIM, 3)
    y = sum(seq[j:j + 16 * Tp] @ w[:, :, j].contiguous().T for j in range(3)) + t[pfx + "decoder.layers.3.mapping.bias"].double()
    return y[:16 * T].reshape(16 * T, 2, 256).transpose(0, 1).reshape(2, 4096 * T)


def exact(case, seed):
    kind = case["kind"]
    if kind == "chain":
        x, g, b, sc, sh = (a.double() for a in _chain_inputs(case, seed))
        y = (x - x.mean(-1, keepdim=True)) * torch.rsqrt(x.var(-1, unbiased=False, keepdim=True) + 1e-6) * g + b
        return _gelu(y * (1 + sc[:, None]) + sh[:, None]) + x
    if kind == "softmax":
        return torch.softmax(_randn(_gen(seed), case["rows"], case["cols"], sigma=2.0).double(), -1)
    if kind == "linear":
        x, w, b = _linear_inputs(case, seed)
        x = _rows_q8(x.float()) if case["wtype"] == "q8a8" else x.double()
        y = x @ _weight(case["wtype"], w).T
        return y if b is None else y + b.double()
    if kind == "attention":
        q, k, v = (t.double() for t in _attention_inputs(case, seed))
        o = _attend(q, k, v).reshape(case["B"], HEADS, case["Nq"], 64)
        return o.transpose(1, 2).reshape(case["B"], case["Nq"], HEADS * 64)
    if kind == "block":
        w, x, ctx, gcond = _block_inputs(case, seed)
        wt = _exact_weights(w, case["precision"])
        cos, sin = (c.double().cuda() for c in _rope_tables(case["S"], ROT))
        B, S, Sc = case["B"], case["S"], case["Sc"]
        return torch.cat([_exact_block(w, wt, case["ffn"] == "glu", x[b * S:(b + 1) * S].double(),
                                       *_exact_cross(w, ctx[b * Sc:(b + 1) * Sc]), gcond[b], cos, sin,
                                       case["precision"] == "auto") for b in range(B)])
    if kind == "step":
        m, sets, x, ced, gcond = _step_inputs(case, seed)
        m = {k: v if k == "memory_tokens" else v.half() for k, v in m.items()}
        m = {k: v.double() for k, v in m.items()}
        wts = [_exact_weights(w, case["precision"]) for w in sets]
        cos, sin = (c.double().cuda() for c in _rope_tables(N_MEM + case["T"], ROT))
        out = []
        for b in range(case["B"]):
            h = x[b].double().T.contiguous()
            h = h + h @ m["preprocess"].T
            h = torch.cat((m["memory_tokens"], h @ m["project_in"].T))
            cross = [_exact_cross(w, ced[b]) for w in sets]
            for i in range(DEPTH):
                j = i % DISTINCT
                h = _exact_block(sets[j], wts[j], True, h, *cross[j], gcond[b], cos, sin, case["precision"] == "auto")
            h = h[N_MEM:] @ m["project_out"].T
            out.append((h + h @ m["postprocess"].T).T)
        return torch.stack(out).contiguous()
    return _exact_decode(case, seed)
