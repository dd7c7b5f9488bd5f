"""Workloads of the quantized linear that its users run, with inputs, plain 64-bit results and costs.

A case is one of four ways a program calls the library:

  layer   the four projections of Qwen3-4B decoder layers on device rows, as an engine that keeps its
          activations on the GPU calls them: qkv = RMSNorm -> linear, h1 = x + o(attention), middle =
          SiLU-gate(gate_up(RMSNorm(h1))), h2 = h1 + down(middle).  Attention itself is the engine's,
          so every layer gets its own hidden and attention rows.
  linear  one K x N linear over several weight sets (the same projection of several layers).
  chain   decoder layers' projections in one launch (qlin_chain_run), 1..4 rows.
  host    the synchronous host-buffer calls (qlin_run_f32 / qlin_run_swiglu_f32), float32 rows in and out.

The calls go through the C ABI with their arguments bound once, as a native engine makes them.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from open_rknpu2_lm_infer_amd import _lib, synth
from open_rknpu2_lm_infer_amd import qlinear as ql

EPS = 1e-6
FLT_MIN = 1.17549435e-38
_TORCH = {"f16": torch.float16, "f32": torch.float32}
_QLIN = {"f16": _lib.QLIN_F16, "f32": _lib.QLIN_F32}
_BYTES = {"f16": 2, "f32": 4}


def listed():
    return [
        # the smallest calls: one token through the W8 2560 x 2560 projection of sixteen layers (round half to even)
        {"name": "w8_2560_m1", "kind": "linear", "rows": 1, "K": 2560, "N": 2560, "bits": 8, "copies": 16, "act": "f16",
         "out": "f16", "swiglu": False, "norm": False, "residual": False, "half_even": True},
        # decoding one token: W4 decoder layers
        {"name": "layer_w4_m1", "kind": "layer", "rows": 1, "layers": 4, "qg": 4, "od": 4, "act": "f16", "dist": "normal"},
        # a speculative verify step: one token and three drafted ones, o and down in 8 bits
        {"name": "layer_mixed_m4", "kind": "layer", "rows": 4, "layers": 4, "qg": 4, "od": 8, "act": "f16", "dist": "normal"},
        # decoding one token with the layers' projections in one launch
        {"name": "chain_mixed_m1", "kind": "chain", "rows": 1, "layers": 4, "qg": 4, "od": 8},
        # the vocabulary head of one token, float32 logits
        {"name": "lm_head_w8_m1", "kind": "linear", "rows": 1, "K": 2560, "N": 151936, "bits": 8, "copies": 1, "act": "f16",
         "out": "f32", "swiglu": False, "norm": True, "residual": False, "half_even": False},
        # batched decoding: 24 sequences a step
        {"name": "layer_w4_m24", "kind": "layer", "rows": 24, "layers": 4, "qg": 4, "od": 4, "act": "f16", "dist": "normal"},
        # prefill by the reference's default chunk of 128 tokens
        {"name": "layer_w4_m128", "kind": "layer", "rows": 128, "layers": 4, "qg": 4, "od": 4, "act": "f16", "dist": "normal"},
        # a ragged prompt of 300 tokens, float32 rows as the reference keeps them, o and down in 8 bits
        {"name": "layer_mixed_m300", "kind": "layer", "rows": 300, "layers": 4, "qg": 4, "od": 8, "act": "f32",
         "dist": "normal"},
        # prefill of 512 tokens
        {"name": "layer_w4_m512", "kind": "layer", "rows": 512, "layers": 4, "qg": 4, "od": 4, "act": "f16", "dist": "normal"},
        # a long prompt with heavy-tailed activations
        {"name": "layer_w4_m4096", "kind": "layer", "rows": 4096, "layers": 1, "qg": 4, "od": 4, "act": "f16",
         "dist": "student_t3"},
        # the drop-in calls of an engine whose activations live on the host: one token, and a prefill chunk
        {"name": "host_w4_m1", "kind": "host", "rows": 1, "layers": 2, "qg": 4, "od": 4},
        {"name": "host_w4_m128", "kind": "host", "rows": 128, "layers": 2, "qg": 4, "od": 4},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "layer", "layer", "chain", "host"])
    bits = lambda: rng.choice([4, 4, 8])  # noqa: E731
    if kind == "layer":
        rows = _log_int(rng, 1, 2048)
        return {"kind": kind, "rows": rows, "layers": 4 if rows <= 700 else 1, "qg": bits(), "od": bits(),
                "act": rng.choice(["f16", "f16", "f32"]), "dist": rng.choice(["normal", "student_t3"])}
    if kind == "chain":
        return {"kind": kind, "rows": rng.randint(1, 4), "layers": rng.randint(2, 8), "qg": 4, "od": rng.choice([4, 8])}
    if kind == "host":
        return {"kind": kind, "rows": _log_int(rng, 1, 256), "layers": rng.randint(1, 3), "qg": bits(), "od": bits()}
    b = bits()
    K, N, rows = _log_int(rng, 384, 9728), _log_int(rng, 256, 19456), _log_int(rng, 1, 4096)
    if rng.random() < 0.6:  # most projections are whole multiples of 128
        K, N = (K + 127) // 128 * 128, (N + 127) // 128 * 128
    elif b == 4:
        K += K & 1
    form = rng.choice(["plain", "plain", "norm", "residual", "swiglu", "norm_swiglu"])
    if "swiglu" in form:
        N += N & 1
    copies = max(1, min(8, int(200e6 / (K * N * b / 8)), int(4e11 / (2.0 * rows * K * N))))
    return {"kind": "linear", "rows": rows, "K": K, "N": N, "bits": b, "copies": copies, "act": rng.choice(["f16", "f16", "f32"]),
            "out": rng.choice(["f16", "f16", "f32"]), "swiglu": "swiglu" in form, "norm": "norm" in form,
            "residual": form == "residual", "half_even": rng.random() < 0.25}


# ---- inputs, from the seed alone ---------------------------------------------------------


def _linears(case):
    """(K, N, bits, swiglu) of one case's weights, in the order they are made."""
    if case["kind"] == "linear":
        return [(case["K"], case["N"], case["bits"], case["swiglu"])] * case["copies"]
    per = [(K, N, case["qg"] if name in ("qkv", "gate_up") else case["od"], name == "gate_up")
           for name, K, N in synth.LAYER]
    return per * case["layers"]


def _codes(case, seed, i):
    """int8 [N, K] codes and float32 [N] scales of weight i: variance preserving, so that rows keep their size."""
    K, N, bits, _ = _linears(case)[i]
    codes = synth.codes(N, K, bits, seed * 1000 + 2 * i, "cuda")
    g = synth.gen(seed * 1000 + 2 * i + 1, "cuda")
    std = 73.3 if bits == 8 else 4.61
    u = torch.rand((N,), generator=g, device="cuda") + 0.5
    return codes, (u / (std * math.sqrt(K))).contiguous()


def _rows(case, seed, i, K, act):
    x = synth.activations(case["rows"], K, seed * 1000 + 500 + i, "cuda", case.get("dist", "normal"))
    return x.to(_TORCH[act])


def _gamma(seed, i, K):
    return synth.gamma(K, seed * 1000 + 800 + i, "cuda")


# ---- the program's side -------------------------------------------------------------------


def _weights(case, seed):
    made = []
    for i, (K, N, bits, _) in enumerate(_linears(case)):
        codes, scales = _codes(case, seed, i)
        if bits == 4 and K % 2:
            raise ValueError("W4 codes come in pairs")
        packed = synth.pack_w4(codes) if bits == 4 else codes
        made.append(ql.Weights.from_packed_device(bits, K, N, packed, scales))
    return made


class _Call:
    """One C ABI call with its arguments bound."""

    def __init__(self, name, *args):
        self.fn, self.args, self.name = getattr(_lib.load(), name), args, name

    def __call__(self):
        rc = self.fn(*self.args)
        if rc:
            _lib.check(rc, self.name)


def _bind(ws, w, x, out, flags, stream, gamma=None, residual=None):
    head = (ws.handle, w.handle, x.shape[0], x.data_ptr(), ql._DT[x.dtype], x.stride(0))
    tail = (out.data_ptr(), ql._DT[out.dtype], out.stride(0), flags, stream)
    if gamma is not None:
        return _Call("qlin_run_rmsnorm", *head, gamma.data_ptr(), EPS, *tail)
    if residual is not None:
        return _Call("qlin_run_residual", *head, residual.data_ptr(), ql._DT[residual.dtype], residual.stride(0), 1.0, *tail)
    return _Call("qlin_run", *head, *tail)


def prepare(case, seed):
    kind, M = case["kind"], case["rows"]
    weights = _weights(case, seed)
    shapes = _linears(case)
    stream = torch.cuda.current_stream().cuda_stream
    state = {"weights": weights, "calls": [], "out": [], "keep": []}
    if kind == "chain":
        stages, keep = [], []
        for l in range(case["layers"]):
            g1, g2 = _gamma(seed, 2 * l, synth.HIDDEN), _gamma(seed, 2 * l + 1, synth.HIDDEN)
            keep += [g1, g2]
            h, b = 4 * l - 1, 4 * l  # the stage that holds this layer's hidden rows; its first stage
            stages += [dict(weights=weights[b], gamma=g1, eps=EPS, input=h),
                       dict(weights=weights[b + 1], input=b, offset=0, residual=h),
                       dict(weights=weights[b + 2], gamma=g2, eps=EPS, input=b + 1, flags=ql.QLIN_SWIGLU),
                       dict(weights=weights[b + 3], input=b + 2, residual=b + 1)]
        x = (_rows(case, seed, 0, synth.HIDDEN, "f32") * 0.3).to(torch.float16)
        out = torch.empty((M, synth.HIDDEN), dtype=torch.float16, device="cuda")
        state.update(chain=ql.Chain(stages, max_rows=M), x=x, out=[out], keep=keep)
        return state
    ws = ql.Workspace(M, max(s[0] for s in shapes), max(s[1] for s in shapes))
    state["ws"] = ws
    if kind == "host":
        for i, (K, N, _, sw) in enumerate(shapes):
            a = np.ascontiguousarray(_rows(case, seed, i, K, "f32").cpu().numpy())
            c = np.zeros((M, N // 2 if sw else N), np.float32)
            state["keep"].append(a)
            state["out"].append(c)
            state["calls"].append(_Call("qlin_run_swiglu_f32" if sw else "qlin_run_f32", ws.handle, weights[i].handle, M,
                                        a.ctypes.data_as(ctypes.c_void_p), c.ctypes.data_as(ctypes.c_void_p)))
        return state
    if kind == "linear":
        flags = (ql.QLIN_SWIGLU if case["swiglu"] else 0) | (ql.QLIN_ROUND_HALF_EVEN if case["half_even"] else 0)
        K, N = case["K"], case["N"]
        for i, w in enumerate(weights):
            x = _rows(case, seed, i, K, case["act"])
            out = torch.empty((M, N // 2 if case["swiglu"] else N), dtype=_TORCH[case["out"]], device="cuda")
            gamma = _gamma(seed, i, K) if case["norm"] else None
            res = _rows(case, seed, 200 + i, N, case["out"]) if case["residual"] else None
            state["keep"] += [x, gamma, res]
            state["out"].append(out)
            state["calls"].append(_bind(ws, w, x, out, flags, stream, gamma, res))
        return state
    dt = _TORCH[case["act"]]
    (_, qkv_k, qkv_n), (_, o_k, _), (_, _, gu_n), _ = synth.LAYER
    for l in range(case["layers"]):
        x, att = _rows(case, seed, 2 * l, qkv_k, case["act"]), _rows(case, seed, 2 * l + 1, o_k, case["act"])
        g1, g2 = _gamma(seed, 2 * l, qkv_k), _gamma(seed, 2 * l + 1, qkv_k)
        qkv, h1, mid, h2 = (torch.empty((M, n), dtype=dt, device="cuda") for n in (qkv_n, qkv_k, gu_n // 2, qkv_k))
        wq, wo, wg, wd = weights[4 * l:4 * l + 4]
        state["calls"] += [_bind(ws, wq, x, qkv, 0, stream, gamma=g1), _bind(ws, wo, att, h1, 0, stream, residual=x),
                           _bind(ws, wg, h1, mid, ql.QLIN_SWIGLU, stream, gamma=g2),
                           _bind(ws, wd, mid, h2, 0, stream, residual=h1)]
        state["keep"] += [x, att, g1, g2]
        state["out"] += [qkv, h1, mid, h2]
    return state


def run(state):
    if "chain" in state:
        state["chain"].run(state["x"], state["out"][0])
    else:
        for call in state["calls"]:
            call()
    return state["out"]


# ---- costs and results ----------------------------------------------------------------------


def work(case):
    M, kind = case["rows"], case["kind"]
    a = 4 if kind == "host" else 2 if kind == "chain" else _BYTES[case["act"]]
    nbytes = flops = 0
    for K, N, bits, sw in _linears(case):
        nbytes += N * K * bits // 8 + 4 * N
        flops += 2 * M * N * K
        if kind != "chain":
            nbytes += M * (N // 2 if sw else N) * (_BYTES[case["out"]] if kind == "linear" else a)
        if kind == "linear" or kind == "host":
            nbytes += M * K * a
    if kind == "chain":
        nbytes += 2 * M * synth.HIDDEN * 2
    if kind == "layer":
        nbytes += case["layers"] * M * (synth.HIDDEN + synth.LAYER[1][1]) * a
    if kind == "linear":
        nbytes += case["copies"] * ((case["K"] * 4 if case["norm"] else 0)
                                    + (M * case["N"] * _BYTES[case["out"]] if case["residual"] else 0))
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # About four times what the path shows against exact(): fp16 rows their own rounding (2e-4), and on top of it the
    # activations whose 8-bit code falls the other way when 1 / scale is a float32, which a following linear carries on
    # (single linears up to 4e-4, a layer's SiLU-gate rows 1.4e-3, a chain's four layers in a row 1.6e-2).
    return {"rel": {"chain": 3e-2, "layer": 5e-3}.get(case["kind"], 2e-3)}


def _linear64(x, codes, scales, half_even=False, gamma=None, swiglu=False, residual=None):
    x = x.double()
    if gamma is not None:
        x = x / torch.sqrt(x.square().mean(1, keepdim=True) + EPS) * gamma.double()
    top = x.abs().amax(1, keepdim=True)
    s = torch.where(top == 0, torch.ones_like(top), (top / 127).clamp_min(FLT_MIN))
    v = x / s
    q = torch.round(v) if half_even else torch.sign(v) * torch.floor(v.abs() + 0.5)
    y = (q @ codes.double().t()) * s * scales.double()
    if swiglu:
        n = y.shape[1] // 2
        y = y[:, :n] * torch.sigmoid(y[:, :n]) * y[:, n:]
    return y if residual is None else residual.double() + y


def exact(case, seed):
    kind, shapes = case["kind"], _linears(case)
    if kind == "linear":
        out = []
        for i in range(case["copies"]):
            x = _rows(case, seed, i, case["K"], case["act"])
            gamma = _gamma(seed, i, case["K"]) if case["norm"] else None
            res = _rows(case, seed, 200 + i, case["N"], case["out"]) if case["residual"] else None
            out.append(_linear64(x, *_codes(case, seed, i), case["half_even"], gamma, case["swiglu"], res))
        return out
    if kind == "host":
        return [_linear64(_rows(case, seed, i, K, "f32"), *_codes(case, seed, i), swiglu=sw).cpu().numpy()
                for i, (K, N, _, sw) in enumerate(shapes)]
    # rows handed from one linear to the next are rounded to the type they are stored in
    act = _TORCH["f16" if kind == "chain" else case["act"]]
    out, h = [], None
    if kind == "chain":
        h = (_rows(case, seed, 0, synth.HIDDEN, "f32") * 0.3).to(torch.float16)
    for l in range(case["layers"]):
        wq, wo, wg, wd = (_codes(case, seed, 4 * l + j) for j in range(4))
        g1, g2 = _gamma(seed, 2 * l, synth.HIDDEN), _gamma(seed, 2 * l + 1, synth.HIDDEN)
        x = h if kind == "chain" else _rows(case, seed, 2 * l, synth.HIDDEN, case["act"])
        qkv = _linear64(x, *wq, gamma=g1)
        att = qkv.to(act)[:, :synth.LAYER[1][1]] if kind == "chain" else _rows(case, seed, 2 * l + 1, synth.LAYER[1][1],
                                                                               case["act"])
        h1 = _linear64(att, *wo, residual=x)
        mid = _linear64(h1.to(act), *wg, gamma=g2, swiglu=True)
        h2 = _linear64(mid.to(act), *wd, residual=h1.to(act))
        out += [qkv, h1, mid, h2]
        h = h2.to(act)
    return [h2] if kind == "chain" else out
