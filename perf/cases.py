"""The work that a user of this library has it do, as timed cases.

An engine holds a stack of Gated DeltaNet (GDN) layers with, after every
third, a gated full-attention layer, and calls them for tokens and prompts:

  token     one token per call through host pointers (the C engine's own call)
  decode    the cores of many layers in one launch, one sequence slot per pass
  batch     a serving step: one token for each of B sequences through a layer
  verify    a speculative step: snapshot of the state, then T draft tokens
  prompt    T prompt tokens of one sequence through a GDN layer
  core      the same on pre-projected inputs (projections run elsewhere)
  attn      T tokens at position pos through an attention layer: T = 1 is a
            decode token, a few tokens a speculative step, more a prompt or
            the continuation of one

Layers have the 35B-A3B shapes (GDN: Q35B; attention: 16 query and 2 kv heads
of 256, 64 of them rotated), some drawn ones half of that width.  Weights are
int8 with a scale per row, as the engine streams them, or fp32, as it holds
them otherwise.  Activations are N(0, 1), as a norm leaves them.
"""
from __future__ import annotations

import ctypes
import itertools
import math

import numpy as np
import torch

from overhang_amd import gdn
from overhang_amd.dims import Q35B, GdnDims

HALF = GdnDims(kh=8, vh=16, kd=128, vd=128, K=4, hidden=1024)
GDN = {"35b": Q35B, "half": HALF}
# hidden, query heads, kv heads, head width, rotated dims
ATTN = {"35b": (2048, 16, 2, 256, 64), "half": (1024, 8, 2, 128, 64)}
THETA, EPS = 1e7, 1e-6
MAX_T = 32768                                # an attention layer's cache positions
SLOTS = 17                                   # sequence slots of a decode case: 1 GiB of state at 30 layers


def listed():
    return [
        # the engine's token loop: latency of one host call, launches and copies
        {"name": "token", "kind": "token", "shape": "35b", "int8": True, "B": 1},
        # a token step of a whole model with its projections batched elsewhere
        {"name": "decode_30_layers", "kind": "decode", "shape": "35b", "nl": 30, "B": 1},
        # a server's step over a full and over a partly filled batch
        {"name": "batch_64", "kind": "batch", "shape": "35b", "int8": True, "B": 64},
        {"name": "batch_f32_6", "kind": "batch", "shape": "35b", "int8": False, "B": 6},
        # speculative decoding: five draft tokens checked at once
        {"name": "verify_5", "kind": "verify", "shape": "35b", "int8": True, "T": 5},
        # prompts: a short chat turn, a page, a long document
        {"name": "prompt_150", "kind": "prompt", "shape": "35b", "int8": True, "T": 150},
        {"name": "prompt_4096", "kind": "prompt", "shape": "35b", "int8": True, "T": 4096},
        {"name": "core_32768", "kind": "core", "shape": "35b", "T": 32768},
        # a decode token far into a conversation
        {"name": "attn_token_32767", "kind": "attn", "shape": "35b", "int8": True, "pos": 32767, "T": 1},
        # the attention layer's part of the speculative step
        {"name": "attn_verify_5", "kind": "attn", "shape": "35b", "int8": True, "pos": 8001, "T": 5},
        # a chat turn appended to a conversation
        {"name": "attn_append_333", "kind": "attn", "shape": "35b", "int8": True, "pos": 6000, "T": 333},
        # a long first prompt
        {"name": "attn_prompt_4096", "kind": "attn", "shape": "35b", "int8": True, "pos": 0, "T": 4096},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["token", "decode", "batch", "verify", "prompt", "prompt", "core", "attn1", "attn_few", "append",
                       "attn0"])
    shape = "half" if rng.random() < 0.2 else "35b"
    int8 = rng.random() < 0.75
    if kind == "token":
        return {"kind": "token", "shape": shape, "int8": int8, "B": rng.randint(1, 4)}
    if kind == "decode":
        nl = rng.randint(1, 30)
        return {"kind": "decode", "shape": shape, "nl": nl, "B": rng.randint(1, max(1, 60 // nl))}
    if kind == "batch":
        return {"kind": "batch", "shape": shape, "int8": int8, "B": _log(rng, 1, 64)}
    if kind == "verify":
        return {"kind": "verify", "shape": shape, "int8": int8, "T": rng.randint(2, 16)}
    if kind == "prompt":
        return {"kind": "prompt", "shape": shape, "int8": int8, "T": _log(rng, 17, 4096 if int8 else 1500)}
    if kind == "core":
        return {"kind": "core", "shape": shape, "T": _log(rng, 17, 32768)}
    if kind == "attn1":
        return {"kind": "attn", "shape": shape, "int8": int8, "pos": _log(rng, 1, MAX_T - 1), "T": 1}
    if kind == "attn_few":
        return {"kind": "attn", "shape": shape, "int8": int8, "pos": _log(rng, 100, MAX_T - 16), "T": rng.randint(2, 16)}
    if kind == "append":
        T = _log(rng, 17, 2048)
        most = min(MAX_T - T, 4096 * 4096 // (2 * T))
        return {"kind": "attn", "shape": shape, "int8": int8 or T > 1000, "pos": _log(rng, 100, most), "T": T}
    return {"kind": "attn", "shape": shape, "int8": True, "pos": 0, "T": _log(rng, 17, 4096)}


# ---- inputs, on the GPU, from the seed alone

class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed * 1000003 + 17)

    def normal(self, *shape, mean=0.0, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda").mul_(std).add_(mean)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(shape, generator=self.g, device="cuda").mul_(hi - lo).add_(lo)


def _quantized(W):
    """The engine's load-time rule: per row s = max|w| / 127, q = rint(w / s)."""
    s = (W.abs().amax(1) / 127.0).clamp_min(1e-8)
    return (W / s[:, None]).round_().clamp_(-128, 127).to(torch.int8), s


def _projections(r, rows, int8, std=0.02):
    """{name: (rows, inputs)} as W_* tensors, or as Q_* and S_*."""
    w = {}
    for name, (o, i) in rows.items():
        W = r.normal(o, i, std=std)
        if int8:
            w["Q_" + name], w["S_" + name] = _quantized(W)
        else:
            w["W_" + name] = W
    return w


def _gdn_weights(r, d, projections, int8):
    w = {"conv_w": r.normal(d.conv_dim, d.K, std=0.1), "A_log": r.uniform(d.vh, hi=math.log(16.0)),
         "dt_bias": r.normal(d.vh, std=0.1), "gnorm": r.normal(d.vd, mean=1.0, std=0.1)}
    if projections:
        w.update(_projections(r, {"qkv": (d.conv_dim, d.hidden), "z": (d.val_dim, d.hidden),
                                  "out": (d.hidden, d.val_dim)}, int8))
        w.update(_projections(r, {"b": (d.vh, d.hidden), "a": (d.vh, d.hidden)}, False))
    return w


def _gdn_state(r, d, n):
    """Conv history and recurrent state of n sequences, mid-conversation."""
    return r.normal(n, d.conv_dim, d.K - 1), r.normal(n, d.vh, d.kd, d.vd, std=0.05)


def _core_inputs(r, d, n):
    return {"qkv": r.normal(n, d.conv_dim), "z": r.normal(n, d.val_dim), "a": r.normal(n, d.vh), "b": r.normal(n, d.vh)}


def _inputs(case, seed):
    r, kind = _Rand(seed), case["kind"]
    if kind == "attn":
        D, H, KV, hd, _ = ATTN[case["shape"]]
        w = _projections(r, {"q": (2 * H * hd, D), "k": (KV * hd, D), "v": (KV * hd, D), "o": (D, H * hd)}, case["int8"])
        w.update(q_norm=r.normal(hd, std=0.1), k_norm=r.normal(hd, std=0.1))
        return {"w": w, "K": r.normal(KV, case["pos"], hd), "V": r.normal(KV, case["pos"], hd), "x": r.normal(case["T"], D)}
    d = GDN[case["shape"]]
    n = case.get("B", 1)
    nl = case.get("nl", 1)
    proj = kind not in ("decode", "core")
    w = [_gdn_weights(r, d, proj, case.get("int8", False)) for _ in range(nl)]
    state = [_gdn_state(r, d, n) for _ in range(nl)]
    rows = case["T"] if "T" in case else nl * n
    x = r.normal(rows, d.hidden) if proj else _core_inputs(r, d, rows)
    return {"w": w, "state": state, "x": x}


# ---- what a program holds before the call

_gdn_ids = itertools.cycle(range(4096))
_attn_ids = itertools.cycle(range(4096))


class _State:
    """A program's layers, inputs and output buffers; the layers are given back with it."""

    def __init__(self, case):
        self.case, self.layers, self.step = case, [], 0

    def __del__(self):
        for layer in self.layers:
            layer.free()


def _host(t):
    return t.cpu().numpy()


def prepare(case, seed):
    s, inp, kind = _State(case), _inputs(case, seed), case["kind"]
    if kind == "attn":
        D, H, KV, hd, rot = ATTN[case["shape"]]
        layer = gdn.AttnLayer(next(_attn_ids), D, H, KV, hd, rot, THETA, EPS, MAX_T,
                              {k: _host(v) for k, v in inp["w"].items()})
        s.layers.append(layer)
        if case["pos"]:
            layer.cache_set(0, 0, case["pos"], _host(inp["K"]), _host(inp["V"]))
        s.x, s.out = inp["x"], torch.empty_like(inp["x"])
        return s
    d = GDN[case["shape"]]
    B = case.get("B", 1)
    slots = {"decode": SLOTS * B, "verify": 2}.get(kind, B)
    for w, (conv, S) in zip(inp["w"], inp["state"]):
        layer = gdn.GdnLayer(next(_gdn_ids), d, {k: _host(v) for k, v in w.items()}, max_seqs=slots)
        s.layers.append(layer)
        for b, (c, m) in enumerate(zip(_host(conv), _host(S))):
            layer.set_state(b, c, m)
    s.lis = [layer.li for layer in s.layers]
    if kind == "decode":
        for slot in range(B, slots):
            gdn.state_copy(s.lis, slot % B, slot)
    s.x = inp["x"]
    if kind == "token":
        s.x = _host(s.x)
    elif kind in ("decode", "core"):
        s.out = torch.empty_like(s.x["z"])
    else:
        s.out = torch.empty_like(s.x)
    return s


def run(s):
    case, x = s.case, s.x
    kind = case["kind"]
    if kind == "token":
        return s.layers[0].decode(x)
    stream = torch.cuda.current_stream()
    if kind == "attn":
        gdn.attn_forward_dev(s.layers[0].li, 0, case["pos"], case["T"], x, s.out, stream)
    elif kind == "decode":
        # the next group of sequence slots in every layer
        slot = s.step % SLOTS * case["B"]
        s.step += 1
        gdn.decode_core_seq_dev(s.lis, slot, case["B"], x["qkv"], x["z"], x["a"], x["b"], s.out, stream)
    elif kind == "batch":
        gdn.decode_dev(s.lis[0], case["B"], x, s.out, stream)
    elif kind == "core":
        gdn.prefill_core_dev(s.lis[0], 0, case["T"], x["qkv"], x["z"], x["a"], x["b"], s.out, stream)
    else:
        if kind == "verify":
            gdn.state_copy_dev(s.lis, 0, 1, stream)      # what a rejected draft goes back to
        gdn.prefill_dev(s.lis[0], 0, case["T"], x, s.out, stream)
    return s.out


# ---- what a pass cannot do without

def _matrix(rows, cols, int8):
    return rows * cols * (1 if int8 else 4) + (4 * rows if int8 else 0)


def work(case):
    kind = case["kind"]
    if kind == "attn":
        D, H, KV, hd, _ = ATTN[case["shape"]]
        T, pos = case["T"], case["pos"]
        rows, o = 2 * H * hd + 2 * KV * hd, H * hd
        weights = _matrix(rows, D, case["int8"]) + _matrix(D, o, case["int8"])
        cache = 2 * KV * hd * 4 * (pos + T)
        pairs = T * pos + T * (T + 1) // 2
        return {"bytes": weights + cache + 8 * T * D, "flops": 2 * T * (rows * D + D * o) + 4 * H * hd * pairs}
    d = GDN[case["shape"]]
    tokens = case["T"] if "T" in case else case.get("nl", 1) * case["B"]
    states = 1 if "T" in case else tokens
    io = d.conv_dim + 2 * d.val_dim + 2 * d.vh                          # pre-projected rows in, core rows out
    state = 2 * d.state_bytes + 4 * d.conv_dim * d.K
    nbytes, flops = states * state, tokens * 7 * d.vh * d.kd * d.vd    # decay, S^T k, rank-1 update, S^T q
    if kind in ("decode", "core"):
        nbytes += 4 * tokens * io
    else:
        rows = d.conv_dim + d.val_dim
        nbytes += (_matrix(rows, d.hidden, case["int8"]) + _matrix(d.hidden, d.val_dim, case["int8"]) +
                   _matrix(2 * d.vh, d.hidden, False) + 8 * tokens * d.hidden)
        flops += 2 * tokens * d.hidden * (rows + 2 * d.vh + d.val_dim)
    if kind == "verify":
        nbytes += state
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Four times what these paths differ from 64 bits by.  Several tokens at
    # once: 3e-6 to 8e-6, x entering the int8 projections to 2^-20 of its
    # row's largest value and attention's products being of bf16 pairs (2^-16
    # each).  fp32 sums alone, in another order: 2e-7 to 1.3e-6.
    if case["kind"] == "attn":
        return {"rel": 3e-5 if case["T"] > 1 else 5e-6}
    if case["kind"] in ("batch", "verify", "prompt"):
        return {"rel": 3e-5 if case["int8"] else 1e-5}
    return {"rel": 5e-6}


# ---- the same in 64 bits, from the definitions

def _dequantized(w, name):
    if "Q_" + name in w:
        return w["Q_" + name].double() * w["S_" + name].double()[:, None]
    return w["W_" + name].double()


def _gdn_core64(d, w, x, conv, S):
    """x: rows [n][T][...] of n sequences; conv [n][conv_dim][K-1], S [n][vh][kd][vd]."""
    n, T = x["qkv"].shape[:2]
    hist = torch.cat([conv.double(), x["qkv"].double().transpose(1, 2)], 2)
    c = sum(hist[:, :, j:j + T] * w["conv_w"].double()[None, :, j, None] for j in range(d.K)).transpose(1, 2)
    c = c * torch.sigmoid(c)
    q, k, v = c.split([d.key_dim, d.key_dim, d.val_dim], 2)
    q, k = (t.reshape(n, T, d.kh, d.kd) for t in (q, k))
    q, k = (t / (t.square().sum(3, True) + 1e-6).sqrt() for t in (q, k))
    q, k = (t.repeat_interleave(d.rep, 2) for t in (q / math.sqrt(d.kd), k))
    v = v.reshape(n, T, d.vh, d.vd)
    decay = torch.exp(-w["A_log"].double().exp() * torch.nn.functional.softplus(x["a"].double() + w["dt_bias"].double()))
    beta = torch.sigmoid(x["b"].double())
    S, o = S.double().clone(), torch.empty(n, T, d.vh, d.vd, dtype=torch.float64, device=S.device)
    for t in range(T):
        kt = k[:, t, :, None, :]
        S *= decay[:, t, :, None, None]
        delta = beta[:, t, :, None, None] * (v[:, t, :, None, :] - kt @ S)
        S += kt.transpose(2, 3) * delta
        o[:, t] = (q[:, t, :, None, :] @ S)[:, :, 0]
    z = x["z"].double().reshape(o.shape)
    o = o / (o.square().mean(3, True) + d.eps).sqrt() * w["gnorm"].double() * z * torch.sigmoid(z)
    return o.reshape(n, T, d.val_dim)


def _attn64(case, inp):
    D, H, KV, hd, rot = ATTN[case["shape"]]
    w, T, pos = inp["w"], case["T"], case["pos"]
    x = inp["x"].double()
    qg = (x @ _dequantized(w, "q").T).reshape(T, H, 2 * hd)
    q, gate = qg[..., :hd], qg[..., hd:]
    k = (x @ _dequantized(w, "k").T).reshape(T, KV, hd)
    v = (x @ _dequantized(w, "v").T).reshape(T, KV, hd)
    # the angles are the engine's fp32 ones: position times the C library's powf
    powf = ctypes.CDLL("libm.so.6").powf
    powf.restype, powf.argtypes = ctypes.c_float, [ctypes.c_float, ctypes.c_float]
    inv = np.array([powf(THETA, -(2.0 * j) / rot) for j in range(rot // 2)], np.float32)
    ang = torch.from_numpy(np.arange(pos, pos + T, dtype=np.float32)[:, None] * inv).to(x.device).double()[:, None]
    cos, sin = ang.cos(), ang.sin()

    def head(t, norm):
        t = t / (t.square().mean(2, True) + EPS).sqrt() * (1 + norm.double())
        a, b, rest = t.split([rot // 2, rot // 2, hd - rot], 2)
        return torch.cat([a * cos - b * sin, b * cos + a * sin, rest], 2)

    q, k = head(q, w["q_norm"]), head(k, w["k_norm"])
    out = torch.empty(T, H, hd, dtype=torch.float64, device=x.device)
    hidden = torch.arange(pos + T, device=x.device) > torch.arange(pos, pos + T, device=x.device)[:, None]
    for h in range(H):
        g = h // (H // KV)
        keys, values = torch.cat([inp["K"][g].double(), k[:, g]]), torch.cat([inp["V"][g].double(), v[:, g]])
        score = (q[:, h] @ keys.T / math.sqrt(hd)).masked_fill_(hidden, -math.inf)
        out[:, h] = torch.softmax(score, 1) @ values
    return (out * torch.sigmoid(gate)).reshape(T, H * hd) @ _dequantized(w, "o").T


def exact(case, seed):
    inp = _inputs(case, seed)
    if case["kind"] == "attn":
        return _attn64(case, inp)
    d = GDN[case["shape"]]
    n = case.get("B", 1)
    if case["kind"] in ("decode", "core"):
        out, x = [], inp["x"]
        for i, (w, (conv, S)) in enumerate(zip(inp["w"], inp["state"])):
            rows = {k: v.reshape(len(inp["w"]), n, -1, v.shape[1])[i] for k, v in x.items()}
            out.append(_gdn_core64(d, w, rows, conv, S))
        return torch.cat(out).reshape(x["z"].shape)
    w, (conv, S) = inp["w"][0], inp["state"][0]
    x = inp["x"].double().reshape(n, -1, d.hidden)
    rows = {k: x @ _dequantized(w, k).T for k in ("qkv", "z", "a", "b")}
    core = _gdn_core64(d, w, rows, conv, S)
    return (core @ _dequantized(w, "out").T).reshape(inp["x"].shape)
