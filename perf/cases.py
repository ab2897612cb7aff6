"""The token-mixer calls that a serving program makes, as timed cases.

A program decodes (one token of each of B sequences per call), verifies a few
drafted tokens, and prefills prompts, each through the C ABI of libvx27_hip
on device-resident data:

  dn_step      the Gated DeltaNet mixer core, one token of B sequences
  gqa_step     the gated GQA mixer core over a bf16 KV cache, one token
  dn_layer     a DeltaNet layer (projections, core, output projection), one token
  gqa_layer    a gated GQA layer, one token, every sequence at its own position
  decode_step  three DeltaNet layers and one GQA layer (the period of the
               64-mixer stack), captured once as a graph and replayed per token
  dn_verify    a DeltaNet layer over a window of drafted tokens with a state
               checkpoint after each
  dn_prompt    a DeltaNet layer over a prompt
  gqa_prompt   a gated GQA layer over a prompt, or over a later turn of a
               conversation whose first pos0 positions are cached
  dn_prefill   the DeltaNet mixer core over a prompt, bf16 q, k and v

Shapes are those of the Qwen 27B hybrid's mixers: hidden 5120; DeltaNet 16 QK
and 48 value heads of 128 (16 and 16 for the core alone); GQA 24 query and 4
KV heads of 256, RoPE over 64 dimensions.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from vx27_amd import lib as L

H = 5120                       # hidden size
NQK, NV, HD = 16, 48, 128      # DeltaNet heads of a layer
NQ, NKV, GD = 24, 4, 256       # GQA heads
ROPE, THETA = 64, 1e7
DEV = "cuda"

_ctx = None


def ctx():
    """The process's context, as a serving program keeps one per GPU."""
    global _ctx
    if _ctx is None:
        _ctx = L.Ctx(0)
    return _ctx


# ------------------------------------------------------------------- cases
def listed():
    return [
        # one user, the smallest call: launch latency and one short chain
        {"name": "dn_step_b1", "kind": "dn_step", "B": 1, "conv": True},
        # one user at an ordinary context: three launches around 34 MB of cache
        {"name": "gqa_step_b1_8k", "kind": "gqa_step", "B": 1, "ctx": 8191, "gate": True},
        # a small server's decode: the weights bound it
        {"name": "dn_layer_b4", "kind": "dn_layer", "B": 4, "conv_bf16": True},
        # a busy server's decode, many vectors per pass over the weights
        {"name": "dn_layer_b64", "kind": "dn_layer", "B": 64, "conv_bf16": True},
        # continuous batching: an odd batch, every sequence at another position
        {"name": "gqa_layer_b23", "kind": "gqa_layer", "B": 23, "ctx": 5000},
        # long-context decode through a captured graph
        {"name": "decode_step_b4_128k", "kind": "decode_step", "B": 4, "ctx": 131072},
        # speculative decoding: the verify batch of six drafted tokens
        {"name": "dn_verify_t6", "kind": "dn_verify", "B": 1, "T": 6},
        # an ordinary short question
        {"name": "dn_prompt_t187", "kind": "dn_prompt", "B": 1, "T": 187, "conv_bf16": True},
        # a long prompt
        {"name": "dn_prompt_t4096", "kind": "dn_prompt", "B": 1, "T": 4096, "conv_bf16": True},
        {"name": "gqa_prompt_t4096", "kind": "gqa_prompt", "B": 1, "T": 4096, "pos0": 0},
        # the next turn of two conversations of equal length
        {"name": "gqa_prompt_b2_t613", "kind": "gqa_prompt", "B": 2, "T": 613, "pos0": 2891},
        # the recurrence alone over a long prompt, for programs with their own projections
        {"name": "dn_prefill_t4096", "kind": "dn_prefill", "B": 1, "T": 4096, "bf16": False},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["dn_step", "gqa_step", "dn_layer", "gqa_layer", "decode_step", "dn_verify", "dn_prompt",
                       "gqa_prompt", "dn_prefill"])
    if kind == "dn_step":
        return {"kind": kind, "B": _log_int(rng, 1, 64), "conv": rng.random() < 0.7}
    if kind == "gqa_step":
        B = _log_int(rng, 1, 32)
        return {"kind": kind, "B": B, "ctx": _log_int(rng, 30, 524288 // max(B, 4)), "gate": rng.random() < 0.75}
    if kind == "dn_layer":
        return {"kind": kind, "B": _log_int(rng, 1, 64), "conv_bf16": rng.random() < 0.75}
    if kind == "gqa_layer":
        B = _log_int(rng, 1, 64)
        return {"kind": kind, "B": B, "ctx": _log_int(rng, 100, 262144 // max(B, 8))}
    if kind == "decode_step":
        B = _log_int(rng, 1, 8)
        return {"kind": kind, "B": B, "ctx": _log_int(rng, 500, 524288 // max(B, 4))}
    if kind == "dn_verify":
        return {"kind": kind, "B": rng.randint(1, 4), "T": rng.randint(2, 8)}
    B = rng.choice([1, 1, 1, 2, 3])
    T = _log_int(rng, 9, 4096 // B)
    if kind == "dn_prompt":
        return {"kind": kind, "B": B, "T": T, "conv_bf16": rng.random() < 0.75}
    if kind == "gqa_prompt":
        return {"kind": kind, "B": B, "T": T, "pos0": rng.choice([0, rng.randint(1, 4096 - T)]) if T < 4096 else 0}
    return {"kind": kind, "B": B, "T": T, "bf16": rng.random() < 0.25}


# ------------------------------------------------------------------ inputs
class _Rand:
    """Device tensors from the seed alone, in call order."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(1000003 * int(seed) + 17)

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.g, device=DEV, dtype=torch.float32) * std + mean).to(dtype)

    def bf16(self, *shape):
        """N(0, 1) in bf16, made in place (for large caches)."""
        return torch.empty(*shape, device=DEV, dtype=torch.bfloat16).normal_(generator=self.g)

    def uniform(self, *shape, lo, hi):
        return torch.rand(*shape, generator=self.g, device=DEV) * (hi - lo) + lo

    def ints(self, lo, hi, n):
        return torch.randint(lo, hi + 1, (n,), generator=self.g, device=DEV, dtype=torch.int32)


def _tiled(w):
    """Row-major weights in the layout that the layer calls read (laid out once, when a program loads them)."""
    out = torch.empty_like(w)
    torch.cuda.synchronize()
    c = ctx()
    L.check(L.lib().vx27_hip_pack_weights_bf16(c.h, w.data_ptr(), w.shape[0], w.shape[1], out.data_ptr()), "pack")
    c.sync()
    return out


def _dn_heads(r, nv):
    return {"A_log": r.uniform(nv, lo=-2.0, hi=1.0), "dt_bias": r.normal(nv, std=0.1)}


def _dn_weights(r, conv_bf16=True):
    """A DeltaNet layer's weights, row-major."""
    Cc = (2 * NQK + NV) * HD
    w = _dn_heads(r, NV)
    w["w_in"] = r.normal(Cc + NV * HD + 2 * NV, H, std=0.02, dtype=torch.bfloat16)
    w["w_out"] = r.normal(H, NV * HD, std=0.02, dtype=torch.bfloat16)
    w["conv_w"] = r.normal(Cc, 4, std=0.2, dtype=torch.bfloat16 if conv_bf16 else torch.float32)
    w["norm_w"] = r.normal(HD, std=0.1, mean=1.0)
    return w


def _dn_state(r, B, nqk, nv):
    return {"S": r.normal(B, nv, HD, HD, std=0.02), "conv_state": r.normal(B, (2 * nqk + nv) * HD, 3, std=0.5)}


def _gqa_weights(r):
    return {"w_qkv": r.normal(2 * NQ * GD + 2 * NKV * GD, H, std=0.02, dtype=torch.bfloat16),
            "w_o": r.normal(H, NQ * GD, std=0.02, dtype=torch.bfloat16),
            "q_norm_w": r.normal(GD, std=0.1), "k_norm_w": r.normal(GD, std=0.1)}


def _capacity(n):
    return (n + 63) // 64 * 64


def _caches(r, B, n):
    cap = _capacity(n)
    return {"k_cache": r.bf16(B, NKV, cap, GD), "v_cache": r.bf16(B, NKV, cap // 32, GD, 32)}


def _inputs(case, seed):
    """Everything the call reads, as plain tensors (weights row-major)."""
    r, kind, B = _Rand(seed), case["kind"], case["B"]
    if kind == "dn_step":
        i = {**_dn_heads(r, 16), **_dn_state(r, B, 16, 16), "a": r.normal(B, 16), "b": r.normal(B, 16)}
        if case["conv"]:
            i["x"] = r.normal(B, 48 * HD)
            i["conv_w"] = r.normal(48 * HD, 4, std=0.2, dtype=torch.bfloat16)
        else:
            i.update(q=r.normal(B, 16, HD), k=r.normal(B, 16, HD), v=r.normal(B, 16, HD))
            del i["conv_state"]
        return i
    if kind == "gqa_step":
        i = {"qg": r.normal(B, NQ, 2 * GD), "k_new": r.normal(B, NKV, GD), "v_new": r.normal(B, NKV, GD),
             "q_norm_w": r.normal(GD, std=0.1), "k_norm_w": r.normal(GD, std=0.1),
             **_caches(r, B, case["ctx"] + 1)}
        i["pos"] = torch.full((B,), case["ctx"], device=DEV, dtype=torch.int32)
        return i
    if kind == "dn_layer":
        return {"x": r.normal(B, H), **_dn_weights(r, case["conv_bf16"]), **_dn_state(r, B, NQK, NV)}
    if kind == "gqa_layer":
        return {"x": r.normal(B, H), **_gqa_weights(r), **_caches(r, B, case["ctx"] + 1),
                "pos": r.ints(case["ctx"] // 4, case["ctx"], B)}
    if kind == "decode_step":
        return {"x": r.normal(B, H), "dn": [{**_dn_weights(r), **_dn_state(r, B, NQK, NV)} for _ in range(3)],
                "gqa": {**_gqa_weights(r), **_caches(r, B, case["ctx"] + 1)},
                "pos": r.ints(case["ctx"] - case["ctx"] // 16, case["ctx"], B)}
    T = case["T"]
    if kind in ("dn_verify", "dn_prompt"):
        return {"x": r.normal(B, T, H), **_dn_weights(r, case.get("conv_bf16", True)), **_dn_state(r, B, NQK, NV)}
    if kind == "gqa_prompt":
        return {"x": r.normal(B, T, H), **_gqa_weights(r), **_caches(r, B, case["pos0"] + T)}
    i = {**_dn_heads(r, 16), "S": r.normal(B, 16, HD, HD, std=0.02)}
    i.update(q=r.bf16(B, T, 16, HD), k=r.bf16(B, T, 16, HD), v=r.bf16(B, T, 16, HD))
    i.update(a=r.normal(B, T, 16), b=r.normal(B, T, 16))
    return i


# ------------------------------------------------------------- the calls
def _p(t):
    return t.data_ptr() if t is not None else None


def _dt(t):
    return L.BF16 if t.dtype == torch.bfloat16 else L.F32


def _new(*shape):
    return torch.empty(*shape, device=DEV)


class _Graph:
    """A captured step, given back when its owner goes."""

    def __init__(self, calls):
        c = ctx()
        for fn, d in calls:     # once eagerly: the context's scratch has its size before the capture
            L.check(fn(c.h, C.byref(d)), "warm-up")
        c.sync()
        c.graph_begin()
        for fn, d in calls:
            L.check(fn(c.h, C.byref(d)), "capture")
        self.exec = c.graph_end()

    def __del__(self):
        L.lib().vx27_hip_graph_destroy(self.exec)


def _dn_layer_desc(i, x, B, out):
    return L.DnLayerDesc(B, NQK, NV, HD, H, _p(x), None, _p(i["w_in"]), _p(i["w_out"]), _p(i["conv_w"]),
                         _dt(i["conv_w"]), _p(i["A_log"]), _p(i["dt_bias"]), _p(i["norm_w"]), _p(i["S"]),
                         _p(i["conv_state"]), _p(out))


def _gqa_layer_desc(i, x, pos, B, out):
    return L.GqaLayerDesc(B, NQ, NKV, GD, H, ROPE, THETA, 1.0, i["k_cache"].shape[2], _p(x), None, _p(i["w_qkv"]),
                          _p(i["w_o"]), _p(i["q_norm_w"]), _p(i["k_norm_w"]), _p(pos), _p(i["k_cache"]),
                          _p(i["v_cache"]), _p(out), 0)


def prepare(case, seed):
    i, kind, B, lib = _inputs(case, seed), case["kind"], case["B"], L.lib()
    for w in [i, *i.get("dn", []), i.get("gqa", {})]:
        for n in ("w_in", "w_out", "w_qkv", "w_o"):
            if n in w:
                w[n] = _tiled(w[n])
    s = {"in": i, "h": ctx().h}     # the tensors are kept: the descriptors hold their addresses
    if kind == "dn_step":
        out = _new(B, 16, HD)
        d = L.DnDesc()
        d.B, d.nqk, d.nv, d.hd, d.steps = B, 16, 16, HD, 1
        d.flags = L.DN_CONV | L.DN_PRE_L2 if case["conv"] else 0
        for n in ("S", "conv_state", "conv_w", "x", "q", "k", "v", "a", "b", "A_log", "dt_bias"):
            setattr(d, n, _p(i.get(n)))
        d.conv_w_dtype, d.out = L.BF16, _p(out)
        s.update(fn=lib.vx27_hip_dn_decode, d=d, outs=[out, i["S"], i.get("conv_state")])
    elif kind == "gqa_step":
        out = _new(B, NQ, GD)
        d = L.GqaDesc()
        d.B, d.n_q, d.n_kv, d.hd, d.rope_dim, d.rope_theta, d.rope_yarn = B, NQ, NKV, GD, ROPE, THETA, 1.0
        d.L, d.flags = i["k_cache"].shape[2], 0 if case["gate"] else L.GQA_NO_GATE
        for n in ("pos", "k_new", "v_new", "q_norm_w", "k_norm_w", "k_cache", "v_cache"):
            setattr(d, n, _p(i[n]))
        d.q, d.gate, d.out = _p(i["qg"]), _p(i["qg"]) + 4 * GD, _p(out)
        d.q_seq_stride = d.gate_seq_stride = NQ * 2 * GD
        d.q_head_stride = d.gate_head_stride = 2 * GD
        s.update(fn=lib.vx27_hip_gqa_decode, d=d, outs=[out, i["k_cache"], i["v_cache"]])
    elif kind == "dn_layer":
        out = _new(B, H)
        s.update(fn=lib.vx27_hip_dn_layer_decode, d=_dn_layer_desc(i, i["x"], B, out),
                 outs=[out, i["S"], i["conv_state"]])
    elif kind == "gqa_layer":
        out = _new(B, H)
        s.update(fn=lib.vx27_hip_gqa_layer_decode, d=_gqa_layer_desc(i, i["x"], i["pos"], B, out),
                 outs=[out, i["k_cache"], i["v_cache"]])
    elif kind == "decode_step":
        outs = [_new(B, H) for _ in range(4)]
        calls = [(lib.vx27_hip_dn_layer_decode, _dn_layer_desc(w, i["x"], B, o)) for w, o in zip(i["dn"], outs)]
        calls.append((lib.vx27_hip_gqa_layer_decode, _gqa_layer_desc(i["gqa"], i["x"], i["pos"], B, outs[3])))
        before = [(w["S"].clone(), w["conv_state"].clone()) for w in i["dn"]]
        torch.cuda.synchronize()
        s["graph"] = _Graph(calls)
        ctx().sync()
        for w, (S, cs) in zip(i["dn"], before):     # the warm-up took a step
            w["S"].copy_(S)
            w["conv_state"].copy_(cs)
        s["outs"] = [*outs, *(w["S"] for w in i["dn"]), *(w["conv_state"] for w in i["dn"]), i["gqa"]["k_cache"],
                     i["gqa"]["v_cache"]]
    elif kind in ("dn_verify", "dn_prompt"):
        T, out = case["T"], _new(B, case["T"], H)
        d = L.DnLayerPrefillDesc()
        d.B, d.T, d.nqk, d.nv, d.hd, d.hidden, d.conv_w_dtype = B, T, NQK, NV, HD, H, _dt(i["conv_w"])
        for n in ("x", "w_in", "w_out", "conv_w", "A_log", "dt_bias", "norm_w", "S", "conv_state"):
            setattr(d, n, _p(i[n]))
        d.out, outs = _p(out), [out, i["S"], i["conv_state"]]
        if kind == "dn_verify":
            ckpt = [_new(B, T, NV, HD, HD), _new(B, T, (2 * NQK + NV) * HD, 3)]
            d.S_ckpt, d.conv_ckpt = _p(ckpt[0]), _p(ckpt[1])
            outs += ckpt
        s.update(fn=lib.vx27_hip_dn_layer_prefill, d=d, outs=outs)
    elif kind == "gqa_prompt":
        T, out = case["T"], _new(B, case["T"], H)
        d = L.GqaLayerPrefillDesc()
        d.B, d.T, d.n_q, d.n_kv, d.hd, d.hidden = B, T, NQ, NKV, GD, H
        d.rope_dim, d.rope_theta, d.rope_yarn = ROPE, THETA, 1.0
        d.L, d.pos0, d.flags, d.out = i["k_cache"].shape[2], case["pos0"], 0, _p(out)
        for n in ("x", "w_qkv", "w_o", "q_norm_w", "k_norm_w", "k_cache", "v_cache"):
            setattr(d, n, _p(i[n]))
        s.update(fn=lib.vx27_hip_gqa_layer_prefill, d=d, outs=[out, i["k_cache"], i["v_cache"]])
    else:
        T, out = case["T"], _new(B, case["T"], 16, HD)
        d = L.DnPrefillDesc()
        d.B, d.T, d.nqk, d.nv, d.hd, d.flags = B, T, 16, 16, HD, L.DN_BF16 if case["bf16"] else 0
        for n in ("S", "q", "k", "v", "a", "b", "A_log", "dt_bias"):
            setattr(d, n, _p(i[n]))
        d.out = _p(out)
        s.update(fn=lib.vx27_hip_dn_prefill, d=d, outs=[out, i["S"]])
    s["outs"] = [o for o in s["outs"] if o is not None]
    torch.cuda.synchronize()
    return s


def run(s):
    if "graph" in s:
        rc = L.lib().vx27_hip_graph_launch(s["h"], s["graph"].exec)
    else:
        rc = s["fn"](s["h"], C.byref(s["d"]))
    if rc != 0:
        L.check(rc, "run")
    return s["outs"]


# -------------------------------------------------------------- the work
DN_CH = (2 * NQK + NV) * HD                      # q|k|v channels of a layer
DN_W = (DN_CH + NV * HD + 2 * NV) * H + H * NV * HD
GQ_N = 2 * NQ * GD + 2 * NKV * GD
GQ_W = GQ_N * H + H * NQ * GD


def _dn_core(tokens, B, nv):
    """(bytes of the state, read and written; operations of the recurrence: kv, the rank-1 update and the output)."""
    return 2 * B * nv * HD * HD * 4, tokens * nv * 6 * HD * HD


def work(case):
    kind, B = case["kind"], case["B"]
    if kind == "dn_step":
        by, fl = _dn_core(B, B, 16)
        ch = 48 * HD
        by += B * (ch + 16 * HD + 32) * 4 + (B * ch * 6 * 4 + ch * 8 if case["conv"] else 0)
        return {"bytes": by, "flops": fl}
    if kind == "gqa_step":
        n = case["ctx"] + 1
        return {"bytes": B * (n * NKV * GD * 4 + (NQ * 3 + NKV * 2) * GD * 4), "flops": B * n * NQ * GD * 4}
    if kind == "dn_layer":
        by, fl = _dn_core(B, B, NV)
        return {"bytes": by + 2 * DN_W + B * (2 * H + 6 * DN_CH) * 4, "flops": fl + 2 * B * DN_W}
    if kind == "gqa_layer":
        n = B * (case["ctx"] * 5 // 8 + 1)
        return {"bytes": n * NKV * GD * 4 + 2 * GQ_W + 2 * B * H * 4, "flops": n * NQ * GD * 4 + 2 * B * GQ_W}
    if kind == "decode_step":
        dn = work({"kind": "dn_layer", "B": B})
        n = B * (case["ctx"] * 31 // 32 + 1)
        return {"bytes": 3 * dn["bytes"] + n * NKV * GD * 4 + 2 * GQ_W + 2 * B * H * 4,
                "flops": 3 * dn["flops"] + n * NQ * GD * 4 + 2 * B * GQ_W}
    R = B * case["T"]
    if kind in ("dn_verify", "dn_prompt"):
        by, fl = _dn_core(R, B, NV)
        by += 2 * DN_W + R * 2 * H * 4 + B * 6 * DN_CH * 4
        if kind == "dn_verify":
            by += R * (NV * HD * HD + 3 * DN_CH) * 4
        return {"bytes": by, "flops": fl + 2 * R * DN_W}
    if kind == "gqa_prompt":
        keys = R * case["pos0"] + B * case["T"] * (case["T"] + 1) // 2
        return {"bytes": 2 * GQ_W + R * 2 * H * 4 + B * (case["pos0"] + case["T"]) * NKV * GD * 4,
                "flops": keys * NQ * GD * 4 + 2 * R * GQ_W}
    by, fl = _dn_core(R, B, 16)
    return {"bytes": by + R * 16 * (3 * HD * 2 + HD * 4 + 8), "flops": fl}


def tolerance(case):
    """About four times the distance from the 64-bit results that the calls measured at over these ranges."""
    kind = case["kind"]
    if kind in ("dn_step", "dn_layer", "dn_verify"):
        return {"rel": 2e-6}        # 32-bit state and sums: 1e-7 .. 4e-7
    if kind == "dn_prompt":
        return {"rel": 4e-5}        # chunk products of bf16 pairs: 6e-6 .. 9e-6
    if kind == "dn_prefill":
        return {"rel": 2e-2 if case["bf16"] else 2e-5}      # bf16 operands, or pairs of them: 5e-6
    return {"rel": 1.4e-2}          # bf16 queries, keys, values and weights of the softmax: 2e-3 .. 3.6e-3


# ------------------------------------------------------- the same in 64 bits
def _d(t):
    return t.double()


def _silu(t):
    return t * torch.sigmoid(t)


def _l2(t):
    return t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)


def _rms(t):
    return t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-6)


def _dn_exact(i, x, a, b, T, flags_conv, layer, qkv=None, z=None, every=False):
    """The DeltaNet branch over [B][T] tokens: x [B][T][C] or qkv = (q, k, v).
    Returns out [B][T][nv][128], the final state and conv state, and with
    `every` the state and conv state after each token."""
    nqk, nv = (NQK, NV) if layer else (16, 16)
    S = _d(i["S"])
    B, cs, conv_all = S.shape[0], None, []
    if flags_conv:
        w, cat = _d(i["conv_w"]), torch.cat([_d(i["conv_state"]).transpose(1, 2), x], 1)    # [B][T+3][C]
        act = _silu(sum(w[:, j] * cat[:, j:j + T] for j in range(4)))
        cs = cat[:, T:].transpose(1, 2).contiguous()
        conv_all = [cat[:, t + 1:t + 4].transpose(1, 2) for t in range(T)] if every else []
        q, k, v = torch.split(act, [nqk * HD, nqk * HD, nv * HD], -1)
        q, k, v = q.reshape(B, T, nqk, HD), k.reshape(B, T, nqk, HD), v.reshape(B, T, nv, HD)
        if layer:
            w1 = 1 + _d(i["norm_w"])
            q, k = _rms(q) * w1, _rms(k) * w1
        q, k = _l2(q) / math.sqrt(HD), _l2(k)
    else:
        q, k, v = (_d(t) for t in qkv)
    q, k = _l2(q) / math.sqrt(HD), _l2(k)
    q, k = (t.repeat_interleave(nv // nqk, 2) for t in (q, k))
    beta = torch.sigmoid(b)
    decay = torch.exp(-torch.exp(_d(i["A_log"])) * torch.nn.functional.softplus(a + _d(i["dt_bias"])))
    out, S_all = torch.empty(B, T, nv, HD, device=DEV, dtype=torch.float64), []
    for t in range(T):
        kt, qt = k[:, t].unsqueeze(-1), q[:, t].unsqueeze(-1)
        S = S * decay[:, t, :, None, None]
        delta = (v[:, t] - (S * kt).sum(2)) * beta[:, t, :, None]
        S = S + kt * delta.unsqueeze(2)
        out[:, t] = (S * qt).sum(2)
        if every:
            S_all.append(S)
    if layer:
        out = _rms(out) * _d(i["norm_w"]) * _silu(z)
    return out, S, cs, S_all, conv_all


def _dn_layer_exact(i, x, every=False):
    B, T = x.shape[:2]
    y = (_d(x).reshape(B * T, H) @ _d(i["w_in"]).t()).reshape(B, T, -1)
    qkv, z, a, b = torch.split(y, [DN_CH, NV * HD, NV, NV], -1)
    o, S, cs, S_all, c_all = _dn_exact(i, qkv, a, b, T, True, True, z=z.reshape(B, T, NV, HD), every=every)
    out = (o.reshape(B * T, NV * HD) @ _d(i["w_out"]).t()).reshape(B, T, H)
    return out, S, cs, S_all, c_all


def _rope(t, pos):
    """Rotate t [T][heads][256] at positions pos [T] (the angle is the product of two 32-bit floats)."""
    half = ROPE // 2
    freq = np.power(np.float32(THETA), (np.float32(-2.0) * np.arange(half, dtype=np.float32)) / np.float32(ROPE))
    ang = pos.to(torch.float32).unsqueeze(1) * torch.from_numpy(freq.astype(np.float32)).to(DEV)
    c, s = torch.cos(ang.double()).unsqueeze(1), torch.sin(ang.double()).unsqueeze(1)
    u, w = t[..., :half], t[..., half:ROPE]
    return torch.cat([u * c - w * s, u * s + w * c, t[..., ROPE:]], -1)


def _gqa_exact(i, q, gate, k_new, v_new, pos):
    """q, gate [B][T][24][256], k_new, v_new [B][T][4][256] raw; pos [B] of the first token.
    Returns out [B][T][24*256] and the caches with the new rows."""
    B, T = q.shape[:2]
    kc, vc = i["k_cache"].double(), i["v_cache"].double()
    out = torch.empty(B, T, NQ, GD, device=DEV, dtype=torch.float64)
    qw, kw = 1 + _d(i["q_norm_w"]), 1 + _d(i["k_norm_w"])
    for b in range(B):
        p0 = int(pos[b])
        at, n = torch.arange(p0, p0 + T, device=DEV), p0 + T
        qb, kb = _rope(_rms(q[b]) * qw, at), _rope(_rms(k_new[b]) * kw, at)
        ok = torch.arange(n, device=DEV).unsqueeze(0) <= at.unsqueeze(1)
        for h in range(NKV):
            kc[b, h, p0:n] = kb[:, h]
            vc[b, h, torch.div(at, 32, rounding_mode="floor"), :, at % 32] = v_new[b][:, h]
            V = vc[b, h].transpose(1, 2).reshape(-1, GD)[:n]
            for g in range(h * NQ // NKV, (h + 1) * NQ // NKV):
                s = (qb[:, g] @ kc[b, h, :n].t()) / math.sqrt(GD)
                out[b, :, g] = torch.softmax(s.masked_fill(~ok, float("-inf")), 1) @ V
    if gate is not None:
        out = out * torch.sigmoid(gate)
    return out.reshape(B, T, NQ * GD), kc, vc


def _gqa_layer_exact(i, x, pos):
    B, T = x.shape[:2]
    y = (_d(x).reshape(B * T, H) @ _d(i["w_qkv"]).t()).reshape(B, T, -1)
    qg, k, v = torch.split(y, [2 * NQ * GD, NKV * GD, NKV * GD], -1)
    qg = qg.reshape(B, T, NQ, 2 * GD)
    o, kc, vc = _gqa_exact(i, qg[..., :GD], qg[..., GD:], k.reshape(B, T, NKV, GD), v.reshape(B, T, NKV, GD), pos)
    return (o.reshape(B * T, -1) @ _d(i["w_o"]).t()).reshape(B, T, H), kc, vc


def exact(case, seed):
    """What run returns, from plain torch in 64 bits."""
    i, kind, B = _inputs(case, seed), case["kind"], case["B"]
    if kind == "dn_step":
        x = _d(i["x"]).unsqueeze(1) if case["conv"] else None
        qkv = None if case["conv"] else [i[n].unsqueeze(1) for n in "qkv"]
        o, S, cs, _, _ = _dn_exact(i, x, _d(i["a"]).unsqueeze(1), _d(i["b"]).unsqueeze(1), 1, case["conv"], False,
                                   qkv=qkv)
        return [t for t in (o[:, 0], S, cs) if t is not None]
    if kind == "gqa_step":
        qg = _d(i["qg"]).unsqueeze(1)
        o, kc, vc = _gqa_exact(i, qg[..., :GD], qg[..., GD:] if case["gate"] else None, _d(i["k_new"]).unsqueeze(1),
                               _d(i["v_new"]).unsqueeze(1), i["pos"])
        return [o.reshape(B, NQ, GD), kc, vc]
    if kind == "dn_layer":
        o, S, cs, _, _ = _dn_layer_exact(i, i["x"].unsqueeze(1))
        return [o[:, 0], S, cs]
    if kind == "gqa_layer":
        o, kc, vc = _gqa_layer_exact(i, i["x"].unsqueeze(1), i["pos"])
        return [o[:, 0], kc, vc]
    if kind == "decode_step":
        x = i["x"].unsqueeze(1)
        dn = [_dn_layer_exact(w, x) for w in i["dn"]]
        o, kc, vc = _gqa_layer_exact(i["gqa"], x, i["pos"])
        return [*(d[0][:, 0] for d in dn), o[:, 0], *(d[1] for d in dn), *(d[2] for d in dn), kc, vc]
    if kind in ("dn_verify", "dn_prompt"):
        o, S, cs, S_all, c_all = _dn_layer_exact(i, i["x"], every=kind == "dn_verify")
        return [o, S, cs] + ([torch.stack(S_all, 1), torch.stack(c_all, 1)] if kind == "dn_verify" else [])
    if kind == "gqa_prompt":
        return list(_gqa_layer_exact(i, i["x"], [case["pos0"]] * B))
    o, S, _, _, _ = _dn_exact(i, None, _d(i["a"]), _d(i["b"]), case["T"], False, False,
                              qkv=[i[n] for n in "qkv"])
    return [o, S]
