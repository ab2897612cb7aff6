"""GPU tests of the token-tile projections (batches and prompts of more
vectors than the operand groups of one pass hold), of the projections that
read fp32 rows, and of the checkpointed multi-step recurrence: all keep the
sums of the single-vector, single-step calls, so every comparison is bit for
bit.

Sizes: a small layer (hidden 160: fewer k-steps than the eight classes of the
sum; 161 row blocks: no multiple of any workgroup's; 16 value heads where the
segments of the input projection need them), batches at the edges of
16-vector blocks, 64-vector tiles and of both layouts' ranges, windows at the
edges of the recurrence's 8-token blocks."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HID, NQK, NV = 160, 2, 8


def channels(nv):
    return (2 * NQK + nv) * 128


@pytest.fixture(scope="module")
def ctx():
    from vx27_amd import lib as L
    c = L.Ctx(0)
    yield c
    c.close()


def weights(ctx, r, conv_bf16=True, NV=NV):
    from vx27_amd import workloads as W
    bf = lambda shape, std: W.bf16_bits(W.normal(r, shape, std))
    CH = channels(NV)
    cw = W.normal(r, (CH, 4), 0.2)
    host = {"A_log": W.normal(r, NV, 0.5), "dt_bias": W.normal(r, NV, 0.1), "norm_w": 1 + W.normal(r, 128, 0.1),
            "conv_w": W.bf16_bits(cw) if conv_bf16 else cw}
    dev = {k: ctx.put(v) for k, v in host.items()}
    dev["w_in"] = ctx.put_tiled(bf((CH + NV * 128 + 2 * NV, HID), 0.1))
    dev["w_out"] = ctx.put_tiled(bf((HID, NV * 128), 0.03))
    dev["dt"], dev["nv"] = 1 if conv_bf16 else 0, NV
    return dev


def pack(ctx, xb, B):
    """vx27_hip_pack_x of the B vectors at xb, in a buffer of vx27_hip_pack_bytes."""
    from vx27_amd import lib as L
    pk = ctx.buf(L.lib().vx27_hip_pack_bytes(HID, B))
    L.check(L.lib().vx27_hip_pack_x(ctx.h, xb.ptr, B, HID, pk.ptr), "pack_x")
    return pk


def decode(ctx, dev, x, S, conv, skew=0, xskew=0, in_place=False, packed=False):
    """One layer step of x [B][HID]; the conv state `skew` and x `xskew` floats off their buffers' starts; in_place: out
    is x; packed: x comes packed (the fp32 rows it was packed from hold something else)."""
    from vx27_amd import lib as L
    B = x.shape[0]
    cs = np.concatenate([np.zeros(skew, np.float32), conv.ravel()])
    xs = np.concatenate([np.zeros(xskew, np.float32), x.ravel()])
    Sd, cd, xb, ob = ctx.put(S), ctx.put(cs), ctx.put(xs), ctx.buf(B * HID * 4)
    op = xb if in_place else ob
    pk = pack(ctx, xb, B) if packed else None
    if packed:
        xb.upload(np.zeros_like(xs))
    d = L.DnLayerDesc(B, NQK, dev["nv"], 128, HID, xb.ptr + 4 * xskew, pk and pk.ptr, dev["w_in"].ptr, dev["w_out"].ptr, dev["conv_w"].ptr,
                      dev["dt"], dev["A_log"].ptr, dev["dt_bias"].ptr, dev["norm_w"].ptr, Sd.ptr, cd.ptr + 4 * skew,
                      op.ptr)
    L.check(L.lib().vx27_hip_dn_layer_decode(ctx.h, C.byref(d)), "dn_layer")
    res = (op.download((B, HID), np.float32), Sd.download(S.shape, np.float32),
           cd.download(cs.shape, np.float32)[skew:].reshape(conv.shape))
    for b in (Sd, cd, xb, ob) + ((pk,) if packed else ()):
        b.free()
    return res


def inputs(r, B, NV=NV):
    from vx27_amd import workloads as W
    return W.normal(r, (B, HID)), W.normal(r, (B, NV, 128, 128), 0.02), W.normal(r, (B, channels(NV), 3), 0.5)


@pytest.mark.parametrize("B,conv_bf16,skew", [(35, True, 0), (36, True, 0), (48, False, 0), (49, True, 1), (64, True, 0),
                                              (65, False, 1), (66, True, 0), (131, True, 0)])
def test_decode_batch_bits(ctx, B, conv_bf16, skew):
    """A batch gives the bits of its sequences one by one (outputs, states and
    conv states; unaligned conv states too)."""
    from vx27_amd import workloads as W
    r = W.rng(31, f"tok_decode_{B}")
    dev = weights(ctx, r, conv_bf16)
    x, S, conv = inputs(r, B)
    got = decode(ctx, dev, x, S, conv, skew)
    for b in sorted({0, 1, 15, 16, 33, 34, B // 2, B - 2, B - 1}):
        one = decode(ctx, dev, x[b:b + 1], S[b:b + 1], conv[b:b + 1])
        for g, o, n in zip(got, one, ("out", "S", "conv")):
            assert np.array_equal(g[b], o[0]), (n, b)


@pytest.mark.parametrize("B", [1, 2, 5, 6, 40])
def test_rows_or_packed_bits(ctx, B):
    """Up to 5 vectors are read as fp32 rows, or packed (unaligned rows, rows
    that the output overwrites): the same bits."""
    from vx27_amd import workloads as W
    r = W.rng(34, f"rows_{B}")
    dev = weights(ctx, r)
    x, S, conv = inputs(r, B)
    for kw in ({"xskew": 1}, {"in_place": True}):
        for a, b in zip(decode(ctx, dev, x, S, conv), decode(ctx, dev, x, S, conv, **kw)):
            assert np.array_equal(a, b), kw


@pytest.mark.parametrize("B,T", [(1, 1), (3, 2), (1, 8), (2, 9), (1, 17), (5, 7), (1, 36), (2, 33), (1, 70)])
def test_checkpoint_window_bits(ctx, B, T):
    """A window with checkpoints gives the bits of T decode calls."""
    window_bits(ctx, B, T, NV)


@pytest.mark.parametrize("B,T", [(1, 1), (2, 2), (1, 5), (3, 2), (1, 35), (1, 36), (1, 66), (2, 65)])
def test_checkpoint_window_segment_bits(ctx, B, T):
    """The same with 16 value heads: the input projection stores q|k|v, z, a and
    b as four segments, from fp32 rows (up to 5 of them), operand groups and
    token tiles (8 heads go through one matrix and copies)."""
    window_bits(ctx, B, T, 16)


@pytest.mark.parametrize("B", [5, 35, 36, 65, 66])
def test_packed_input_bits(ctx, B):
    """x handed over packed gives the bits of the rows, in either layout."""
    from vx27_amd import lib as L, workloads as W
    r = W.rng(35, f"packed_{B}")
    dev = weights(ctx, r)
    x, S, conv = inputs(r, B)
    for a, b in zip(decode(ctx, dev, x, S, conv), decode(ctx, dev, x, S, conv, packed=True)):
        assert np.array_equal(a, b)
    bf = lambda shape, std: W.bf16_bits(W.normal(r, shape, std))
    wq, wo = ctx.put_tiled(bf((24 * 512 + 2048, HID), 0.1)), ctx.put_tiled(bf((HID, 24 * 256), 0.03))
    qn, kn = ctx.put(W.normal(r, 256, 0.1)), ctx.put(W.normal(r, 256, 0.1))
    pos = ctx.put((np.arange(B) % 60).astype(np.int32))
    kv = bf((B * 4 * 64 * 256,), 1.0)
    got = []
    for packed in (False, True):
        xb, ob, kc, vc = ctx.put(x), ctx.buf(x.nbytes), ctx.put(kv), ctx.put(kv)
        pk = pack(ctx, xb, B) if packed else None
        if packed:
            xb.upload(np.zeros_like(x))
        d = L.GqaLayerDesc(B, 24, 4, 256, HID, 64, 1e7, 1.0, 64, xb.ptr, pk and pk.ptr, wq.ptr, wo.ptr, qn.ptr, kn.ptr,
                           pos.ptr, kc.ptr, vc.ptr, ob.ptr, 0)
        L.check(L.lib().vx27_hip_gqa_layer_decode(ctx.h, C.byref(d)), "gqa_layer")
        got.append((ob.download(x.shape, np.float32), kc.download(kv.shape, np.uint16), vc.download(kv.shape, np.uint16)))
        for b in (xb, ob, kc, vc) + ((pk,) if packed else ()):
            b.free()
    for a, b in zip(*got):
        assert np.array_equal(a, b)


def window_bits(ctx, B, T, NV):
    from vx27_amd import lib as L, workloads as W
    r = W.rng(32, f"tok_window_{B}_{T}")
    dev = weights(ctx, r, NV=NV)
    _, S, conv = inputs(r, B, NV)
    x = W.normal(r, (B, T, HID))
    Sd, cd, xb, ob = ctx.put(S), ctx.put(conv), ctx.put(x), ctx.buf(B * T * HID * 4)
    sk, ck = ctx.buf(T * S.nbytes), ctx.buf(T * conv.nbytes)
    d = L.DnLayerPrefillDesc(B, T, NQK, NV, 128, HID, 0, xb.ptr, dev["w_in"].ptr, dev["w_out"].ptr, dev["conv_w"].ptr,
                             dev["dt"], dev["A_log"].ptr, dev["dt_bias"].ptr, dev["norm_w"].ptr, Sd.ptr, cd.ptr,
                             ob.ptr)
    d.S_ckpt, d.conv_ckpt = sk.ptr, ck.ptr
    L.check(L.lib().vx27_hip_dn_layer_prefill(ctx.h, C.byref(d)), "dn_layer_prefill")
    out = ob.download((B, T, HID), np.float32)
    S_all, c_all = sk.download((B, T) + S.shape[1:], np.float32), ck.download((B, T) + conv.shape[1:], np.float32)
    for t in range(T):
        o, S, conv = decode(ctx, dev, np.ascontiguousarray(x[:, t]), S, conv)
        assert np.array_equal(out[:, t], o) and np.array_equal(S_all[:, t], S) and np.array_equal(c_all[:, t], conv), t
    assert np.array_equal(Sd.download(S.shape, np.float32), S)
    assert np.array_equal(cd.download(conv.shape, np.float32), conv)
    for b in (Sd, cd, xb, ob, sk, ck):
        b.free()


@pytest.mark.parametrize("T", [36, 66, 255])
def test_gqa_prompt_cache_bits(ctx, T):
    """The cache rows of a prompt in one call and in single-token calls (bf16
    segments of the token tiles and of the operand groups)."""
    from vx27_amd import lib as L, workloads as W
    r = W.rng(33, f"tok_gqa_{T}")
    bf = lambda shape, std: W.bf16_bits(W.normal(r, shape, std))
    wq, wo = ctx.put_tiled(bf((24 * 512 + 2048, HID), 0.1)), ctx.put_tiled(bf((HID, 24 * 256), 0.03))
    qn, kn = ctx.put(W.normal(r, 256, 0.1)), ctx.put(W.normal(r, 256, 0.1))
    x = W.normal(r, (T, HID))

    def run(chunks):
        kc, vc = ctx.put(np.zeros((4, 256, 256), np.uint16)), ctx.put(np.zeros((4, 8, 256, 32), np.uint16))
        for p0, n in chunks:
            xb, ob = ctx.put(np.ascontiguousarray(x[p0:p0 + n])), ctx.buf(n * HID * 4)
            d = L.GqaLayerPrefillDesc(1, n, 24, 4, 256, HID, 64, 1e7, 1.0, 256, p0, 0, xb.ptr, wq.ptr, wo.ptr, qn.ptr,
                                      kn.ptr, kc.ptr, vc.ptr, ob.ptr)
            L.check(L.lib().vx27_hip_gqa_layer_prefill(ctx.h, C.byref(d)), "gqa_layer_prefill")
            o = ob.download((n, HID), np.float32)
            xb.free(), ob.free()
        res = kc.download((4, 256, 256), np.uint16), vc.download((4, 8, 256, 32), np.uint16), o
        kc.free(), vc.free()
        return res

    kc, vc, _ = run([(0, T)])
    k1, v1, _ = run([(p, 1) for p in range(0, T)] if T < 100 else [(p, min(33, T - p)) for p in range(0, T, 33)])
    assert np.array_equal(kc, k1) and np.array_equal(vc, v1)
