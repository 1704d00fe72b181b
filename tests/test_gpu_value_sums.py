"""The attention's value sums at the edges of the FP64 form (one fused
operation per term, values in [-2^51, 2^51), weights in [0, ONE] that add up
to at most ONE) and just outside it, where the general products take over,
against the oracle: decode attention (one block per head, and split over the
cache) and batched-prefill attention, head_dim 32, 64 and 128.
"""
import numpy as np
import pytest

import spec

pytestmark = pytest.mark.gpu
ONE = spec.ONE
EDGE = 1 << 51


def say(*a):
    print("[case]", *a, flush=True)


def values(kind, rng, n):
    v = (rng.standard_normal(n) * ONE).astype(np.int64)
    if kind == "low_edge":          # every sum at the lower bound
        v[:] = -EDGE
    elif kind == "high_edge":
        v[:] = EDGE - 1
    elif kind == "both_edges":
        v = rng.choice(np.array([-EDGE, EDGE - 1, -EDGE + 1, 0, -1], dtype=np.int64), n)
    elif kind == "one_out":         # a single value past the range
        v[n // 2] = EDGE
    elif kind == "one_out_low":
        v[n // 2] = -EDGE - 1
    elif kind == "wide":            # every value past the range, bits at both ends
        v = (rng.standard_normal(n) * 100 * ONE).astype(np.int64)
    elif kind == "full":
        v = rng.integers(spec.INT64_MIN, spec.INT64_MAX, size=n, dtype=np.int64, endpoint=True)
    return v


KINDS = ["low_edge", "high_edge", "both_edges", "one_out", "one_out_low", "wide", "full"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("nh,nkv,hd,positions", [
    (8, 2, 32, [0, 15, 200, 300]),
    (32, 4, 64, [17, 128, 255, 256, 700]),
    (6, 2, 128, [31, 130, 400]),
])
def test_decode_value_sums(ctx, oracle, nh, nkv, hd, positions, kind):
    rng = np.random.default_rng(nh + hd)
    max_seq, kvd = 704, nkv * hd
    kc = (rng.standard_normal(max_seq * kvd) * ONE).astype(np.int64)
    vc = values(kind, rng, max_seq * kvd)
    cos_t = np.empty(max_seq * hd // 2, dtype=np.int64)
    sin_t = np.empty_like(cos_t)
    oracle.q48o_rope_tables(cos_t.ctypes.data, sin_t.ctypes.data, hd, max_seq, 10000)
    ctx.rope_init(hd, max_seq, 10000)
    dk, dv = ctx.to_device(kc), ctx.to_device(vc)
    bufs = [dk, dv]
    try:
        for i, pos in enumerate(positions):
            # equal weights, and peaked ones
            q = (rng.standard_normal(nh * hd) * (0 if i == 1 else 3) * ONE).astype(np.int64)
            kn = (rng.standard_normal(kvd) * ONE).astype(np.int64)
            vn = values(kind, rng, kvd)
            qr, kr = q.copy(), kn.copy()
            for v, n in ((qr, nh), (kr, nkv)):
                for h in range(n):
                    oracle.q48o_rope_apply(cos_t.ctypes.data, sin_t.ctypes.data, hd // 2,
                                           v[h * hd:].ctypes.data, pos)
            want = np.empty(nh * hd, dtype=np.int64)
            oracle.q48o_attn_decode(want.ctypes.data, qr.ctypes.data, kc.ctypes.data,
                                    vc.ctypes.data, kr.ctypes.data, vn.ctypes.data, 0, pos, nh,
                                    nkv, hd, max_seq)
            dq, dkn, dvn = ctx.to_device(q), ctx.to_device(kn), ctx.to_device(vn)
            do = ctx.buffer(nh * hd)
            bufs += [dq, dkn, dvn, do]
            say("decode", nh, nkv, hd, "pos", pos, kind)
            ctx.attn_decode_rope(do.ptr, dq.ptr, dk.ptr, dv.ptr, dkn.ptr, dvn.ptr, 0, pos, nh,
                                 nkv, hd, max_seq)
            assert np.array_equal(do.download(), want), pos
            assert np.array_equal(dv.download(), vc)
        assert ctx.attn_status() == 0
    finally:
        for b in bufs:
            b.free()


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("nh,nkv,hd,p0,T", [(8, 2, 32, 20, 33), (8, 2, 64, 0, 90),
                                            (8, 4, 64, 63, 16), (3, 3, 128, 7, 50)])
def test_prefill_value_sums(ctx, oracle, nh, nkv, hd, p0, T, kind):
    rng = np.random.default_rng(nh + hd + T)
    max_seq, kvd, row = 160, nkv * hd, (nh + 2 * nkv) * hd
    kc = (rng.standard_normal(max_seq * kvd) * ONE).astype(np.int64)
    vc = values(kind, rng, max_seq * kvd)
    qkv = (rng.standard_normal(T * row) * 3 * ONE).astype(np.int64)
    qkv[:row] = 0                   # equal weights
    want = np.empty((T, nh * hd), dtype=np.int64)
    for t in range(T):
        at = slice((p0 + t) * kvd, (p0 + t + 1) * kvd)
        kn, vn = kc[at].copy(), vc[at].copy()
        q = qkv[t * row:t * row + nh * hd].copy()
        oracle.q48o_attn_decode(want[t].ctypes.data, q.ctypes.data, kc.ctypes.data,
                                vc.ctypes.data, kn.ctypes.data, vn.ctypes.data, 0, p0 + t, nh,
                                nkv, hd, max_seq)
    ctx.rope_init(hd, max_seq, 10000)
    dk, dv, dq = ctx.to_device(kc), ctx.to_device(vc), ctx.to_device(qkv)
    do = ctx.buffer(T * nh * hd)
    try:
        for mfma in (True, False):
            say("prefill", nh, nkv, hd, "p0", p0, "T", T, kind, "mfma", mfma)
            ctx.set_pf_attn_mfma(mfma)
            ctx.attn_prefill(do.ptr, dq.ptr, dk.ptr, dv.ptr, 0, p0, T, nh, nkv, hd, max_seq)
            assert np.array_equal(do.download().reshape(T, nh * hd), want), mfma
    finally:
        ctx.set_pf_attn_mfma(True)
        for b in (dk, dv, dq, do):
            b.free()
