"""The fused GEMVs on rows that start on 8 bytes (odd K), where they change from
one launch to separate ones: the same words as the composition they name, on
both sides of every line; and no long unaligned projection that takes much
longer than its GEMV."""
import numpy as np
import pytest

import intllm
import spec

pytestmark = pytest.mark.gpu
ONE = spec.ONE


def stats_of(v):
    """Partial sums of squares, eight values a pair of words"""
    out = np.zeros(intllm.stats_words(len(v)), dtype=np.uint64)
    for b in range((len(v) + 7) // 8):
        ss = sum(int(e) ** 2 for e in v[8 * b:8 * b + 8]) % (1 << 128)
        out[2 * b], out[2 * b + 1] = ss & (2 ** 64 - 1), ss >> 64
    return out


# rows and K around 8192, 4096 and 2048 rows of K <= 1024, and 5 2^17, 5 2^18, 2^21,
# 2^22 and 2^23 weights of 1024 < K <= 2048, and past both
@pytest.mark.parametrize("M,K", [
    (2048, 33), (2050, 33), (4096, 65), (4098, 65), (8192, 129), (8194, 129), (100, 1023),
    (638, 1025), (640, 1025), (1278, 1025), (1280, 1025), (2046, 1025), (2048, 1025),
    (4090, 1025), (4094, 1025), (8182, 1025), (8186, 1025), (320, 2047), (322, 2047),
    (60, 2049), (300, 3001),
])
def test_fused_gemvs_are_their_compositions(ctx, M, K):
    rng = np.random.default_rng(M + K)
    hx = rng.integers(-2 * ONE, 2 * ONE, size=K, dtype=np.int64)
    W = ctx.to_device(rng.integers(-ONE // 8, ONE // 8, size=M * K, dtype=np.int64))
    x, nw = ctx.to_device(hx), ctx.to_device(rng.integers(-ONE, ONE, size=K, dtype=np.int64))
    h0 = rng.integers(-ONE, ONE, size=M, dtype=np.int64)
    xn, t, want, got = ctx.buffer(K), ctx.buffer(M), ctx.buffer(M), ctx.buffer(M)
    st, r, so = ctx.buffer(intllm.stats_words(K)), ctx.buffer(1), ctx.buffer(intllm.stats_words(M))
    bufs = [W, x, nw, xn, t, want, got, st, r, so]
    print("[case] gemv routes", M, K, flush=True)
    ctx.rms_stats(st.ptr, x.ptr, K)
    ctx.rms_inv(r.ptr, x.ptr, K)
    ctx.rmsnorm(xn.ptr, x.ptr, nw.ptr, K)
    ctx.gemv(t.ptr, W.ptr, xn.ptr, M, K)
    gold = t.download()
    for f, a in ((ctx.rmsnorm_gemv, ()), (ctx.norm_gemv, (r.ptr,)), (ctx.norm_gemv_stats, (st.ptr,))):
        f(got.ptr, W.ptr, x.ptr, nw.ptr, *a, M, K)
        assert np.array_equal(got.download(), gold), f.__name__
    F = M // 2
    ctx.silu_mul(want.ptr, t.ptr, t.at(F), F)
    for f, a in ((ctx.rmsnorm_gemv_swiglu, ()), (ctx.norm_gemv_swiglu, (r.ptr,)),
                 (ctx.norm_gemv_swiglu_stats, (st.ptr,))):
        f(got.ptr, W.ptr, x.ptr, nw.ptr, *a, F, K)
        assert np.array_equal(got.download(F), want.download(F)), f.__name__
    ctx.gemv(t.ptr, W.ptr, x.ptr, M, K)
    gold = t.download() + h0
    for f, a in ((ctx.gemv_residual, ()), (ctx.gemv_residual_stats, (so.ptr,)),
                 (ctx.gemv_residual_rms, (r.ptr,))):
        got.upload(h0)
        f(got.ptr, W.ptr, x.ptr, M, K, *a)
        assert np.array_equal(got.download(), gold), f.__name__
        if f == ctx.gemv_residual_stats:
            assert np.array_equal(so.download().view(np.uint64), stats_of(gold))
    ctx.rms_inv(st.ptr, got.ptr, M)
    assert r.download()[0] == st.download(1)[0]
    for b in bufs:
        b.free()


def test_long_unaligned_projection_costs_its_gemv(ctx):
    """Normed gate|up of 2 x 5631 rows of 2047: 1.2 times the plain GEMV (as one
    launch on unaligned rows 1.75 times)."""
    F, K = 5631, 2047
    rng = np.random.default_rng(1)
    W = ctx.to_device(rng.integers(-ONE, ONE, size=2 * F * K, dtype=np.int64))
    x, nw = (ctx.to_device(rng.integers(-ONE, ONE, size=K, dtype=np.int64)) for _ in range(2))
    y, st = ctx.buffer(2 * F), ctx.buffer(intllm.stats_words(K))
    ctx.rms_stats(st.ptr, x.ptr, K)
    us = []
    for f in (lambda: ctx.gemv(y.ptr, W.ptr, x.ptr, 2 * F, K),
              lambda: ctx.norm_gemv_swiglu_stats(y.ptr, W.ptr, x.ptr, nw.ptr, st.ptr, F, K)):
        best = None
        for rep in range(6):
            n = 10 if rep == 0 else 100
            ctx.timer_start()
            for _ in range(n):
                f()
            t = ctx.timer_stop() / n
            best = t if best is None else min(best, t)
        us.append(best)
    print("[case] plain, fused:", us, flush=True)
    for b in (W, x, nw, y, st):
        b.free()
    assert us[1] < 1.45 * us[0], us
