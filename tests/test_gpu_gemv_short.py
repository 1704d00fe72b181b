"""The fused GEMVs on short rows (int64 weights, K <= 512 and K <= 1024 staged
in one batch): lengths about the tiles, the segments and both limits, against
the oracle; and the block argmax's ties and extremes."""
import numpy as np
import pytest

import intllm
import spec

pytestmark = pytest.mark.gpu
ONE = spec.ONE


def full(rng, n):
    v = rng.integers(spec.INT64_MIN, spec.INT64_MAX, size=n, dtype=np.int64, endpoint=True)
    v[:: max(1, n // 5)] = spec.INT64_MIN
    return v


def gemv(oracle, W, x, M, K):
    y = np.empty(M, dtype=np.int64)
    oracle.q48o_gemv(y.ctypes.data, W.ctypes.data, x.ctypes.data, M, K)
    return y


@pytest.mark.parametrize("K", [1, 7, 16, 127, 128, 129, 256, 500, 511, 512, 513, 688, 1000, 1023,
                               1024, 1025, 1041])
def test_short_rows_vs_oracle(ctx, oracle, K):
    rng = np.random.default_rng(K)
    M, ffn = 43, 18
    W = full(rng, M * K)
    x = (rng.standard_normal(K) * 3 * ONE).astype(np.int64)
    w = (rng.standard_normal(K) * ONE).astype(np.int64)
    n = np.empty(K, dtype=np.int64)
    oracle.q48o_rmsnorm(n.ctypes.data, x.ctypes.data, w.ctypes.data, K)
    dW, dx, dw = ctx.to_device(W), ctx.to_device(x), ctx.to_device(w)
    ds, dt = ctx.buffer(intllm.stats_words(K)), ctx.buffer(intllm.stats_words(M))
    dy, do = ctx.buffer(M), ctx.buffer(ffn)
    ctx.rms_stats(ds.ptr, dx.ptr, K)

    print("[case] norm_gemv_stats", K, flush=True)
    ctx.norm_gemv_stats(dy.ptr, dW.ptr, dx.ptr, dw.ptr, ds.ptr, M, K)
    assert np.array_equal(dy.download(), gemv(oracle, W, n, M, K))

    print("[case] norm_gemv_swiglu_stats", K, flush=True)
    t = gemv(oracle, W, n, 2 * ffn, K)
    g, u = t[:ffn].copy(), t[ffn:].copy()
    want = np.empty(ffn, dtype=np.int64)
    oracle.q48o_silu_mul(want.ctypes.data, g.ctypes.data, u.ctypes.data, ffn)
    ctx.norm_gemv_swiglu_stats(do.ptr, dW.ptr, dx.ptr, dw.ptr, ds.ptr, ffn, K)
    assert np.array_equal(do.download(), want)

    print("[case] residual_stats", K, flush=True)
    h, xf = full(rng, M), full(rng, K)
    dh, dxf = ctx.to_device(h), ctx.to_device(xf)
    ctx.gemv_residual_stats(dh.ptr, dW.ptr, dxf.ptr, M, K, dt.ptr)
    want = gemv(oracle, W, xf, M, K) + h              # int64, wrapping
    assert np.array_equal(dh.download(), want)
    words = dt.download().view(np.uint64)
    for b in range((M + 7) // 8):
        ss = sum(int(v) ** 2 for v in want[8 * b:8 * b + 8]) % (1 << 128)
        assert int(words[2 * b]) + (int(words[2 * b + 1]) << 64) == ss, b
    for b in (dW, dx, dw, ds, dt, dy, do, dh, dxf):
        b.free()


@pytest.mark.parametrize("n", [1, 63, 64, 1024, 1025, 32767, 32769])
def test_argmax_first_of_equals(ctx, n):
    rng = np.random.default_rng(n)
    for v in (np.full(n, spec.INT64_MIN, dtype=np.int64),
              np.full(n, spec.INT64_MAX, dtype=np.int64),
              rng.integers(-2, 2, size=n, dtype=np.int64),
              np.arange(n, dtype=np.int64), -np.arange(n, dtype=np.int64)):
        dv = ctx.to_device(v)
        print("[case] argmax", n, flush=True)
        assert ctx.argmax(dv.ptr, n) == int(np.argmax(v))
        dv.free()
