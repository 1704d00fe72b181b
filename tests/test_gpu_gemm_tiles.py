"""The planes GEMM with row tiles of different magnitudes: each row tile of a
block of two has its own window of digit planes, so neither sends the other to
the 63-product form.  Results against the oracle; and the time, by which a
shared window shows."""
import numpy as np
import pytest

import intllm
import spec

pytestmark = pytest.mark.gpu
ONE = spec.ONE


def weights(rng, N, K):
    w = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    w = (w.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)   # bfloat16 values
    return (w.astype(np.float64) * ONE).astype(np.int64)


def scaled(kind, rng, W):
    """Row tile i of W changed by kind and i"""
    for i in range(0, (W.shape[0] + 63) // 64):
        rows = W[64 * i:64 * i + 64]
        if kind == "alternate":           # 24 bits apart, either tile the smaller
            rows >>= 24 if (i + i // 2) % 2 else 0
        elif kind == "every_plane":       # top planes 0 .. 6, neighbours apart
            rows >>= 8 * (5 * i % 7) if 5 * i % 7 < 6 else 0
            if 5 * i % 7 == 6:
                rows <<= 8
        elif kind == "one_out":           # one of a pair out of its window, the other low
            if i % 3 == 0:
                rows[rng.integers(0, len(rows)), rng.integers(0, W.shape[1])] = spec.INT64_MAX
            else:
                rows >>= 20
        elif kind == "low_digits":        # TOP - 4 in one tile's steps, not in the other's
            if i % 2:
                rows[::9, ::96] = 3
    return W


@pytest.mark.parametrize("kind", ["alternate", "every_plane", "one_out", "low_digits"])
@pytest.mark.parametrize("T,N,K", [(1024, 1090, 250), (1030, 1100, 160), (70, 1030, 416),
                                   (3, 200, 20000)])
def test_gemm_mixed_tiles_vs_oracle(ctx, oracle, T, N, K, kind):
    rng = np.random.default_rng(T + N + K)
    W = np.ascontiguousarray(scaled(kind, rng, weights(rng, N, K))).ravel()
    X = (rng.standard_normal(T * K) * ONE).astype(np.int64)
    want = np.empty(T * N, dtype=np.int64)
    oracle.q48o_gemm(want.ctypes.data, W.ctypes.data, X.ctypes.data, T, N, K)
    dW, dX, dY = ctx.to_device(W), ctx.to_device(X), ctx.buffer(T * N)
    Wp = intllm.Buffer(ctx, ctx.gemm_planes_bytes(N, K), 1)
    try:
        print("[case] gemm tiles", T, N, K, kind, flush=True)
        ctx.gemm(dY.ptr, dW.ptr, dX.ptr, T, N, K, intllm.GEMM_I8_PLANES)
        assert np.array_equal(dY.download(), want), "split in the call"
        ctx.zero(dY.ptr, T * N * 8)
        ctx.gemm_prepare(Wp.ptr, dW.ptr, N, K)
        ctx.gemm_prepared(dY.ptr, dW.ptr, Wp.ptr, dX.ptr, T, N, K)
        assert np.array_equal(dY.download(), want), "prepared"
    finally:
        for b in (dW, dX, dY, Wp):
            b.free()


def test_gemm_small_tiles_cost_no_more(ctx):
    """Row tiles 24 bits apart in turn, and weights that are all 2^-24 of the
    rest, take the time of equal ones of ordinary size: with one window for two
    tiles the first took 3.0 times as long, with windows that do not go below
    plane 4 they took 1.4 and 1.5 times."""
    T, N, K = 1024, 4096, 2048
    rng = np.random.default_rng(5)
    W = weights(rng, N, K)
    X = (rng.standard_normal(T * K) * ONE).astype(np.int64)
    dX, dY = ctx.to_device(X), ctx.buffer(T * N)
    Wp = intllm.Buffer(ctx, ctx.gemm_planes_bytes(N, K), 1)
    us = []
    for kind in ("equal", "alternate", "small"):
        w = W >> 24 if kind == "small" else scaled(kind, rng, W.copy())
        dW = ctx.to_device(np.ascontiguousarray(w).ravel())
        print("[case] gemm tiles, time", T, N, K, kind, flush=True)
        ctx.gemm_prepare(Wp.ptr, dW.ptr, N, K)
        best = None
        for rep in range(6):
            n = 5 if rep == 0 else 20
            ctx.timer_start()
            for _ in range(n):
                ctx.gemm_prepared(dY.ptr, dW.ptr, Wp.ptr, dX.ptr, T, N, K)
            t = ctx.timer_stop() / n
            best = t if best is None else min(best, t)
        us.append(best)
        dW.free()
    print("[case] equal, alternate, small:", us, flush=True)
    for b in (dX, dY, Wp):
        b.free()
    assert us[1] < 1.25 * us[0] and us[2] < 1.25 * us[0], us
