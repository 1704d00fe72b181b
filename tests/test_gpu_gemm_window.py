"""The planes GEMM (k_gemm_i8p) where its window, its shifted weight planes and
its blocks of one or two row tiles can go wrong, against the oracle: row tiles
whose planes need a fourth or fifth plane in a few steps, magnitudes at a
plane's edge, digits out of the window in one tile of a pair, k loops of every
remainder of four, empty K splits, and an odd number of row tiles.  With the
weights split in the call and prepared.
"""
import numpy as np
import pytest

import spec

ONE = spec.ONE


def weights(kind, rng, N, K):
    w = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    w = (w.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)   # bfloat16 values
    w = (w.astype(np.float64) * ONE).astype(np.int64)
    if kind == "low_digits":        # TOP - 3, TOP - 4 in scattered steps
        for d, every in ((1 << 20, 7), (1 << 12, 11), (3, 13)):
            w[::5, ::every * 32] = d + rng.integers(0, 7)
    elif kind == "edges":           # largest magnitudes on both sides of a plane's limit
        lim = sum(127 << (8 * i) for i in range(6))
        for r, v in enumerate((lim, lim + 1, -lim, -lim - 1, (1 << 47) - 1, -(1 << 47),
                               lim >> 1, (lim >> 1) + 1, 1, -1)):
            w[(r * 67) % N, (r * 31) % K] = v
    elif kind == "tiny":            # planes 0 and 1 only, an all-zero row tile
        w = rng.integers(-300, 300, size=(N, K)).astype(np.int64)
        w[64:128] = 0
    elif kind == "one_full":        # one tile of a pair leaves the window
        w[min(70, N - 2), K // 2] = spec.INT64_MIN
        w[min(200, N - 1), K - 1] = spec.INT64_MAX
    return w


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["bf16", "low_digits", "edges", "tiny", "one_full"])
@pytest.mark.parametrize("T,N,K", [
    (1024, 1088, 33),     # two row tiles a block, the last block one; 2 k-steps
    (1030, 1100, 160),    # ragged tokens and rows; 5 k-steps
    (1024, 1090, 250),    # 8 k-steps, the last ragged
    (70, 1030, 416),      # one row tile, 13 k-steps
    (3, 70, 20000),       # K past one run: splits, the last ones empty
])
def test_gemm_window_vs_oracle(ctx, oracle, T, N, K, kind):
    import intllm
    rng = np.random.default_rng(T + N + K)
    W = np.ascontiguousarray(weights(kind, rng, N, K)).ravel()
    X = (rng.standard_normal(T * K) * ONE).astype(np.int64)
    want = np.empty(T * N, dtype=np.int64)
    oracle.q48o_gemm(want.ctypes.data, W.ctypes.data, X.ctypes.data, T, N, K)
    dW, dX, dY = ctx.to_device(W), ctx.to_device(X), ctx.buffer(T * N)
    Wp = intllm.Buffer(ctx, ctx.gemm_planes_bytes(N, K), 1)
    try:
        print("[case] gemm window", T, N, K, kind, flush=True)
        ctx.gemm(dY.ptr, dW.ptr, dX.ptr, T, N, K, intllm.GEMM_I8_PLANES)
        assert np.array_equal(dY.download(), want), "split in the call"
        ctx.zero(dY.ptr, T * N * 8)
        ctx.gemm_prepare(Wp.ptr, dW.ptr, N, K)
        ctx.gemm_prepared(dY.ptr, dW.ptr, Wp.ptr, dX.ptr, T, N, K)
        assert np.array_equal(dY.download(), want), "prepared"
    finally:
        for b in (dW, dX, dY, Wp):
            b.free()


def test_block_numbering():
    """tile_of and its inverse block_of (csrc/q48_gemm.hip), restated."""
    def tile_of(b, nn, nt):
        q, r = divmod(nn * nt, 8)
        x, l = b % 8, b // 8
        pid = x * (q + 1) + l if x < r else r * (q + 1) + (x - r) * q + l
        first = pid // (8 * nt) * 8
        gs, i = min(nn - first, 8), pid - first * nt
        return first + i % gs, i // gs

    def block_of(n, t, nn, nt):
        q, r = divmod(nn * nt, 8)
        first = n // 8 * 8
        pid = first * nt + t * min(nn - first, 8) + n - first
        if pid < r * (q + 1):
            return 8 * (pid % (q + 1)) + pid // (q + 1)
        pid -= r * (q + 1)
        return 8 * (pid % max(q, 1)) + r + pid // max(q, 1)

    for nn in range(1, 30):
        for nt in range(1, 12):
            assert all(block_of(*tile_of(b, nn, nt), nn, nt) == b for b in range(nn * nt))


@pytest.mark.gpu
def test_gemm_long_k_vs_oracle(oracle):
    """A row tile of more than 4 GB of digit planes: its zero planes, which fill
    up a split's last group of four k-steps, are past a 32-bit offset from the
    first splits, whose lengths are therefore multiples of four."""
    import intllm
    T, N, K = 2, 3, 32 * (262144 + 601) - 5
    rng = np.random.default_rng(11)
    W = np.ascontiguousarray(weights("bf16", rng, N, K)).ravel()
    X = (rng.standard_normal(T * K) * ONE).astype(np.int64)
    want = np.empty(T * N, dtype=np.int64)
    oracle.q48o_gemm(want.ctypes.data, W.ctypes.data, X.ctypes.data, T, N, K)
    ctx = intllm.Context(0)   # its own: 9 GB of workspace go with it
    dW, dX, dY = ctx.to_device(W), ctx.to_device(X), ctx.buffer(T * N)
    try:
        print("[case] gemm long k", T, N, K, flush=True)
        ctx.gemm(dY.ptr, dW.ptr, dX.ptr, T, N, K, intllm.GEMM_I8_PLANES)
        assert np.array_equal(dY.download(), want)
    finally:
        for b in (dW, dX, dY):
            b.free()
        ctx.close()
