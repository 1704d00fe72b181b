"""q48_gemv at shapes that are not the decode kernel's (k_gemv_d: one to eight
waves per row, or four short rows per wave) and on rows that start on 8 bytes
(odd K, or W itself), and the fused GEMVs on odd K, against the oracle."""
import numpy as np
import pytest

import spec

pytestmark = pytest.mark.gpu


def full(rng, n):
    v = rng.integers(spec.INT64_MIN, spec.INT64_MAX, size=n, dtype=np.int64, endpoint=True)
    v[:: max(1, n // 5)] = spec.INT64_MIN
    return v


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("M,K", [
    (1, 1), (2, 1), (1, 129), (9, 127), (5, 128), (3, 12289), (17, 2049), (70, 3001),
    (520, 1027), (1031, 513), (2049, 257), (2100, 1100), (8193, 131), (8200, 510), (8192, 1),
])
def test_gemv_any_shape_vs_oracle(ctx, oracle, M, K, off):
    rng = np.random.default_rng(M * 7 + K)
    W, x = full(rng, M * K), full(rng, K)
    want = np.empty(M, dtype=np.int64)
    oracle.q48o_gemv(want.ctypes.data, W.ctypes.data, x.ctypes.data, M, K)
    dW = ctx.to_device(np.concatenate([np.zeros(off, np.int64), W]))
    dx = ctx.to_device(np.concatenate([np.zeros(off, np.int64), x]))
    dy = ctx.buffer(M)
    print("[case] gemv", M, K, "offset", off, flush=True)
    ctx.gemv(dy.ptr, dW.at(off), dx.at(off), M, K)
    assert np.array_equal(dy.download(), want)
    for b in (dW, dx, dy):
        b.free()


@pytest.mark.parametrize("M,K", [(40, 173), (256, 2049), (9, 1), (33, 5631)])
def test_residual_stats_odd_k_vs_oracle(ctx, oracle, M, K):
    """q48_gemv_residual_stats and q48_gemv_residual on odd K: the sums, the
    residual add and the partial sums of squares."""
    import intllm
    rng = np.random.default_rng(M + K)
    W, x, h = full(rng, M * K), full(rng, K), full(rng, M)
    want = np.empty(M, dtype=np.int64)
    oracle.q48o_gemv(want.ctypes.data, W.ctypes.data, x.ctypes.data, M, K)
    want = want + h                                   # int64, wrapping
    dW, dx = ctx.to_device(W), ctx.to_device(x)
    st = ctx.buffer(intllm.stats_words(M))
    for stats in (True, False):
        dh = ctx.to_device(h)
        print("[case] residual", M, K, "stats", stats, flush=True)
        if stats:
            ctx.gemv_residual_stats(dh.ptr, dW.ptr, dx.ptr, M, K, st.ptr)
            words = st.download().view(np.uint64)
            for b in range((M + 7) // 8):
                ss = sum(int(v) ** 2 for v in want[8 * b:8 * b + 8]) % (1 << 128)
                assert int(words[2 * b]) + (int(words[2 * b + 1]) << 64) == ss, b
        else:
            ctx.gemv_residual(dh.ptr, dW.ptr, dx.ptr, M, K)
        assert np.array_equal(dh.download(), want)
        dh.free()
    for b in (dW, dx, st):
        b.free()
