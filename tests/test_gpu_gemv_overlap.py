"""GEMVs whose output shares words with the vectors they read: the result is
that of the same call on separate buffers.  The fused calls go through a
temporary then (a fused launch writes rows while other blocks read), the plain
one runs as a single block where its rows fit one."""
import numpy as np
import pytest

import intllm
import spec

pytestmark = pytest.mark.gpu

ONE = 1 << 48


def vec(rng, n):
    return rng.integers(-4 * ONE, 4 * ONE, size=n, dtype=np.int64)


# rows and row length: odd K, more rows than a block has, both around a segment
SHAPES = [(40, 173), (173, 173), (300, 1031), (1031, 2047), (64, 256), (9, 33)]
CALLS = ["rmsnorm_gemv", "gemv_residual", "rmsnorm_gemv_swiglu", "norm_gemv", "norm_gemv_swiglu",
         "gemv_residual_rms", "norm_gemv_stats", "norm_gemv_swiglu_stats", "gemv_residual_stats"]


@pytest.mark.parametrize("call", CALLS)
@pytest.mark.parametrize("M,K", SHAPES)
def test_fused_gemv_over_its_input(ctx, call, M, K):
    rng = np.random.default_rng(M + 31 * K + len(call))
    swiglu, residual = "swiglu" in call, "residual" in call
    W = ctx.to_device(vec(rng, (2 * M if swiglu else M) * K) >> 6)
    x, nw = vec(rng, K), ctx.to_device(vec(rng, K))
    sx, so = ctx.buffer(intllm.stats_words(K)), ctx.buffer(intllm.stats_words(M))

    def one(out, px):
        if residual:
            extra = {"gemv_residual": (), "gemv_residual_rms": (so.ptr,),
                     "gemv_residual_stats": (so.ptr,)}[call]
            getattr(ctx, call)(out, W.ptr, px, M, K, *extra)
        elif call.startswith("rmsnorm"):
            getattr(ctx, call)(out, W.ptr, px, nw.ptr, M, K)
        else:
            (ctx.rms_stats if "stats" in call else ctx.rms_inv)(sx.ptr, px, K)
            getattr(ctx, call)(out, W.ptr, px, nw.ptr, sx.ptr, M, K)

    # the output on x's words, and on its tail and what follows
    for at in (0, K - min(K, M) // 2):
        n = max(K, at + M)
        words = np.concatenate([x, vec(rng, n - K)])
        joint, apart = ctx.to_device(words), ctx.to_device(words)
        dx = ctx.to_device(x)
        print("[case]", call, M, K, "output at", at, flush=True)
        one(apart.at(at), dx.ptr)
        one(joint.at(at), joint.ptr)
        want, got = apart.download(), joint.download()
        assert np.array_equal(got[at:at + M], want[at:at + M])
        assert np.array_equal(got[:at], x[:at])
        for b in (joint, apart, dx):
            b.free()
    for b in (W, nw, sx, so):
        b.free()


@pytest.mark.parametrize("M,K", [(1, 9), (4, 1031), (8, 2047), (8, 2048), (8, 5632), (5, 8191)])
def test_plain_gemv_over_its_input(ctx, M, K):
    rng = np.random.default_rng(M + 31 * K)
    x = vec(rng, K)
    W, dx, y = ctx.to_device(vec(rng, M * K)), ctx.to_device(x), ctx.buffer(M)
    print("[case] gemv", M, K, flush=True)
    ctx.gemv(y.ptr, W.ptr, dx.ptr, M, K)
    want = y.download()
    ctx.gemv(dx.ptr, W.ptr, dx.ptr, M, K)
    got = dx.download()
    assert np.array_equal(got[:M], want)
    assert np.array_equal(got[M:], x[M:])
    for b in (W, dx, y):
        b.free()
