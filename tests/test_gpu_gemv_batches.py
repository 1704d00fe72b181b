"""k_gemv_d's last batch of tiles: every number of tiles that can be left, against
the oracle; and that a row whose tiles do not fill its batches costs what its
weights do."""
import numpy as np
import pytest

import spec

pytestmark = pytest.mark.gpu
ONE = spec.ONE


@pytest.mark.parametrize("M", [2050, 40])       # one wave a row, several
def test_gemv_every_tile_count_vs_oracle(ctx, oracle, M):
    rng = np.random.default_rng(M)
    for tiles in list(range(1, 18)) + [23, 31]:
        for extra in (0, 1, 127):
            K = 128 * tiles + extra
            W = rng.integers(spec.INT64_MIN, spec.INT64_MAX, size=M * K, dtype=np.int64,
                             endpoint=True)
            x = rng.integers(spec.INT64_MIN, spec.INT64_MAX, size=K, dtype=np.int64, endpoint=True)
            want = np.empty(M, dtype=np.int64)
            oracle.q48o_gemv(want.ctypes.data, W.ctypes.data, x.ctypes.data, M, K)
            dW, dx, dy = ctx.to_device(W), ctx.to_device(x), ctx.buffer(M)
            print("[case] gemv tiles", M, K, flush=True)
            ctx.gemv(dy.ptr, dW.ptr, dx.ptr, M, K)
            assert np.array_equal(dy.download(), want), K
            for b in (dW, dx, dy):
                b.free()


def test_gemv_incomplete_batches_cost_their_tiles(ctx):
    """16384 x 700 (five tiles and a part) against 8192 x 2048 + 8 (sixteen and a
    part), a weight: 1.1 times; with whole batches of repeated tiles 1.4."""
    rng = np.random.default_rng(0)
    per = []
    for M, K in ((8192, 2056), (16384, 700)):
        W = ctx.to_device(rng.integers(-ONE, ONE, size=M * K, dtype=np.int64))
        x, y = ctx.to_device(rng.integers(-ONE, ONE, size=K, dtype=np.int64)), ctx.buffer(M)
        best = None
        for rep in range(6):
            n = 10 if rep == 0 else 100
            ctx.timer_start()
            for _ in range(n):
                ctx.gemv(y.ptr, W.ptr, x.ptr, M, K)
            t = ctx.timer_stop() / n
            best = t if best is None else min(best, t)
        per.append(best / (M * K))
        for b in (W, x, y):
            b.free()
    print("[case] gemv, ms a weight:", per, flush=True)
    assert per[1] < 1.25 * per[0], per
