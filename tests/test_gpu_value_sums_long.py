"""The prefill attention's three value sums (values outside [-2^51, 2^51)) at
the longest rows it takes, where the sum of the weights' low parts comes
closest to its bound, against the oracle."""
import numpy as np
import pytest

import spec

pytestmark = pytest.mark.gpu
ONE = spec.ONE


@pytest.mark.parametrize("hd", [32, 64, 128])
def test_prefill_value_sums_at_the_longest_rows(ctx, oracle, hd):
    """Equal weights (a zero query) over 16288 to 16320 positions: p mod 2^24 is
    0.97 of 2^24 at 16289 and 0.96 at 16305; values at both ends of int64."""
    nh = nkv = 1
    p0, T, max_seq = 16287, 33, 16320
    rng = np.random.default_rng(hd)
    kc = (rng.standard_normal(max_seq * hd) * ONE).astype(np.int64)
    vc = rng.integers(spec.INT64_MIN, spec.INT64_MAX, size=(max_seq, hd), dtype=np.int64,
                      endpoint=True)
    vc[:, 0] = spec.INT64_MIN
    vc[:, 1] = spec.INT64_MAX
    vc[:, 2] = spec.INT64_MIN + rng.integers(0, 1 << 40, size=max_seq)
    vc = np.ascontiguousarray(vc).ravel()
    qkv = np.zeros(T * 3 * hd, dtype=np.int64)
    qkv[-3 * hd:] = (rng.standard_normal(3 * hd) * ONE).astype(np.int64)   # one peaked row
    want = np.empty((T, hd), dtype=np.int64)
    for t in range(T):
        at = slice((p0 + t) * hd, (p0 + t + 1) * hd)
        kn, vn = kc[at].copy(), vc[at].copy()
        q = qkv[t * 3 * hd:t * 3 * hd + hd].copy()
        oracle.q48o_attn_decode(want[t].ctypes.data, q.ctypes.data, kc.ctypes.data,
                                vc.ctypes.data, kn.ctypes.data, vn.ctypes.data, 0, p0 + t, nh,
                                nkv, hd, max_seq)
    ctx.rope_init(hd, max_seq, 10000)
    dk, dv, dq = ctx.to_device(kc), ctx.to_device(vc), ctx.to_device(qkv)
    do = ctx.buffer(T * hd)
    try:
        print("[case] prefill, long value sums", hd, p0, T, flush=True)
        ctx.attn_prefill(do.ptr, dq.ptr, dk.ptr, dv.ptr, 0, p0, T, nh, nkv, hd, max_seq)
        assert np.array_equal(do.download().reshape(T, hd), want)
    finally:
        for b in (dk, dv, dq, do):
            b.free()
