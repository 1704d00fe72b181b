"""q48_gemm's choice between the digit split inside the k loop and planes split
once per call: the same words from both and from the chosen one on either side
of the line, no shape that takes much longer than the other form, and the
other form when there is no workspace for the chosen one."""
import numpy as np
import pytest

import intllm
import spec

pytestmark = pytest.mark.gpu
ONE = spec.ONE


def operands(ctx, T, N, K):
    rng = np.random.default_rng(T + N + K)
    W = (rng.standard_normal(N * K) * 0.02).astype(np.float32)
    W = ((W.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32).astype(np.float64) * ONE)
    X = (rng.standard_normal(T * K) * ONE).astype(np.int64)
    W = W.astype(np.int64)
    return W, X, [ctx.to_device(W), ctx.to_device(X), ctx.buffer(T * N)]


@pytest.mark.parametrize("T,N,K", [
    (159, 2049, 257), (160, 2048, 320), (193, 1030, 1024), (256, 1024, 96), (300, 500, 2048),
    (1024, 130, 1000), (2048, 511, 130), (65, 4097, 512),
])
def test_forms_agree_vs_oracle(ctx, oracle, T, N, K):
    W, X, (dW, dX, dY) = operands(ctx, T, N, K)
    want = np.empty(T * N, dtype=np.int64)
    oracle.q48o_gemm(want.ctypes.data, W.ctypes.data, X.ctypes.data, T, N, K)
    for kernel in (None, intllm.GEMM_I8, intllm.GEMM_I8_FUSED, intllm.GEMM_I8_PLANES):
        print("[case] gemm choice", T, N, K, kernel, flush=True)
        ctx.zero(dY.ptr, T * N * 8)
        ctx.gemm(dY.ptr, dW.ptr, dX.ptr, T, N, K, kernel)
        assert np.array_equal(dY.download(), want), kernel
    for b in (dW, dX, dY):
        b.free()


@pytest.mark.parametrize("T,N,K", [(192, 5632, 2048), (2048, 512, 2048), (256, 1024, 1024),
                                   (128, 2560, 2048), (2048, 2048, 2048)])
def test_choice_is_not_the_slow_form(ctx, T, N, K):
    """Within 12% of the better form; the first three took 21 to 30% longer by a
    line at 256 tokens and 1024 rows."""
    _, _, (dW, dX, dY) = operands(ctx, T, N, K)
    us = {}
    for kernel in (None, intllm.GEMM_I8_FUSED, intllm.GEMM_I8_PLANES):
        print("[case] gemm choice, time", T, N, K, kernel, flush=True)
        for rep in range(6):
            n = 5 if rep == 0 else 30
            ctx.timer_start()
            for _ in range(n):
                ctx.gemm(dY.ptr, dW.ptr, dX.ptr, T, N, K, kernel)
            t = ctx.timer_stop() / n
            us[kernel] = t if rep == 0 else min(us[kernel], t)
    for b in (dW, dX, dY):
        b.free()
    print("[case] chosen, in the loop, planes:", us, flush=True)
    assert us[None] < 1.12 * min(us[intllm.GEMM_I8_FUSED], us[intllm.GEMM_I8_PLANES]), us


def test_other_form_where_the_workspace_cannot_grow(oracle):
    """In a capture the workspace keeps its size: a call whose chosen form needs
    more runs the other one (planes chosen here, 90 MB; the split in the loop
    needs the redo flags only)."""
    T, N, K = 1024, 2048, 2048
    c, lib = intllm.Context(0), intllm.hip_lib()
    W, X, (dW, dX, dY) = operands(c, T, N, K)
    want = np.empty(T * N, dtype=np.int64)
    oracle.q48o_gemm(want.ctypes.data, W.ctypes.data, X.ctypes.data, T, N, K)
    try:
        c.gemm(dY.ptr, dW.ptr, dX.ptr, 2, 64, 64)     # a workspace, of the least size
        print("[case] gemm choice in a capture", T, N, K, flush=True)
        intllm.check("q48_graph_begin", lib.q48_graph_begin(c.h))
        try:
            c.gemm(dY.ptr, dW.ptr, dX.ptr, T, N, K)
        finally:
            intllm.check("q48_graph_end", lib.q48_graph_end(c.h))
        for _ in range(3):
            c.zero(dY.ptr, T * N * 8)
            intllm.check("q48_graph_launch", lib.q48_graph_launch(c.h, 1))
            assert np.array_equal(dY.download(), want)
        intllm.check("q48_graph_drop", lib.q48_graph_drop(c.h))
    finally:
        for b in (dW, dX, dY):
            b.free()
        c.close()
