"""mi355x_gemv_batched with a few Q4_0 activations on the matrix cores (one
launch, activations as two f16 planes) on the GPU against the CPU oracle and 64 bits:
sizes around the 16-row tiles, the 4-block quads of a wavefront and the
8192 values of a launch, strides and unaligned rows, more than one pass, the
allocation-free form, and rows of very different scales."""
import numpy as np
import pytest

import mi355x
import synth
from test_gemm_batched_gpu import check, run, weights
from tolerance import F32_SUM

pytestmark = pytest.mark.gpu

# (N, K, M): one tile or less, ragged last tiles, more tiles than workgroups,
# wavefronts with no, one and eight quads and a partial last one, block columns
# of 64 with and without a remainder, two launches (K > 8192), two passes (M > 8)
SIZES = [(1, 256, 2), (15, 512, 3), (17, 1024, 5), (33, 1280, 4), (100, 2304, 8), (16 * 600 + 5, 256, 6),
         (300, 4096, 7), (4097, 5120, 2), (4100, 6144, 4), (4099, 8192, 8), (16387, 8448, 5), (50, 2048, 9)]


def some_rows(N):
    return np.unique(np.concatenate([np.arange(min(N, 48)), np.arange(max(0, N - 48), N)]))


@pytest.mark.parametrize("N,K,M", SIZES)
def test_few_activations_match_oracle(ctx, oracle, N, K, M):
    raw = weights(2, N, K, N + K)
    xs = np.stack([synth.activations(K, seed=100 + m) for m in range(M)])
    y = run(ctx, 2, raw, N, K, xs)
    rows = some_rows(N)
    check(oracle, 2, raw.reshape(N, -1)[rows], len(rows), K, xs, y[:, rows], f"{N}x{K} M={M}", bound=F32_SUM)
    # an activation's result does not depend on the others
    assert np.array_equal(run(ctx, 2, raw, N, K, xs[::-1].copy())[::-1], y)


def test_few_activations_strides_and_noalloc(ctx):
    N, K, M = 4101, 5120, 6
    raw = weights(2, N, K, 8)
    xs = np.stack([synth.activations(K, seed=200 + m) for m in range(M)])
    w = ctx.resident(2, raw, N, K)
    try:
        ref = ctx.gemv_batched(w, xs)
        for xst, yst in ((K + 1, N + 3), (K + 64, N)):
            assert np.array_equal(ctx.gemv_batched(w, xs, x_stride=xst, y_stride=yst), ref), (xst, yst)
        xb, yb = ctx.to_device(xs), ctx.alloc(4 * M * N)
        try:
            mi355x.check(ctx.lib.mi355x_gemv_batched_noalloc(ctx.h, 2, w.ptr, N, K, xb.ptr, K, yb.ptr, N, M))
            ctx.sync()
            assert np.array_equal(yb.download(np.float32, M * N).reshape(M, N), ref)
        finally:
            xb.free()
            yb.free()
    finally:
        w.free()


def test_few_activations_scales(ctx, oracle):
    """Rows of 1e-30 to 1e30 beside each other, a zero row, and one whose parts differ by 2^20."""
    N, K = 40, 4096
    raw = weights(2, N, K, 3)
    x = synth.activations(K, seed=5)
    step = np.where(np.arange(K) < K // 2, 2.0 ** -20, 1.0).astype(np.float32)
    xs = np.stack([x * np.float32(1e-30), x, x * np.float32(1e30), np.zeros_like(x), x * step])
    y = run(ctx, 2, raw, N, K, xs)
    check(oracle, 2, raw, N, K, xs, y, "scales", bound=F32_SUM)
    assert not y[3].any()
    # the small part on its own: the weights of the other are 0
    small = raw.reshape(N, K // 32, 18).copy()
    small[:, K // 64:, :2] = 0
    alone = np.where(np.arange(K) < K // 2, xs[4:], 0.0)
    check(oracle, 2, small.reshape(N, -1), N, K, alone, run(ctx, 2, small.reshape(N, -1), N, K, xs)[4:], "small part",
          bound=F32_SUM)
