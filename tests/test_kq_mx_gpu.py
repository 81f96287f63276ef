"""mi355x_gemv_batched with a few activations of a K/IQ type (one launch, digit
arithmetic on the integer matrix cores) on the GPU against the CPU oracle:
sizes around the 16-row tiles, the 8-superblock groups and the registers of a
wavefront, as many activations as the LDS holds, strides, unaligned rows, the
allocation-free form, and each activation's independence of the others."""
import numpy as np
import pytest

import mi355x
import synth
from test_gemm_batched_gpu import TYPES, check, install_grids, run, weights  # noqa: F401 (fixture)
from tolerance import DIGIT_SUM

pytestmark = pytest.mark.gpu

KQ = {n: t for n, t in TYPES.items() if t != 2}

# (N, K, M): ragged and single rows, one superblock to 64 (odd: rows that start
# 2 mod 4; a partial group), units of one to eight steps per wavefront, more
# tiles than workgroups hold sums for (16 x 512 rows and up)
SIZES = [(1, 256, 2), (15, 512, 3), (17, 1792, 4), (33, 2048, 5), (100, 2304, 8), (300, 4096, 6), (70, 8448, 4),
         (40, 16384, 3), (16 * 512 * 4 + 5, 256, 8), (16 * 512 * 9 + 19, 256, 3), (4100, 1024, 7)]


@pytest.mark.parametrize("name", list(KQ))
@pytest.mark.parametrize("N,K,M", SIZES)
def test_few_activations_match_oracle(ctx, oracle, name, N, K, M):
    t = KQ[name]
    raw = weights(t, N, K, N + K)
    xs = np.stack([synth.activations(K, seed=100 + m) for m in range(M)])
    ctx.set_option(mi355x.OPT_VARIANT, mi355x.VARIANT_DIGITS)  # AUTO leaves small codebook matrices to the f32 rows
    try:
        y = run(ctx, t, raw, N, K, xs)
        one = run(ctx, t, raw, N, K, np.stack([xs[M - 1], xs[0]]))
    finally:
        ctx.set_option(mi355x.OPT_VARIANT, mi355x.VARIANT_AUTO)
    rows = np.unique(np.concatenate([np.arange(min(N, 64)), np.arange(max(0, N - 64), N)]))
    sub = raw.reshape(N, -1)[rows]
    check(oracle, t, sub, len(rows), K, xs, y[:, rows], f"{name} {N}x{K} M={M}", bound=DIGIT_SUM)
    if (t not in (14, 11, 18, 21, 22) or K <= 8192) and (t != 22 or K <= 4096):  # else two one-row launches
        assert np.array_equal(one, y[[M - 1, 0]])


@pytest.mark.parametrize("name", list(KQ))
def test_few_activations_strides_and_noalloc(ctx, name):
    t, N, K, M = KQ[name], 4101, 4096, 5
    raw = weights(t, N, K, 8)
    xs = np.stack([synth.activations(K, seed=200 + m) for m in range(M)])
    w = ctx.resident(t, raw, N, K)
    try:
        ref = ctx.gemv_batched(w, xs)
        for xst, yst in ((K + 1, N + 3), (K + 64, N)):
            assert np.array_equal(ctx.gemv_batched(w, xs, x_stride=xst, y_stride=yst), ref), (xst, yst)
        xb, yb = ctx.to_device(xs), ctx.alloc(4 * M * N)
        try:
            mi355x.check(ctx.lib.mi355x_gemv_batched_noalloc(ctx.h, t, w.ptr, N, K, xb.ptr, K, yb.ptr, N, M))
            ctx.sync()
            assert np.array_equal(yb.download(np.float32, M * N).reshape(M, N), ref)
        finally:
            xb.free()
            yb.free()
    finally:
        w.free()
