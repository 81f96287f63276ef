"""Matrix-core batched GEMV (mi355x_gemv_batched with many activations) on the
GPU against the CPU oracle and 64 bits: every weight type, sizes around the tiles (256
weight rows per workgroup, 64 per wavefront, 32 or 64 activations per tile,
256-value superblocks, K segments), strides and unaligned rows, extreme
activation scales, and the allocation-free form, which must give the same
bits."""
import numpy as np
import pytest

import mi355x
import synth
from tolerance import F32_SUM, check_gemv, check_sum, product64

pytestmark = pytest.mark.gpu

TYPES = {"Q4_0": 2, "Q3_K": 11, "Q4_K": 12, "Q5_K": 13, "Q6_K": 14, "IQ4_XS": 23, "IQ3_S": 21, "IQ3_XXS": 18,
         "IQ2_S": 22}


def synthetic_grid(t, top=61):
    # odd magnitudes, as ggml's (the same shape the other K/IQ GPU tests install)
    rng = np.random.default_rng(t)
    n, w = (256, 4) if t == 18 else (1024, 8)
    g = (2 * rng.integers(0, (top + 1) // 2, (n, w)) + 1).astype(np.uint8)
    return g.view(np.uint32 if w == 4 else np.uint64).reshape(n)


GRIDS = {t: synthetic_grid(t) for t in (18, 22)}


@pytest.fixture(scope="module", autouse=True)
def install_grids():
    for t, g in GRIDS.items():
        mi355x.set_iq_grid(t, g)
    yield


def weights(t, N, K, seed):
    return synth.random_q4_0(N, K, seed) if t == 2 else synth.random_blocks(t, N, K, seed)


def check(oracle, t, raw, N, K, xs, y, what, grid=None, bound=None):
    """Against the oracle, and against 64 bits within bound * ||w|| * rms(x)."""
    grid = GRIDS.get(t) if grid is None else grid
    if bound:
        check_sum(y, *product64(oracle, t, raw, N, K, xs, grid), xs, bound, what)
    norms = oracle.row_norms(t, raw, N, K, grid=grid)
    for m in range(xs.shape[0]):
        check_gemv(y[m], oracle.gemv(t, raw, N, K, xs[m], grid=grid), norms, xs[m], f"{what} activation {m}")


def run(ctx, t, raw, N, K, xs, **kw):
    w = ctx.resident(t, raw, N, K)
    try:
        return ctx.gemv_batched(w, xs, **kw)
    finally:
        w.free()


# (N, K, M): one column tile or less, ragged rows of the last tile and of the
# last wavefront, one to many superblocks (odd: rows that start 2 mod 4), one
# and several segments, activations below, at and past a tile of 32 or 64
SIZES = [(1, 256, 16), (64, 512, 17), (257, 768, 32), (300, 2304, 33), (511, 1280, 64), (96, 11008, 65),
         (1030, 4096, 24), (40, 16640, 96)]


@pytest.mark.parametrize("name", list(TYPES))
@pytest.mark.parametrize("N,K,M", SIZES)
def test_gemm_matches_oracle(ctx, oracle, name, N, K, M):
    t = TYPES[name]
    raw = weights(t, N, K, N + K)
    xs = np.stack([synth.activations(K, seed=100 + m) for m in range(M)])
    check(oracle, t, raw, N, K, xs, run(ctx, t, raw, N, K, xs), f"{name} {N}x{K} M={M}", bound=F32_SUM)


def test_gemm_q4_0_partial_superblock(ctx, oracle):
    """Q4_0 rows that end inside a superblock (an even number of blocks)."""
    for N, K in ((70, 64), (300, 2048 + 192), (33, 4416)):
        raw = synth.random_q4_0(N, K, 3)
        xs = np.stack([synth.activations(K, seed=m) for m in range(20)])
        check(oracle, 2, raw, N, K, xs, run(ctx, 2, raw, N, K, xs), f"Q4_0 {N}x{K}", bound=F32_SUM)


@pytest.mark.parametrize("name", ["Q4_0", "Q4_K", "IQ3_S"])
def test_gemm_more_rows_than_one_pass(ctx, oracle, name):
    t, N, K, M = TYPES[name], 130, 512, 520
    raw = weights(t, N, K, 4)
    xs = np.stack([synth.activations(K, seed=m) for m in range(M)])
    check(oracle, t, raw, N, K, xs, run(ctx, t, raw, N, K, xs), f"{name} M={M}", bound=F32_SUM)


@pytest.mark.parametrize("name", list(TYPES))
def test_gemm_strides_noalloc_and_unaligned_rows(ctx, name):
    """Padded and (batched form only) unaligned activation rows, padded
    outputs, and mi355x_gemv_batched_noalloc: the same bits."""
    t, N, K, M = TYPES[name], 517, 4096, 35
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


@pytest.mark.parametrize("name", ["Q4_0", "Q5_K", "Q6_K", "IQ2_S"])
def test_gemm_activation_scales_and_nonfinite(ctx, oracle, name):
    """Rows of tiny, huge, zero and mixed magnitudes; a row with an infinity
    or a NaN poisons its own outputs only."""
    t, N, K, M = TYPES[name], 90, 1536, 18
    raw = weights(t, N, K, 12)
    xs = np.stack([synth.activations(K, seed=m) for m in range(M)])
    xs[1] *= 1e-30
    xs[2] *= 1e25
    xs[3] = 0.0
    xs[4, ::256] *= 1e4
    xs[5, :256] = 0.0
    y = run(ctx, t, raw, N, K, xs)
    assert np.all(y[3] == 0.0)
    rows = [m for m in range(M) if m != 3]
    check(oracle, t, raw, N, K, xs[rows], y[rows], name, bound=F32_SUM)
    bad = xs.copy()
    bad[7, 300] = np.inf
    bad[8, 5] = np.nan
    yb = run(ctx, t, raw, N, K, bad)
    assert not np.isfinite(yb[7]).any() and np.isnan(yb[8]).all()
    keep = [m for m in range(M) if m not in (7, 8)]
    assert np.array_equal(yb[keep], y[keep])


@pytest.mark.parametrize("name", ["IQ3_XXS", "IQ2_S"])
def test_gemm_grid_past_f16_products(ctx, oracle, name):
    """A grid whose magnitudes times the largest scale do not fit f16 exactly
    keeps the single-row kernels."""
    t, N, K, M = TYPES[name], 64, 1024, 20
    raw = weights(t, N, K, 2)
    xs = np.stack([synth.activations(K, seed=m) for m in range(M)])
    g = synthetic_grid(t, top=127)
    mi355x.set_iq_grid(t, g)
    try:
        y = run(ctx, t, raw, N, K, xs)
    finally:
        mi355x.set_iq_grid(t, GRIDS[t])
    check(oracle, t, raw, N, K, xs, y, name, grid=g)
