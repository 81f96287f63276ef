"""Batched calls on activation rows whose blocks differ by more than the two f16
planes of a row can hold: a large part that meets zero weights must not cost the
small part its precision.  Against 64 bits, every weight type."""
import numpy as np
import pytest

import mi355x
import synth
from test_gemm_batched_gpu import GRIDS, TYPES, install_grids, run, weights  # noqa: F401 (fixture)
from tolerance import check_f32_sum, product64

pytestmark = pytest.mark.gpu


def zero_scales(t, raw, N, blocks):
    """raw with the fp16 scales of these blocks 0"""
    r = raw.reshape(N, -1, mi355x.BLOCK_BYTES[t]).copy()
    for off in synth.HALF_FIELDS[t]:
        r[:, blocks, off:off + 2] = 0
    return r.reshape(N, -1)


# one and several column and row tiles, one K segment and several, a partial
# superblock (Q4_0)
SIZES = [(300, 1024, 20), (70, 512, 70), (513, 4352, 33), (40, 1024 + 64, 18)]


@pytest.mark.parametrize("name", list(TYPES))
@pytest.mark.parametrize("N,K,M", SIZES)
def test_wide_rows(ctx, oracle, name, N, K, M):
    t = TYPES[name]
    if t != 2:
        K = max(256, K // 256 * 256)
    bv = mi355x.BLOCK_VALUES[t]
    raw = zero_scales(t, weights(t, N, K, N + K), N, [0])
    base = np.stack([synth.activations(K, seed=50 + m) for m in range(M)])
    base[:, :bv] = 0  # what meets the zero weights does not count
    xs = base.copy()
    xs[1, 3] = 2.0 ** 24
    xs[4] *= 2.0 ** -60
    xs[4, 0] = 2.0 ** 60
    # sums of 256 products with codes times scales (up to 2^12) stay finite before
    # they meet the zero scale: 2^20 * 1e30 < 3.4e38
    xs[M - 1, :bv] = 1e30
    grid = GRIDS.get(t)
    ref, norms = product64(oracle, t, raw, N, K, base, grid)
    scale = np.ones(M)
    scale[4] = 2.0 ** -60
    y = run(ctx, t, raw, N, K, xs)
    check_f32_sum(y / scale[:, None], ref, norms, base, f"{name} {N}x{K} M={M}")
    # the other rows do not notice
    plain = [m for m in range(M) if m not in (1, 4, M - 1)]
    assert np.array_equal(run(ctx, t, raw, N, K, base)[plain], y[plain])


# few Q4_0 activations: one quad of blocks and several per wavefront, wavefronts
# without a quad, two launches (K > 8192), more tiles than workgroups, passes of 8
@pytest.mark.parametrize("N,K,M", [(50, 256, 2), (300, 1024, 5), (17, 2560, 3), (4100, 8192, 8), (16400, 9216, 5),
                                   (16 * 600 + 5, 1024, 8), (70, 2048, 13)])
def test_few_wide_q4_0_rows(ctx, oracle, N, K, M):
    raw = zero_scales(2, synth.random_q4_0(N, K, N + K), N, [0, K // 32 - 1])
    base = np.stack([synth.activations(K, seed=50 + m) for m in range(M)])
    base[:, :32] = base[:, -32:] = 0
    base[0, 64:128] = 0  # blocks of zeros are not small
    base[1, np.arange(K) % 4 != K % 7 % 4] = 0  # one value in four, and blocks of a single one
    base[1, 128:192] = 0
    base[1, 131] = 1.0
    xs = base.copy()
    xs[1, 3] = 2.0 ** 24
    xs[M - 1] *= 2.0 ** -60
    xs[M - 1, K - 1] = 2.0 ** 60
    scale = np.ones((M, 1))
    scale[M - 1] = 2.0 ** -60
    rows = np.unique(np.concatenate([np.arange(min(N, 40)), np.arange(max(0, N - 40), N)]))
    ref, norms = product64(oracle, 2, raw[rows], len(rows), K, base)
    y = run(ctx, 2, raw, N, K, xs)
    check_f32_sum(y[:, rows] / scale, ref, norms, base, f"{N}x{K} M={M}")
    plain = [m for m in range(M) if m not in (1, M - 1)]
    assert np.array_equal(run(ctx, 2, raw, N, K, base)[plain], y[plain])
