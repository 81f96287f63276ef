"""Batched calls of the IQ types where one mi355x_gemv sums f32 activations in
f32 (codebook matrices of fewer than 4096 rows, rows longer than 8192 values):
no further from 64 bits than those one-row calls, with and without values of
very different size in a row."""
import numpy as np
import pytest

import mi355x
import synth
from test_gemm_batched_gpu import GRIDS, TYPES, install_grids, run, weights  # noqa: F401 (fixture)
from tolerance import product64

pytestmark = pytest.mark.gpu

# both errors are of fixed inputs (0.9 to 1.35e-7 here, one-row calls 0.9 to
# 2.6e-7); the factor is for the spread over inputs of the smallest size
FACTOR = 1.1
CASES = [(n, N, K, M) for n in ("IQ3_S", "IQ3_XXS", "IQ2_S") for N, K, M in ((90, 256, 40), (300, 1024, 9), (70, 4096, 70))]
CASES += [(n, 60, K, 33) for n in ("IQ4_XS", "IQ3_S", "IQ3_XXS", "IQ2_S") for K in (8448, 14336)]


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("name,N,K,M", CASES)
def test_no_further_from_64_bits_than_one_row_calls(ctx, oracle, name, N, K, M, wide):
    t = TYPES[name]
    raw = weights(t, N, K, K + M)
    xs = np.stack([synth.activations(K, seed=m) for m in range(M)])
    if wide:  # ordinary values and a part 2^16 smaller, which carries the sum where the weights of the rest are zero
        r = raw.reshape(N, -1, mi355x.BLOCK_BYTES[t]).copy()
        for off in synth.HALF_FIELDS[t]:
            r[: N // 2, 1:, off:off + 2] = 0
        raw = r.reshape(N, -1)
        xs[::2, :256] *= np.float32(2.0 ** -16)
    ref, _ = product64(oracle, t, raw, N, K, xs, GRIDS.get(t))

    def error(y):
        half = slice(0, N // 2) if wide else slice(None)
        s = np.linalg.norm(ref[:, half], axis=1)[:, None]
        return np.sqrt((((y - ref)[:, half] / s) ** 2).sum() / M)

    batched = run(ctx, t, raw, N, K, xs)
    ctx.set_option(mi355x.OPT_VARIANT, mi355x.VARIANT_EXACT_F32)
    try:
        one = run(ctx, t, raw, N, K, xs)
    finally:
        ctx.set_option(mi355x.OPT_VARIANT, mi355x.VARIANT_AUTO)
    assert error(batched) <= FACTOR * error(one), (error(batched), error(one))
