"""The workspace of batched calls of many activations: calls that it cannot hold
at once (several passes), sums over fewer K segments than asked for, and a
context that has none."""
import numpy as np
import pytest

import mi355x
import synth
from test_gemm_batched_gpu import GRIDS, TYPES, install_grids, run, weights  # noqa: F401 (fixture)
from tolerance import check_f32_sum, product64

pytestmark = pytest.mark.gpu

# 64 MiB hold 248 rows of 65536 values (passes of 160 and 140 here) and 512 rows
# of 30208 with 2 MiB left for partial sums (4 segments of N = 256, M = 512);
# rows past 124 superblocks in passes of 32 to the end
SIZES = [("Q4_K", 40, 65536, 300), ("Q6_K", 256, 30208, 512), ("IQ3_S", 33, 65536, 260), ("Q3_K", 70, 262144, 70)]


@pytest.mark.parametrize("name,N,K,M", SIZES)
def test_more_than_the_workspace_holds(ctx, oracle, name, N, K, M):
    t = TYPES[name]
    raw = weights(t, N, K, 3)
    rng = np.random.default_rng(K + M)
    xs = rng.standard_normal((M, K), dtype=np.float32)
    y = run(ctx, t, raw, N, K, xs)
    rows = np.arange(N)[:: max(1, N // 16)]
    ref, norms = product64(oracle, t, raw.reshape(N, -1)[rows], len(rows), K, xs)
    check_f32_sum(y[:, rows], ref, norms, xs, f"{name} {N}x{K} M={M}")


@pytest.mark.parametrize("name", list(TYPES))
def test_context_without_a_workspace(ctx, name):
    """The other forms: passes of 8 Q4_0 activations, one GEMV per K/IQ activation."""
    t, N, K, M = TYPES[name], 300, 2048, 21
    raw = weights(t, N, K, 6)
    xs = np.stack([synth.activations(K, seed=m) for m in range(M)])
    w = ctx.resident(t, raw, N, K)
    try:
        if t == 2:
            ref = np.concatenate([ctx.gemv_batched(w, xs[a:a + 8]) for a in (0, 8)] + [ctx.gemv_batched(w, xs[16:])])
        else:
            ref = np.stack([ctx.gemv(w, x) for x in xs])
    finally:
        w.free()
    mi355x.inject_fault("mi355x_ctx_workspace", mi355x.HIP_ERROR_OUT_OF_MEMORY)
    try:
        with mi355x.Context(0) as c:
            assert mi355x.last_error() == ""
            assert np.array_equal(run(c, t, raw, N, K, xs), ref)
    finally:
        mi355x.inject_fault(None)
