"""Batched calls keep to the arithmetic and the form that the caller has set:
MI355X_VARIANT_DIGITS is fixed point per 32-value block at every number of
activations, and a form, rows, prefetch or workgroup cap reaches the calls that
run as one GEMV per activation."""
import numpy as np
import pytest

import mi355x
import synth
from tolerance import DIGIT_SUM, check_sum, product64

pytestmark = pytest.mark.gpu

KQ = {"Q3_K": 11, "Q4_K": 12, "Q6_K": 14, "IQ4_XS": 23, "IQ3_S": 21}


class options:
    def __init__(self, ctx, **opts):
        self.ctx, self.opts = ctx, {getattr(mi355x, "OPT_" + k): v for k, v in opts.items()}

    def __enter__(self):
        for k, v in self.opts.items():
            self.ctx.set_option(k, v)

    def __exit__(self, *exc):
        for k in self.opts:
            self.ctx.set_option(k, 0)


def rows(K, M):
    return np.stack([synth.activations(K, seed=700 + m) for m in range(M)])


@pytest.mark.parametrize("N,K", [(130, 2048), (70, 4096), (300, 768), (64, 6144)])
def test_digits_q4_0_many_activations(ctx, N, K):
    """21 activations run as passes of 8, 8 and 5 of the form that 8 and 5 take."""
    xs = rows(K, 21)
    w = ctx.resident(2, synth.random_q4_0(N, K, 5), N, K)
    try:
        with options(ctx, VARIANT=mi355x.VARIANT_DIGITS):
            y = ctx.gemv_batched(w, xs)
            parts = [ctx.gemv_batched(w, xs[a:b]) for a, b in ((0, 8), (8, 16), (16, 21))]
            # 2^-22 beside 1 is less than half a step of 20-bit fixed point
            x = np.zeros((17, K), np.float32)
            x[:, 0] = 1.0
            x[1::2, 1] = 2.0 ** -22
            same = ctx.gemv_batched(w, x)
    finally:
        w.free()
    assert np.array_equal(y, np.concatenate(parts))
    assert np.array_equal(same, np.tile(same[:1], (17, 1)))


@pytest.mark.parametrize("name", list(KQ))
@pytest.mark.parametrize("opts", [dict(VARIANT=2), dict(VARIANT=2, FORM=4), dict(FORM=4), dict(FORM=3, VARIANT=0),
                                  dict(FORM=2), dict(ROWS_PER_WAVE=2), dict(PREFETCH=1), dict(GRID=5)],
                         ids=lambda o: "-".join(f"{k}{v}" for k, v in o.items()))
def test_kq_options_reach_batched_calls(ctx, name, opts):
    """The bits of one mi355x_gemv per activation with the same options (20
    activations; 4 where an option leaves no matrix-core form)."""
    t, N, K = KQ[name], 260, 2048
    w = ctx.resident(t, synth.random_blocks(t, N, K, 9), N, K)
    xs = rows(K, 20)
    try:
        with options(ctx, **opts):
            for M in (20,) if set(opts) <= {"VARIANT", "GRID"} else (20, 4):
                y = ctx.gemv_batched(w, xs[:M])
                one = np.stack([ctx.gemv(w, xs[m]) for m in range(M)])
                assert np.array_equal(y, one), M
    finally:
        w.free()


def test_digits_q4_0_long_rows_stay_refused(ctx):
    """No digit kernel takes rows of more than 16384 values, whatever M is."""
    N, K = 8, 16640
    w = ctx.resident(2, synth.random_q4_0(N, K, 3), N, K)
    x, y = ctx.alloc(4 * 20 * K), ctx.alloc(4 * 20 * N)
    try:
        with options(ctx, VARIANT=mi355x.VARIANT_DIGITS):
            for M in (1, 3, 20):
                assert ctx.gemv_batched_ptr(2, w.ptr, N, K, x.ptr, K, y.ptr, N, M) == mi355x.EUNSUPPORTED, M
    finally:
        for b in (w, x, y):
            b.free()


@pytest.mark.parametrize("name,N,K", [("Q4_0", 300, 2048), ("Q4_0", 70, 8192), ("Q4_K", 300, 2048), ("Q6_K", 64, 8448),
                                      ("IQ3_S", 300, 2048), ("IQ3_S", 4100, 2048), ("IQ4_XS", 64, 4096)])
def test_output_across_batch_sizes(ctx, oracle, name, N, K):
    """The same activation alone, among 4, 9, 21 and 40: the arithmetic depends on
    the number (fixed point per 32 values of 20 bits for Q4_0 and 16 for the other
    types, or two f16 planes, or f32), and each stays within its bound."""
    t = 2 if name == "Q4_0" else KQ[name]
    xs = rows(K, 40)
    w = ctx.resident(t, synth.random_q4_0(N, K, 5) if t == 2 else synth.random_blocks(t, N, K, 5), N, K)
    try:
        ys = [ctx.gemv(w, xs[0])] + [ctx.gemv_batched(w, xs[:M])[0] for M in (4, 9, 21, 40)]
        raw = w.raw_bytes()
    finally:
        w.free()
    ref, norms = product64(oracle, t, raw, N, K, xs[:1])
    for y in ys:
        check_sum(y[None], ref, norms, xs[:1], DIGIT_SUM / 16 if t == 2 else DIGIT_SUM, name)
