"""K/IQ GEMVs that read the activation row as the caller has it: f32 off a
16-byte boundary and BF16 on and off it give the bits of the same values as
aligned f32, at every step count of the row kernels, in both arithmetics and
past one LDS chunk."""
import numpy as np
import pytest

import mi355x
import synth

pytestmark = pytest.mark.gpu

TYPES = {"Q3_K": 11, "Q4_K": 12, "Q5_K": 13, "Q6_K": 14, "IQ4_XS": 23, "IQ3_S": 21}


@pytest.mark.parametrize("variant", [mi355x.VARIANT_DIGITS, mi355x.VARIANT_EXACT_F32])
@pytest.mark.parametrize("name", list(TYPES))
@pytest.mark.parametrize("N,K", [(33, 256), (40, 2816), (70, 5120), (9, 11008), (17, 14336), (8, 16640)])
def test_any_activation_matches_aligned_f32(ctx, name, variant, N, K):
    t = TYPES[name]
    w = ctx.resident(t, synth.random_blocks(t, N, K, N + K), N, K)
    xb = (synth.activations(K, seed=K).view(np.uint32) >> 16).astype(np.uint16)
    xf = (xb.astype(np.uint32) << 16).view(np.float32)
    dev, y = ctx.alloc(4 * K + 64), ctx.alloc(4 * N)
    ctx.set_option(mi355x.OPT_VARIANT, variant)
    try:
        def run(x, off):
            dev.upload(x, offset=off)
            mi355x.check(ctx.gemv_ptr(t, w.ptr, N, K, dev.ptr + off, y.ptr, x.dtype == np.uint16))
            ctx.sync()
            return y.download(np.uint32, N)
        ref = run(xf, 0)
        for x, off in ((xf, 4), (xf, 8), (xb, 0), (xb, 2), (xb, 8)):
            assert np.array_equal(run(x, off), ref), (x.dtype, off)
    finally:
        ctx.set_option(mi355x.OPT_VARIANT, mi355x.VARIANT_AUTO)
        for b in (dev, y, w):
            b.free()
