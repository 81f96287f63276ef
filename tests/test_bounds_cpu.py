"""The bounds of tolerance.py against 64 bits: met by numpy restatements of the
arithmetic they are for, and missed by the same with a part left out."""
import numpy as np
import pytest

import synth
from tolerance import DIGIT_SUM, F32_SUM, product64, times_bound


def rows(K, M=6):
    return np.stack([synth.activations(K, seed=300 + m) for m in range(M)])


def planes(x):
    """hi + lo and hi of the two f16 planes of each row, unscaled again"""
    s = 2.0 ** (14 - np.floor(np.log2(np.abs(x).max(axis=1, keepdims=True))))
    w = x.astype(np.float64) * s
    hi = w.astype(np.float16).astype(np.float64)
    lo = (w - hi).astype(np.float16).astype(np.float64)
    return (hi + lo) / s, hi / s


def digits(x, bits):
    """fixed point of `bits` bits per 32 values"""
    b = x.astype(np.float64).reshape(x.shape[0], -1, 32)
    step = np.abs(b).max(axis=2, keepdims=True) / 2.0 ** (bits - 1)
    return (np.round(b / step) * step).reshape(x.shape)


@pytest.mark.parametrize("t,K", [(2, 256), (2, 11008), (14, 4096), (12, 2304), (23, 1280)])
def test_bounds_see_what_is_left_out(oracle, t, K):
    N = 40
    raw = synth.random_q4_0(N, K, 1) if t == 2 else synth.random_blocks(t, N, K, 1)
    xs = rows(K)
    ref, norms = product64(oracle, t, raw, N, K, xs)
    W = np.stack([oracle.dequant_row(t, r, K) for r in raw.reshape(N, -1)])

    def worst(x, bound, w=W):
        return times_bound(x @ w.T.astype(np.float64), ref, norms, xs, bound)

    both, high = planes(xs)
    assert worst(both, F32_SUM) < 0.3 and worst(high, F32_SUM) > 20
    assert worst(digits(xs, 16), DIGIT_SUM) < 0.8 and worst(digits(xs, 8), DIGIT_SUM) > 20
    # and f32 chains of 256 products, then over the 256s
    y = np.zeros((len(xs), N), np.float32)
    for k in range(0, K, 256):
        part = np.zeros_like(y)
        for i in range(k, min(k + 256, K)):
            part += xs[:, i:i + 1] * W[None, :, i]
        y += part
    assert times_bound(y, ref, norms, xs, F32_SUM) < 1


def test_bound_sees_the_remainder_of_12_bit_weights(oracle):
    """Q6_K's code times scale rounded to f16's 11 bits."""
    t, N, K = 14, 40, 2048
    raw = synth.random_blocks(t, N, K, 2)
    xs = rows(K)
    ref, norms = product64(oracle, t, raw, N, K, xs)
    d = np.frombuffer(raw.reshape(N, -1, 210)[:, :, 208:210].tobytes(), np.float16).reshape(N, -1).astype(np.float32)
    W = np.stack([oracle.dequant_row(t, r, K) for r in raw.reshape(N, -1)]).reshape(N, -1, 256)
    codes = W / d[:, :, None]
    rounded = (codes.astype(np.float16).astype(np.float64) * d[:, :, None]).reshape(N, K)
    assert times_bound(xs.astype(np.float64) @ rounded.T, ref, norms, xs, F32_SUM) > 20
