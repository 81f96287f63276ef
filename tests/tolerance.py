"""Parity bar for floating-point GEMV results against the CPU oracle.

cosine(y, y_ref) >= 0.999999 over the whole output, and per row
|y_r - y_ref_r| <= 1e-4 * ||w_r||_2 * ||x||_2  (the Cauchy-Schwarz scale of
y_r; "max |err| <= 1e-4 x ||row||" of the path's target).
"""
import numpy as np

COS_MIN = 0.999999
ROW_REL = 1e-4


def cosine(a, b) -> float:
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    na, nb = np.linalg.norm(a), np.linalg.norm(b)
    if na == 0.0 and nb == 0.0:
        return 1.0
    if na == 0.0 or nb == 0.0:
        return 0.0
    return float(np.dot(a, b) / (na * nb))


def check_gemv(y, y_ref, row_norms, x, what="") -> dict:
    y = np.asarray(y, dtype=np.float64)
    y_ref = np.asarray(y_ref, dtype=np.float64)
    assert y.shape == y_ref.shape, what
    assert np.all(np.isfinite(y)), f"{what}: non-finite output"
    bound = ROW_REL * np.asarray(row_norms, dtype=np.float64) * float(np.linalg.norm(np.asarray(x, np.float64)))
    err = np.abs(y - y_ref)
    worst = int(np.argmax(err - bound)) if y.size else 0
    c = cosine(y, y_ref)
    stats = {"cosine": c, "max_abs_err": float(err.max()) if y.size else 0.0,
             "worst_row": worst}
    assert c >= COS_MIN, f"{what}: cosine {c:.9f} < {COS_MIN} ({stats})"
    assert np.all(err <= bound), (f"{what}: row {worst} err {err[worst]:.3e} > bound {bound[worst]:.3e}")
    return stats


# Results against 64 bits, per output: at most BOUND * ||w|| * rms(x), with ||w||
# rms(x) the standard deviation of an output whose activations are independent.
# F32_SUM, f32-accurate arithmetic (f32 or two-f16-plane activations, f32 sums):
# two planes are off by at most 2^-23 of a value (rms 4e-8), f32 sums of these
# lengths by 1e-7 to 2.5e-7; the bound is eight times that.  One f16 plane alone
# is off by 1.5e-4.
# DIGIT_SUM, 16-bit fixed point per 32 values: half a step is 2^-16 of the block's
# largest value, 2 to 4 times rms(x), uniform, so 2e-5 to 4e-5; the bound is six
# times that.  One 8-bit digit plane alone is off by 256 times as much.
# (tests/test_bounds_cpu.py shows both sides.)
F32_SUM = 2e-6
DIGIT_SUM = 2.5e-4


def product64(oracle, t, raw, N, K, xs, grid=None):
    """(xs @ W^T, ||w|| per row) in float64 from the oracle's weights."""
    rows = np.ascontiguousarray(raw).reshape(N, -1)
    W = np.stack([oracle.dequant_row(t, r, K, grid=grid) for r in rows]).astype(np.float64)
    return np.asarray(xs, np.float64) @ W.T, np.linalg.norm(W, axis=1)


def times_bound(y, ref, norms, xs, bound):
    xs = np.asarray(xs, np.float64)
    b = bound * np.sqrt((xs * xs).mean(axis=1))[:, None] * norms[None, :]
    err = np.abs(np.asarray(y, np.float64) - ref)
    return float((err / np.maximum(b, 1e-300)).max()) if err.size else 0.0


def check_sum(y, ref, norms, xs, bound, what=""):
    worst = times_bound(y, ref, norms, xs, bound)
    assert worst <= 1.0, f"{what}: {worst:.2f} times the bound"  # also fails for NaN


def check_f32_sum(y, ref, norms, xs, what=""):
    check_sum(y, ref, norms, xs, F32_SUM, what)
