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


# Results of f32-accurate arithmetic (f32 or 22-bit activations, f32 sums)
# against 64 bits: per output at most F32_SUM * ||w|| * rms(x), the standard
# deviation of an output whose activations are independent.  22-bit activations
# are off by at most 2^-23 each (rms 4e-8 of that scale), a chain of f32 sums of
# this length by 1e-7 to 2.5e-7; the bound is eight times that.  One f16 plane
# alone (2^-12 at worst, rms 1e-4) exceeds it everywhere, 20-bit fixed point
# per 32 values (rms 3e-6) and 16-bit (3e-5) on most outputs.
F32_SUM = 2e-6


def product64(oracle, t, raw, N, K, xs, grid=None):
    """(xs @ W^T, ||w|| per row) in float64 from the oracle's weights."""
    rows = np.ascontiguousarray(raw).reshape(N, -1)
    W = np.stack([oracle.dequant_row(t, r, K, grid=grid) for r in rows]).astype(np.float64)
    return np.asarray(xs, np.float64) @ W.T, np.linalg.norm(W, axis=1)


def check_f32_sum(y, ref, norms, xs, what=""):
    xs = np.asarray(xs, np.float64)
    bound = F32_SUM * np.sqrt((xs * xs).mean(axis=1))[:, None] * norms[None, :]
    err = np.abs(np.asarray(y, np.float64) - ref)
    assert np.isfinite(err).all(), what
    worst = float((err / np.maximum(bound, 1e-300)).max()) if err.size else 0.0
    assert worst <= 1.0, f"{what}: {worst:.2f} times the bound"
    return worst
