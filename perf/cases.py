"""Performance cases of the decode-GEMV library, each one call (or one decode
step's calls) through the public entry points.

Kinds of case (field ``kind``):

* ``gemv``     one mi355x_gemv / mi355x_gemv_bf16 call: a single activation
               row against one resident matrix, the decode matmul itself.
* ``step``     the GEMVs of one decode token of a Qwen2-shaped model: per
               layer q|k|v and gate|up as mi355x_gemv_multi groups, o and down
               as mi355x_gemv, then the vocabulary projection.
* ``batched``  one mi355x_gemv_batched call: M activation rows against one
               matrix, what the plugin's M > 1 MUL_MAT nodes run (a few rows
               when several sequences decode together, up to a 512-row
               micro-batch when a prompt is processed).
* ``decode``   a whole greedy decode of a small Qwen2-shaped model through the
               ggml plugin's graph_compute (tokens and last logits).

Weights are seeded: Q4_0 is N(0, 0.02) quantized by ggml's rule, the other
types random codes and scales with the fp16 scales spread over two binades.
Activations are N(0, 1) with 1% of the columns eight times larger, as hidden
states have.  IQ3_XXS and IQ2_S use a synthetic grid of odd magnitudes up to
61 (ggml's tables are not part of this repository).
"""
import math
import os
import random
import sys
import weakref

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "xdna.cpp_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import decode  # noqa: E402  (after torch, whose HIP runtime the library then shares)
import mi355x  # noqa: E402
import synth  # noqa: E402

TYPES = {"q4_0": 2, "q3_k": 11, "q4_k": 12, "q5_k": 13, "q6_k": 14, "iq3_xxs": 18, "iq3_s": 21, "iq2_s": 22,
         "iq4_xs": 23}
VARIANTS = {"auto": mi355x.VARIANT_AUTO, "ggml_q8": mi355x.VARIANT_GGML_Q8}
# the most multiply-adds a case may take: the largest listed one
MAX_MACS = 512 * 4096 * 14336


def listed():
    return [
        # the smallest decode GEMV, the 3B shape's o projection: one launch's latency
        {"name": "gemv q4_0 2048x2048", "kind": "gemv", "type": "q4_0", "N": 2048, "K": 2048, "variant": "auto",
         "bf16": False},
        # the headline GEMV shape
        {"name": "gemv q4_0 8192x8192", "kind": "gemv", "type": "q4_0", "N": 8192, "K": 8192, "variant": "auto",
         "bf16": False},
        # the vocabulary projection in ggml-cpu's numerics, as a host that wants ggml's tokens runs it
        {"name": "gemv q4_0 vocab ggml", "kind": "gemv", "type": "q4_0", "N": 151936, "K": 2048,
         "variant": "ggml_q8", "bf16": False},
        # the most common K-quant at an FFN up shape
        {"name": "gemv q4_k 14336x4096", "kind": "gemv", "type": "q4_k", "N": 14336, "K": 4096, "variant": "auto",
         "bf16": False},
        # a codebook type (table lookups from LDS) on the square shape
        {"name": "gemv iq3_s 8192x8192", "kind": "gemv", "type": "iq3_s", "N": 8192, "K": 8192, "variant": "auto",
         "bf16": False},
        # odd sizes and BF16 activations: rows that start 2 mod 4, a partial last step
        {"name": "gemv q3_k bf16 ragged", "kind": "gemv", "type": "q3_k", "N": 3001, "K": 2816, "variant": "auto",
         "bf16": True},
        # one decode token's GEMVs of the 3B shape: 145 calls over 1.7 GB of weights
        {"name": "step q4_0 3B", "kind": "step", "layers": 36, "hidden": 2048, "kv": 256, "ffn": 11008,
         "vocab": 151936, "variant": "auto"},
        # eight sequences decoding together
        {"name": "batched q4_0 M=8", "kind": "batched", "type": "q4_0", "N": 8192, "K": 8192, "M": 8,
         "variant": "auto", "xpad": 0, "ypad": 0, "noalloc": False},
        # the last, ragged micro-batch of a prompt on a K-quant
        {"name": "batched q4_k M=37", "kind": "batched", "type": "q4_k", "N": 14336, "K": 4096, "M": 37,
         "variant": "auto", "xpad": 0, "ypad": 0, "noalloc": False},
        # full 512-row micro-batches of a prompt
        {"name": "batched q4_0 M=512", "kind": "batched", "type": "q4_0", "N": 17408, "K": 5120, "M": 512,
         "variant": "auto", "xpad": 0, "ypad": 0, "noalloc": False},
        {"name": "batched q6_k M=512", "kind": "batched", "type": "q6_k", "N": 4096, "K": 14336, "M": 512,
         "variant": "auto", "xpad": 0, "ypad": 0, "noalloc": False},
        # the drop-in path end to end: every GEMV group of 12 forward passes through graph_compute
        {"name": "decode plugin", "kind": "decode", "layers": 2, "hidden": 2048, "heads": 16, "kv_heads": 2,
         "head_dim": 128, "ffn": 11008, "vocab": 32000, "prompt": 6, "gen": 7},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choices(["gemv", "batched", "step", "decode"], [9, 8, 2, 1])[0]
    if kind == "decode":
        heads = rng.choice([4, 8, 12, 16])
        return {"kind": "decode", "layers": rng.randint(1, 3), "hidden": 128 * heads, "heads": heads,
                "kv_heads": rng.choice([1, 2, 4]), "head_dim": 128, "ffn": 256 * rng.randint(4, 43),
                "vocab": 32 * _log_int(rng, 100, 1000), "prompt": rng.randint(2, 8), "gen": rng.randint(2, 7)}
    if kind == "step":
        hidden = 256 * rng.randint(4, 16)
        return {"kind": "step", "layers": _log_int(rng, 2, 24), "hidden": hidden, "kv": 128 * rng.randint(1, 8),
                "ffn": 256 * rng.randint(8, 43), "vocab": 64 * _log_int(rng, 50, 2000),
                "variant": rng.choice(["auto", "ggml_q8"])}
    t = rng.choice(["q4_0", "q4_0", "q4_0", "q4_k", "q4_k"] + list(TYPES))
    K = _log_int(rng, 512, 16384)
    # Q4_0 rows are any number of 32-value blocks; most models keep multiples of 256
    K = max(32, K // 32 * 32) if t == "q4_0" and rng.random() < 0.25 else max(256, K // 256 * 256)
    if kind == "gemv":
        variant = "ggml_q8" if rng.random() < 0.2 else "auto"
        bf16 = rng.random() < 0.15 and not (t == "q4_0" and variant == "ggml_q8")
        return {"kind": "gemv", "type": t, "N": _log_int(rng, 64, 32768), "K": K, "variant": variant, "bf16": bf16}
    M = _log_int(rng, 2, 512)
    N = _log_int(rng, 64, max(64, min(17408, MAX_MACS // (M * K))))
    variant = "ggml_q8" if rng.random() < 0.1 else "auto"
    return {"kind": "batched", "type": t, "N": N, "K": K, "M": M, "variant": variant,
            "xpad": rng.choice([0, 0, 0, 64]), "ypad": rng.choice([0, 0, 0, 3]), "noalloc": rng.random() < 0.1}


# ---- inputs ----------------------------------------------------------------


def _rand(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + 17)
    return g


def _halves(shape, lo, hi, g):
    """fp16 values log-uniform in [lo, hi), as bytes [..., 2]."""
    u = torch.rand(shape, generator=g, device="cuda")
    return (lo * torch.exp(u * math.log(hi / lo))).to(torch.float16).view(torch.uint8).reshape(*shape, 2)


# typical |code * sub-block scale| of a random block, so that d gives weights around 0.02
_SPREAD = {11: 40.0, 12: 270.0, 13: 560.0, 14: 1300.0, 18: 110.0, 21: 140.0, 22: 70.0, 23: 1150.0}


def _raw_weights(t, N, K, g):
    """ggml bytes [N, blocks, block_bytes] of a seeded matrix, on the GPU."""
    bb = mi355x.BLOCK_BYTES[t]
    if t == mi355x.Q4_0:
        raw = torch.empty((N, K // 32, bb), dtype=torch.uint8, device="cuda")
        step = max(1, (1 << 26) // K)
        for r in range(0, N, step):
            w = torch.randn((min(step, N - r), K // 32, 32), generator=g, device="cuda") * 0.02
            m = w.gather(2, w.abs().argmax(2, keepdim=True))
            d = m / -8
            q = (w * torch.where(d != 0, 1 / d, 0.0) + 8.5).to(torch.int32).clamp(max=15).to(torch.uint8)
            raw[r:r + step, :, 0:2] = d.to(torch.float16).view(torch.uint8)
            raw[r:r + step, :, 2:] = q[..., :16] | (q[..., 16:] << 4)
        return raw
    raw = torch.randint(0, 256, (N, K // 256, bb), generator=g, device="cuda", dtype=torch.uint8)
    d = 0.02 / _SPREAD[t]
    for i, off in enumerate(synth.HALF_FIELDS[t]):
        # the second field is dmin, which centres codes of 0..15 (Q4_K) or 0..31 (Q5_K)
        f = d if i == 0 else d * (7.5 if t == mi355x.Q4_K else 15.5)
        raw[..., off:off + 2] = _halves(raw.shape[:2], f / 2, f * 2, g)
    return raw


def _activations(M, K, g):
    x = torch.randn((M, K), generator=g, device="cuda")
    wide = torch.rand((K,), generator=g, device="cuda") < 0.01
    return torch.where(wide, 8 * x, x)


_grids = {}


def _grid(t):
    """The installed grid of IQ3_XXS / IQ2_S: [entries, values] magnitudes."""
    if t not in _grids:
        n, w = (256, 4) if t == mi355x.IQ3_XXS else (1024, 8)
        a = (2 * np.random.default_rng(t).integers(0, 31, (n, w)) + 1).astype(np.uint8)
        mi355x.set_iq_grid(t, a)
        _grids[t] = a
    return _grids[t]


_ctxs = {}


def _ctx(variant):
    """One context per arithmetic, as a program keeps it."""
    if variant not in _ctxs:
        c = mi355x.Context(0)
        c.set_option(mi355x.OPT_VARIANT, VARIANTS[variant])
        _ctxs[variant] = c
    return _ctxs[variant]


def _resident(ctx, t, raw, N, K):
    """The matrix in the library's resident layout."""
    packed = torch.empty(raw.numel(), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    mi355x.check(ctx.lib.mi355x_prepack_from_device(ctx.h, t, N, K, packed.data_ptr(), raw.data_ptr(), 0,
                                                    raw.numel()))
    return packed


def _step_shapes(c):
    h, f = c["hidden"], c["ffn"]
    per = [(h, [h, c["kv"], c["kv"]]), (h, [h]), (h, [f, f]), (f, [h])]
    return per * c["layers"] + [(h, [c["vocab"]])]


def _matrix_inputs(c, seed):
    g = _rand(seed)
    t, N, K = TYPES[c["type"]], c["N"], c["K"]
    raw = _raw_weights(t, N, K, g)
    x = _activations(c.get("M", 1), K, g)
    return t, N, K, raw, x.to(torch.bfloat16) if c.get("bf16") else x


def _step_inputs(c, seed):
    """(raw, x index, N, K) of every matrix in call order, one at a time, and the activations."""
    g = _rand(seed)
    shapes = _step_shapes(c)
    xs = {K: _activations(1, K, g)[0] for K in sorted({K for K, _ in shapes})}
    return g, shapes, xs


class _Decoder:
    def __init__(self, c, seed):
        self.model = decode.Model(threads=8, n_layers=c["layers"], hidden=c["hidden"], n_heads=c["heads"],
                                  n_kv_heads=c["kv_heads"], head_dim=c["head_dim"], ffn=c["ffn"], vocab=c["vocab"],
                                  rope_theta=1e6, norm_eps=1e-6, seed=seed + 1)
        weakref.finalize(self, self.model.close)
        self.model.attach_gpu(0)
        self.model.set_wait(self.model.WAIT_PLUGIN)
        self.model.set_variant(mi355x.VARIANT_GGML_Q8)
        self.prompt = decode.prompt_tokens(c["prompt"], c["vocab"], seed)
        self.model.generate(self.prompt[:1], 1)  # places the weights in the plugin's buffer


def prepare(case, seed):
    c = case
    if c["kind"] == "decode":
        return {"case": c, "decoder": _Decoder(c, seed)}
    ctx = _ctx(c["variant"])
    if c["kind"] == "step":
        g, shapes, xs = _step_inputs(c, seed)
        y = torch.empty(sum(sum(ns) for _, ns in shapes), device="cuda")
        calls, keep, at = [], [], 0
        for K, ns in shapes:
            jobs = []
            for n in ns:
                keep.append(_resident(ctx, mi355x.Q4_0, _raw_weights(mi355x.Q4_0, n, K, g), n, K))
                jobs.append((keep[-1].data_ptr(), n, y.data_ptr() + 4 * at))
                at += n
            calls.append((K, xs[K].data_ptr(), jobs))
        torch.cuda.synchronize()
        return {"case": c, "ctx": ctx, "calls": calls, "keep": keep, "xs": xs, "y": y}
    t, N, K, raw, x = _matrix_inputs(c, seed)
    if t in (mi355x.IQ3_XXS, mi355x.IQ2_S):
        _grid(t)
    s = {"case": c, "ctx": ctx, "t": t, "W": _resident(ctx, t, raw, N, K)}
    if c["kind"] == "gemv":
        s["x"], s["y"] = x[0].contiguous(), torch.empty(N, device="cuda")
        if t in (mi355x.IQ3_XXS, mi355x.IQ2_S):
            run(s)  # the context copies a new grid to the device on its first GEMV
    else:
        M, xst, yst = c["M"], K + c["xpad"], N + c["ypad"]
        s["x"] = torch.zeros((M, xst), device="cuda")
        s["x"][:, :K] = x
        s["y"] = torch.empty((M, yst), device="cuda")
        s["out"] = s["y"][:, :N]
        if t in (mi355x.IQ3_XXS, mi355x.IQ2_S):
            mi355x.check(ctx.gemv_ptr(t, s["W"].data_ptr(), N, K, s["x"].data_ptr(), s["y"].data_ptr()))
    torch.cuda.synchronize()
    return s


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "decode":
        d = s["decoder"]
        tokens, _ = d.model.generate(d.prompt, c["gen"])
        return {"logits": d.model.last_logits(), "tokens": tokens}
    ctx = s["ctx"]
    if c["kind"] == "step":
        for K, x, jobs in s["calls"]:
            if len(jobs) == 1:
                rc = ctx.gemv_ptr(mi355x.Q4_0, jobs[0][0], jobs[0][1], K, x, jobs[0][2])
            else:
                rc = ctx.gemv_multi_ptr(mi355x.Q4_0, K, x, jobs)
            mi355x.check(rc)
        return s["y"]
    if c["kind"] == "gemv":
        mi355x.check(ctx.gemv_ptr(s["t"], s["W"].data_ptr(), c["N"], c["K"], s["x"].data_ptr(), s["y"].data_ptr(),
                                  c["bf16"]))
        return s["y"]
    fn = ctx.lib.mi355x_gemv_batched_noalloc if c["noalloc"] else ctx.lib.mi355x_gemv_batched
    mi355x.check(fn(ctx.h, s["t"], s["W"].data_ptr(), c["N"], c["K"], s["x"].data_ptr(), s["x"].stride(0),
                    s["y"].data_ptr(), s["y"].stride(0), c["M"]))
    return s["out"]


# ---- what a pass cannot do without, and what it may differ by -----------------


def _matrix_work(t, N, K, M, xbytes=4):
    row = K // mi355x.BLOCK_VALUES[t] * mi355x.BLOCK_BYTES[t]
    return {"bytes": N * row + M * (xbytes * K + 4 * N), "flops": 2 * M * N * K}


def work(case):
    c = case
    if c["kind"] in ("gemv", "batched"):
        return _matrix_work(TYPES[c["type"]], c["N"], c["K"], c.get("M", 1), 2 if c.get("bf16") else 4)
    if c["kind"] == "step":
        parts = [_matrix_work(mi355x.Q4_0, n, K, 1) for K, ns in _step_shapes(c) for n in ns]
    else:
        q, kv, h = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"], c["hidden"]
        one = [(h, q), (h, kv), (h, kv), (q, h), (h, c["ffn"]), (h, c["ffn"]), (c["ffn"], h)] * c["layers"]
        passes = c["prompt"] + c["gen"] - 1
        parts = [_matrix_work(mi355x.Q4_0, n, k, 1) for k, n in one] * passes
        parts += [_matrix_work(mi355x.Q4_0, c["vocab"], h, 1)] * c["gen"]
    return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}


def tolerance(case):
    c = case
    # ggml-cpu's numerics are defined to the bit: integer block products,
    # float sums in ggml's order
    if c["kind"] == "decode" or c["variant"] == "ggml_q8":
        return "exact"
    # Q4_0 activations are 20-bit fixed point per 32-value block (or f32), sums
    # f32: 3.3e-6 to 3.5e-6 from the 64-bit results
    if c["kind"] == "step" or c["type"] == "q4_0":
        return {"rel": 1.4e-5}
    # the other types' activations are 16-bit fixed point per block: 2.7e-5 to 3.5e-5
    return {"rel": 1.4e-4}


# ---- 64-bit results ------------------------------------------------------------


def _half64(b):
    return b.contiguous().view(torch.float16)[..., 0].to(torch.float64)


def _signs(bits, n):
    """+1 / -1 of the low n bits of each value of `bits`: [..., n]."""
    return 1 - 2 * ((bits[..., None] >> torch.arange(n, device=bits.device)) & 1)


_KV = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]


def _dequantize(t, raw):
    """float64 [rows, K] from ggml blocks [rows, blocks, bytes], from the formats' definitions."""
    R, B, _ = raw.shape
    b = raw.to(torch.int64)
    dev = raw.device

    def at(off, n):
        return b[..., off:off + n]

    def half(off):
        return _half64(raw[..., off:off + 2])

    if t == 2:
        q = torch.cat([at(2, 16) & 15, at(2, 16) >> 4], -1) - 8
        return (half(0)[..., None] * q).reshape(R, -1)
    if t in (12, 13):
        s = at(4, 12)
        sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1)
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1)
        qs = at(16 if t == 12 else 48, 128).reshape(R, B, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 3).reshape(R, B, 8, 32)
        if t == 13:
            qh = at(16, 32)[:, :, None, :]
            q = q + 16 * ((qh >> torch.arange(8, device=dev)[:, None]) & 1)
        w = (half(0)[..., None] * sc)[..., None] * q - (half(2)[..., None] * mn)[..., None]
        return w.reshape(R, -1)
    if t == 14:
        ql = at(0, 128).reshape(R, B, 2, 2, 32)
        qh = at(128, 64).reshape(R, B, 2, 1, 32)
        q = torch.cat([ql & 15, ql >> 4], 3)
        q = q | (((qh >> (2 * torch.arange(4, device=dev)[:, None])) & 3) << 4)
        sc = at(192, 16)
        sc = torch.where(sc > 127, sc - 256, sc).reshape(R, B, 2, 4, 2, 1)
        return (half(208)[..., None, None, None, None] * sc * (q.reshape(R, B, 2, 4, 2, 16) - 32)).reshape(R, -1)
    if t == 11:
        j = torch.arange(4, device=dev)[:, None]
        q = (at(32, 64).reshape(R, B, 2, 1, 32) >> (2 * j)) & 3
        h = at(0, 32).reshape(R, B, 1, 1, 32) >> (4 * torch.arange(2, device=dev)[:, None, None] + j)
        q = q + 4 * (h & 1) - 4
        s, i = at(96, 12), torch.arange(16, device=dev)
        sc = ((s[..., i % 8] >> (4 * (i // 8))) & 15) | (((s[..., 8 + i % 4] >> (2 * (i // 4))) & 3) << 4)
        sc = (sc - 32).reshape(R, B, 2, 4, 2, 1)
        return (half(108)[..., None, None, None, None] * sc * q.reshape(R, B, 2, 4, 2, 16)).reshape(R, -1)
    if t == 23:
        i = torch.arange(8, device=dev)
        sh = at(2, 1) | (at(3, 1) << 8)
        ls = ((at(4, 4)[..., i // 2] >> (4 * (i % 2))) & 15) | (((sh >> (2 * i)) & 3) << 4)
        qs = at(8, 128).reshape(R, B, 8, 16)
        v = torch.tensor(_KV, device=dev)[torch.cat([qs & 15, qs >> 4], -1)]
        return ((half(0)[..., None] * (ls - 32))[..., None] * v).reshape(R, -1)
    if t == 21:
        table = torch.from_numpy(synth.iq3s_grid().view(np.uint8).reshape(512, 4).astype(np.int64)).to(dev)
        k = torch.arange(8, device=dev)
        idx = at(2, 64).reshape(R, B, 8, 8) | (((at(66, 8)[..., None] >> k) & 1) << 8)
        sg = _signs(at(74, 32), 8).reshape(R, B, 8, 8, 4)
        nib = torch.stack([at(106, 4) & 15, at(106, 4) >> 4], -1).reshape(R, B, 8)
        db = half(0)[..., None] * (1 + 2 * nib)
        return (db[..., None, None] * (table[idx] * sg)).reshape(R, -1)
    table = torch.from_numpy(_grid(t).astype(np.int64)).to(dev)
    if t == 18:
        a = at(66, 32).reshape(R, B, 8, 4)
        aux = a[..., 0] | (a[..., 1] << 8) | (a[..., 2] << 16) | (a[..., 3] << 24)
        i7 = (aux[..., None] >> (7 * torch.arange(4, device=dev))) & 127
        low = _signs(i7, 7)
        sg = torch.cat([low, low.prod(-1, keepdim=True)], -1).reshape(R, B, 8, 8, 4)
        db = half(0)[..., None] * (0.5 + (aux >> 28)) * 0.5
        return (db[..., None, None] * (table[at(2, 64).reshape(R, B, 8, 8)] * sg)).reshape(R, -1)
    hi = (at(66, 8)[..., None] >> (2 * torch.arange(4, device=dev))) & 3
    idx = at(2, 32).reshape(R, B, 8, 4) | (hi << 8)
    sg = _signs(at(34, 32), 8).reshape(R, B, 8, 4, 8)
    nib = torch.stack([at(74, 8) & 15, at(74, 8) >> 4], -1)
    db = (half(0)[..., None, None] * (0.5 + nib) * 0.25).repeat_interleave(2, dim=-1)
    return (db[..., None] * (table[idx] * sg)).reshape(R, -1)


def _product(t, raw, x):
    """x @ W^T in float64, a slab of rows at a time: [M, N]."""
    N, K = raw.shape[0], x.shape[1]
    step = max(1, (1 << 24) // K)
    x = x.to(torch.float64)
    return torch.cat([x @ _dequantize(t, raw[r:r + step]).T.contiguous() for r in range(0, N, step)], 1)


def exact(case, seed):
    c = case
    if c["kind"] == "decode":
        return None  # a whole model: its layers are the other cases
    if c["kind"] == "step":
        g, shapes, xs = _step_inputs(c, seed)
        return torch.cat([_product(mi355x.Q4_0, _raw_weights(mi355x.Q4_0, n, K, g), xs[K][None])[0]
                          for K, ns in shapes for n in ns])
    t, _, _, raw, x = _matrix_inputs(c, seed)
    y = _product(t, raw, x)
    return y[0] if c["kind"] == "gemv" else y
