"""A batched call recorded into a HIP graph shares nothing with the context's
later calls: the graph is replayed on another stream while the context runs
batched calls of its own, and both keep their results, bit for bit."""
import ctypes

import numpy as np
import pytest

import mi355x
import synth

pytestmark = pytest.mark.gpu

TYPES = {"Q4_0": 2, "Q4_K": 12, "Q6_K": 14, "IQ3_S": 21}


def hip_check(rc, what):
    assert rc == 0, f"{what}: hipError_t {rc}"


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("name", list(TYPES))
def test_replays_beside_the_contexts_calls(ctx, name, noalloc):
    t, N, K, M = TYPES[name], 1030, 2048, 40
    hip = ctypes.CDLL("libamdhip64.so")
    raw = synth.random_q4_0(N, K, 3) if t == 2 else synth.random_blocks(t, N, K, 3)
    w = ctx.resident(t, raw, N, K)
    xs = [np.stack([synth.activations(K, seed=1000 * i + m) for m in range(M)]) for i in range(2)]
    # what a call under capture runs: passes of 8 (Q4_0), one GEMV per activation
    if t == 2:
        ref = np.concatenate([ctx.gemv_batched(w, xs[0][a:a + 8]) for a in range(0, M, 8)])
    else:
        ref = np.stack([ctx.gemv(w, x) for x in xs[0]])
    own = ctx.gemv_batched(w, xs[1])
    xb, yb = [ctx.to_device(x) for x in xs], [ctx.alloc(4 * M * N) for _ in range(2)]
    fn = ctx.lib.mi355x_gemv_batched_noalloc if noalloc else ctx.lib.mi355x_gemv_batched
    stream = ctypes.c_void_p(ctx.lib.mi355x_ctx_stream(ctx.h))
    other, graph, ex = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    try:
        ctx.sync()
        hip_check(hip.hipStreamBeginCapture(stream, 1), "begin capture")
        rc = fn(ctx.h, t, w.ptr, N, K, xb[0].ptr, K, yb[0].ptr, N, M)
        hip_check(hip.hipStreamEndCapture(stream, ctypes.byref(graph)), "end capture")
        mi355x.check(rc)
        hip_check(hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)), "instantiate")
        hip_check(hip.hipStreamCreateWithFlags(ctypes.byref(other), 1), "stream")
        for _ in range(4):
            hip_check(hip.hipGraphLaunch(ex, other), "launch")
            for _ in range(3):
                mi355x.check(fn(ctx.h, t, w.ptr, N, K, xb[1].ptr, K, yb[1].ptr, N, M))
            ctx.sync()
            hip_check(hip.hipStreamSynchronize(other), "synchronize")
            assert np.array_equal(yb[0].download(np.float32, M * N).reshape(M, N), ref)
            assert np.array_equal(yb[1].download(np.float32, M * N).reshape(M, N), own)
            ctx.lib.mi355x_fill(ctx.h, yb[0].ptr, 0, 4 * M * N)
            ctx.sync()
    finally:
        if ex:
            hip.hipGraphExecDestroy(ex)
        if graph:
            hip.hipGraphDestroy(graph)
        if other:
            hip.hipStreamDestroy(other)
        for b in (*xb, *yb, w):
            b.free()
