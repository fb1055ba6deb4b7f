"""Calls that use the stream's workspace when they can have it and do without
otherwise: captured on a stream that never ran them (the capture may not
allocate), replayed between eager work, against the eager result on a stream
that has a workspace.  Attention and dense calls whose splits need it, fp32
linears of a few rows, and grouped plans whose k is split.
"""
import ctypes

import numpy as np
import pytest

from vvllm_amd import capi

pytestmark = pytest.mark.gpu

F16, F32 = capi.F16, capi.F32
V = ctypes.c_void_p


def hip():
    lib = ctypes.CDLL("libamdhip64.so.7")
    for name, args in {"hipStreamCreate": [ctypes.POINTER(V)], "hipStreamSynchronize": [V], "hipStreamDestroy": [V],
                       "hipStreamBeginCapture": [V, ctypes.c_int], "hipStreamEndCapture": [V, ctypes.POINTER(V)],
                       "hipGraphGetNodes": [V, V, ctypes.POINTER(ctypes.c_size_t)],
                       "hipGraphInstantiate": [ctypes.POINTER(V), V, V, V, ctypes.c_size_t],
                       "hipGraphLaunch": [V, V], "hipGraphExecDestroy": [V], "hipGraphDestroy": [V]}.items():
        getattr(lib, name).argtypes = args
    return lib


def buf(rng, shape, dt, std=1.0):
    return capi.DevBuf.from_array(rng.normal(0, std, shape).astype(dt))


def attention(rng, d, n_q, len0, H, KVH, D):
    dt = np.float16 if d == F16 else np.float32
    q, k, v = buf(rng, (n_q, H, D), dt), buf(rng, (len0 + n_q, KVH, D), dt), buf(rng, (len0 + n_q, KVH, D), dt)
    return (q, k, v), (n_q, H * D), dt, lambda o, s: capi.call(
        "vvh_attention", o.ptr, q.ptr, k.ptr, v.ptr, n_q, len0, H, KVH, D, float(1 / np.sqrt(D)), d, s)


def dense(rng, d, M, N, K):
    dt = np.float16 if d == F16 else np.float32
    x, w = buf(rng, (M, K), dt), buf(rng, (N, K), dt, 0.05)
    return (x, w), (M, N), dt, lambda o, s: capi.call("vvh_dense", o.ptr, x.ptr, w.ptr, d, None, None, M, N, K, d, s)


def linear(rng, M, N, K, plan, d=F32):
    dt = np.float16 if d == F16 else np.float32
    x = buf(rng, (M, K), dt)
    es = np.dtype(dt).itemsize
    q = capi.DevBuf.from_array(rng.integers(-127, 128, (N, K)).astype(np.int8))
    s = capi.DevBuf.from_array(rng.uniform(1e-4, 3e-4, N).astype(np.float32))

    def run(o, stream):
        if not plan:
            return capi.call("vvh_linear_q8_dev", o.ptr, x.ptr, q.ptr, s.ptr, None, None, M, N, K, d, d, stream)
        half = N // 2  # the two halves of the rows as a plan: its blocks of M x N / 2 outputs one after the other
        pr = [capi.Q8Problem(out=o.addr(i * M * half * es), inp=x.ptr, residual=None, weight=q.addr(i * half * K),
                             scales=s.addr(i * half * 4), bias=None, M=M, N=half, K=K) for i in range(2)]
        key = o.ptr
        if key not in plans:
            h = ctypes.c_uint64()
            capi.call("vvh_plan_create", (capi.Q8Problem * 2)(*pr), 2, d, d, ctypes.byref(h))
            plans[key] = h.value
        return capi.call("vvh_plan_run", plans[key], stream)
    plans = {}
    return (x, q, s, plans), (M, N), dt, run


CASES = {
    "attention_f16": lambda r: attention(r, F16, 7, 4000, 12, 2, 128),
    "attention_f32": lambda r: attention(r, F32, 9, 2000, 14, 2, 64),
    "dense_f16": lambda r: dense(r, F16, 64, 896, 4864),
    "dense_f32": lambda r: dense(r, F32, 128, 896, 4864),
    "linear_f32_few": lambda r: linear(r, 5, 1536, 1536, False),
    "plan_f16": lambda r: linear(r, 40, 256, 896, True, F16),
    "plan_f16_split": lambda r: linear(r, 128, 2048, 1536, True, F16),  # one by one its problems would split k too
    "plan_f32_decode": lambda r: linear(r, 3, 256, 4864, True),
}


@pytest.mark.parametrize("name", CASES)
def test_captured_without_a_workspace(gpu, name):
    print(f"[case] captured without a workspace: {name}", flush=True)
    lib = hip()
    keep, shape, dt, run = CASES[name](np.random.default_rng(len(name)))
    size = int(np.prod(shape)) * np.dtype(dt).itemsize
    want, got = capi.DevBuf(size), capi.DevBuf(size)
    run(want, None)
    capi.sync()
    ref = want.to_array(dt, shape).astype(np.float64)
    if name.startswith("plan"):  # the plan of the captured run exists before the capture
        run(got, None)
        capi.sync()
    stream, graph, ex = V(), V(), V()
    assert lib.hipStreamCreate(ctypes.byref(stream)) == 0
    capi.call("vvh_workspace_release", stream)
    assert lib.hipStreamBeginCapture(stream, 1) == 0  # thread-local: an allocation would fail
    run(got, stream)
    assert lib.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert lib.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, 0) == 0
    zero = np.zeros(shape, dt)
    for _ in range(3):
        capi.call("vvh_memcpy_h2d", got.ptr, zero.ctypes.data, size)
        run(want, None)
        capi.sync()
        assert lib.hipGraphLaunch(ex, stream) == 0 and lib.hipStreamSynchronize(stream) == 0
        y = got.to_array(dt, shape).astype(np.float64)
        # the same sums in another order: a rounding of the output, or fp32 sums of up to 5000 products
        tol = 2.0 ** -10 if dt == np.float16 else 2e-6
        assert np.linalg.norm(y - ref) <= tol * np.linalg.norm(ref)
    assert lib.hipGraphExecDestroy(ex) == 0 and lib.hipGraphDestroy(graph) == 0
    assert lib.hipStreamDestroy(stream) == 0


@pytest.mark.parametrize("name", ["attention_f16", "attention_f32", "dense_f16", "dense_f32", "dense_few_f32", "attention_short_f32"])
def test_graph_holds_no_workspace(gpu, name):
    """A captured vvh_dense, or vvh_attention of several queries, is one kernel
    off the stream's workspace, also where the stream has one: its graph may be
    replayed on another stream while the capturing one runs the same call, and
    after vvh_workspace_release."""
    print(f"[case] graph without workspace: {name}", flush=True)
    lib = hip()
    more = {"dense_few_f32": lambda r: dense(r, F32, 12, 896, 4864),  # these keep the forms without splits
            "attention_short_f32": lambda r: attention(r, F32, 8, 400, 12, 2, 128)}
    keep, shape, dt, run = {**CASES, **more}[name](np.random.default_rng(len(name)))
    size = int(np.prod(shape)) * np.dtype(dt).itemsize
    want, got = capi.DevBuf(size), capi.DevBuf(size)
    first, other, graph, ex = V(), V(), V(), V()
    assert lib.hipStreamCreate(ctypes.byref(first)) == 0 and lib.hipStreamCreate(ctypes.byref(other)) == 0
    run(want, first)  # the stream has a workspace of the call's size
    capi.sync()
    ref = want.to_array(dt, shape).astype(np.float64)
    assert lib.hipStreamBeginCapture(first, 1) == 0
    run(got, first)
    assert lib.hipStreamEndCapture(first, ctypes.byref(graph)) == 0
    n = ctypes.c_size_t()
    assert lib.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    assert n.value == 1  # a split call is two
    assert lib.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, 0) == 0
    zero = np.zeros(shape, dt)
    for released in (False, False, True, True):
        if released:
            capi.call("vvh_workspace_release", first)
        capi.call("vvh_memcpy_h2d", got.ptr, zero.ctypes.data, size)
        assert lib.hipGraphLaunch(ex, other) == 0
        if not released:
            run(want, first)
        assert lib.hipStreamSynchronize(other) == 0
        capi.sync()
        # the same sums in another order, as in test_captured_without_a_workspace
        tol = 2.0 ** -10 if dt == np.float16 else 2e-6
        assert np.linalg.norm(got.to_array(dt, shape).astype(np.float64) - ref) <= tol * np.linalg.norm(ref)
        assert np.array_equal(want.to_array(dt, shape).astype(np.float64), ref)
    assert lib.hipGraphExecDestroy(ex) == 0 and lib.hipGraphDestroy(graph) == 0
    assert lib.hipStreamDestroy(first) == 0 and lib.hipStreamDestroy(other) == 0


@pytest.mark.parametrize("d,M,N,K,nodes", [(F16, 40, 256, 896, 1), (F16, 128, 2048, 1536, 2), (F32, 64, 1024, 896, 3)])
def test_split_plan_in_a_graph(gpu, d, M, N, K, nodes):
    """A grouped plan whose k is split, captured on a stream that has the
    workspace: without it where its problems alone run on k_skinny (one kernel),
    with it (the split of fp32 activations, GEMM and reduction, the eager bits)
    where they would use it as well.  One by one they are twice as many."""
    print(f"[case] split plan in a graph dtype={d} M={M} N={N} K={K}", flush=True)
    lib = hip()
    keep, shape, dt, run = linear(np.random.default_rng(M), M, N, K, True, d)
    size = int(np.prod(shape)) * np.dtype(dt).itemsize
    want, got = capi.DevBuf(size), capi.DevBuf(size)
    stream, graph, ex = V(), V(), V()
    assert lib.hipStreamCreate(ctypes.byref(stream)) == 0
    run(want, stream)
    run(got, stream)
    capi.sync()
    ref = want.to_array(dt, shape)
    assert lib.hipStreamBeginCapture(stream, 1) == 0
    run(got, stream)
    assert lib.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    n = ctypes.c_size_t()
    assert lib.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    assert n.value == nodes
    assert lib.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, 0) == 0
    for _ in range(3):
        capi.call("vvh_memcpy_h2d", got.ptr, np.zeros(shape, dt).ctypes.data, size)
        run(want, stream)
        assert lib.hipGraphLaunch(ex, stream) == 0
        capi.sync()
        y = got.to_array(dt, shape)
        if nodes > 1:
            assert np.array_equal(y, ref)
        assert np.linalg.norm(y.astype(np.float64) - ref) <= 2.0 ** -10 * np.linalg.norm(ref.astype(np.float64))
    assert lib.hipGraphExecDestroy(ex) == 0 and lib.hipGraphDestroy(graph) == 0
    assert lib.hipStreamDestroy(stream) == 0


@pytest.mark.parametrize("name", ["dense_f16", "attention_f16", "plan_f16"])
def test_eager_call_next_to_a_global_capture(gpu, name):
    """A call whose first workspace is allocated while another stream is being
    captured in the global mode leaves that capture whole."""
    print(f"[case] eager next to a capture: {name}", flush=True)
    lib = hip()
    keep, shape, dt, run = CASES[name](np.random.default_rng(len(name)))
    size = int(np.prod(shape)) * np.dtype(dt).itemsize
    want, got, small = capi.DevBuf(size), capi.DevBuf(size), capi.DevBuf(4096)
    captured, eager, graph = V(), V(), V()
    assert lib.hipStreamCreate(ctypes.byref(captured)) == 0 and lib.hipStreamCreate(ctypes.byref(eager)) == 0
    run(want, eager)
    run(got, eager)  # a plan of `got` exists before the capture
    capi.sync()
    capi.call("vvh_workspace_release", eager)
    assert lib.hipStreamBeginCapture(captured, 0) == 0
    capi.call("vvh_eltwise", capi.OP_ADD, small.ptr, small.ptr, small.ptr, 1024, F32, captured)
    run(got, eager)
    assert lib.hipStreamEndCapture(captured, ctypes.byref(graph)) == 0
    capi.sync()
    assert np.array_equal(got.to_array(dt, shape), want.to_array(dt, shape))
    assert lib.hipGraphDestroy(graph) == 0
    assert lib.hipStreamDestroy(captured) == 0 and lib.hipStreamDestroy(eager) == 0


def test_decode_attention_in_a_smaller_workspace(gpu):
    """One query over 64 chunks of 64 keys takes a block per chunk, 2.2 MB of
    partials; captured on a stream whose workspace is the smallest (1 MiB), four
    chunks per block.  Against 64 bits: the output's rounding, scores summed in
    fp32 and weights of 11 bits or more."""
    lib = hip()
    H, KVH, D, n = 64, 4, 128, 4096
    rng = np.random.default_rng(4)
    q, k, v = (rng.normal(0, 1, s).astype(np.float16) for s in ((H, D), (n, KVH, D), (n, KVH, D)))
    dq, dk, dv = (capi.DevBuf.from_array(a) for a in (q, k, v))
    outs = [capi.DevBuf(H * D * 2) for _ in range(2)]
    x = capi.DevBuf.from_array(rng.normal(0, 1, 5000).astype(np.float32))
    i = capi.DevBuf(4)
    stream, graph, ex = V(), V(), V()
    run = lambda o, s: capi.call("vvh_attention", o.ptr, dq.ptr, dk.ptr, dv.ptr, 1, n, H, KVH, D, float(1 / np.sqrt(D)), F16, s)
    run(outs[0], None)
    assert lib.hipStreamCreate(ctypes.byref(stream)) == 0
    capi.call("vvh_argmax", x.ptr, 5000, i.ptr, stream)  # a workspace of the smallest size
    capi.sync()
    assert lib.hipStreamBeginCapture(stream, 1) == 0
    run(outs[1], stream)
    assert lib.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert lib.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, 0) == 0
    ref = np.empty((H, D))
    for h in range(H):
        kh, vh = k[:, h // (H // KVH)].astype(np.float64), v[:, h // (H // KVH)].astype(np.float64)
        s = kh @ q[h].astype(np.float64) / np.sqrt(D)
        p = np.exp(s - s.max())
        ref[h] = p / p.sum() @ vh
    for _ in range(3):
        capi.call("vvh_memcpy_h2d", outs[1].ptr, np.zeros((H, D), np.float16).ctypes.data, H * D * 2)
        assert lib.hipGraphLaunch(ex, stream) == 0
        capi.sync()
        for o in outs:
            got = o.to_array(np.float16, (H, D)).astype(np.float64)
            assert np.linalg.norm(got - ref) <= 2.0 ** -10 * np.linalg.norm(ref)
    assert not np.array_equal(*(o.to_array(np.float16, (H, D)) for o in outs))  # the two plans round apart
    assert lib.hipGraphExecDestroy(ex) == 0 and lib.hipGraphDestroy(graph) == 0
    assert lib.hipStreamDestroy(stream) == 0
