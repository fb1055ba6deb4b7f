"""The forms of the elementwise, RMSNorm and RoPE operators for prompts (chunks
of 8 values, a wave per row, angles shared over the heads) against the general
forms, which the same entry points take for small or unaligned calls and which
tests/test_gpu_ops.py holds to the oracle: the same bits.
"""
import numpy as np
import pytest

from vvllm_amd import capi

pytestmark = pytest.mark.gpu

F16, F32 = capi.F16, capi.F32


def npd(d):
    return np.float32 if d == F32 else np.float16


@pytest.mark.parametrize("d", [F32, F16])
@pytest.mark.parametrize("n", [1 << 21, (1 << 21) + 7, (1 << 21) + 2040, 2999983])
@pytest.mark.parametrize("op", [capi.OP_ADD, capi.OP_MUL, capi.OP_SILU_MUL])
def test_eltwise_chunks(gpu, op, n, d):
    print(f"[case] eltwise chunks op={op} n={n} dtype={d}", flush=True)
    rng = np.random.default_rng(n + op)
    es = np.dtype(npd(d)).itemsize
    x, y = (rng.normal(0, 3, n + 1).astype(npd(d)) for _ in range(2))
    x[:4], y[:4] = [np.inf, -np.inf, np.nan, 0], [1, 2, 3, np.nan]
    dx, dy = capi.DevBuf.from_array(x), capi.DevBuf.from_array(y)
    outs = []
    for off in (0, es):  # 16-byte aligned, and not: out[i] of both is op(x[i], y[i])
        do = capi.DevBuf((n + 1) * es)
        if off:  # the same values, one element on
            ux, uy = (capi.DevBuf.from_array(np.concatenate([a[:1], a[:n]])) for a in (x, y))
            capi.call("vvh_eltwise", op, do.addr(es), ux.addr(es), uy.addr(es), n, d, None)
        else:
            capi.call("vvh_eltwise", op, do.ptr, dx.ptr, dy.ptr, n, d, None)
        capi.sync()
        outs.append(do.to_array(npd(d), (n + 1,))[1:] if off else do.to_array(npd(d), (n + 1,))[:n])
    assert np.array_equal(outs[0], outs[1], equal_nan=True)
    if op == capi.OP_SILU_MUL:  # in place, as a prefill MLP calls it
        capi.call("vvh_eltwise", op, dx.ptr, dx.ptr, dy.ptr, n, d, None)
        capi.sync()
        assert np.array_equal(dx.to_array(npd(d), (n + 1,))[:n], outs[0], equal_nan=True)


@pytest.mark.parametrize("d", [F32, F16])
@pytest.mark.parametrize("rows,n", [(512, 896), (513, 1536), (515, 2048), (600, 8), (1023, 520)])
def test_rms_norm_rows(gpu, rows, n, d):
    print(f"[case] rms rows={rows} n={n} dtype={d}", flush=True)
    rng = np.random.default_rng(rows + n)
    es = np.dtype(npd(d)).itemsize
    x = rng.normal(0, 1, (rows, n)).astype(npd(d))
    x[3, 2] = np.inf
    x[5] = 0
    dx, dw = capi.DevBuf.from_array(x), capi.DevBuf.from_array(rng.normal(1, 0.1, n).astype(np.float32))
    do, dr = capi.DevBuf(rows * n * es), capi.DevBuf(rows * n * es)
    capi.call("vvh_rms_norm", do.ptr, dx.ptr, dw.ptr, rows, n, 1e-6, d, None)
    for r in range(0, rows, 100):  # 100 rows at a time: a block per row
        m = min(100, rows - r)
        capi.call("vvh_rms_norm", dr.addr(r * n * es), dx.addr(r * n * es), dw.ptr, m, n, 1e-6, d, None)
    capi.sync()
    assert np.array_equal(do.to_array(npd(d), (rows, n)), dr.to_array(npd(d), (rows, n)), equal_nan=True)


@pytest.mark.parametrize("d", [F32, F16])
@pytest.mark.parametrize("append", [False, True])
@pytest.mark.parametrize("S,H,KVH,D,pos", [(401, 14, 2, 64, 0), (225, 12, 2, 128, 1000), (4200, 3, 3, 16, 7),
                                           (263, 5, 1, 256, 30000), (261, 2, 1, 512, 3), (3127, 0, 2, 64, 5),
                                           (6251, 1, 1, 32, 0)])
def test_rope_rows(gpu, S, H, KVH, D, pos, append, d):
    print(f"[case] rope rows S={S} H={H} KVH={KVH} D={D} pos={pos} append={append} dtype={d}", flush=True)
    rng = np.random.default_rng(S + D)
    es = np.dtype(npd(d)).itemsize
    q, k, v = (rng.normal(0, 1, (S, n, D)).astype(npd(d)) for n in (H, KVH, KVH))
    got = []
    for step in (S, 199):  # all positions in one call; 199 at a time, a thread per pair
        dq, dk, dv = (capi.DevBuf.from_array(a) for a in (q, k, v))
        kc, vc = (capi.DevBuf.from_array(np.zeros((pos + S, KVH, D), npd(d))) for _ in range(2))
        for s in range(0, S, step):
            m = min(step, S - s)
            a = (dq.addr(s * H * D * es) if H else None, dk.addr(s * KVH * D * es))
            if append:
                capi.call("vvh_rope_append", *a, dv.addr(s * KVH * D * es), kc.ptr, vc.ptr, m, H, KVH, D, pos + s, 1e6,
                          d, None)
            else:
                capi.call("vvh_rope", *a, m, H, KVH, D, pos + s, 1e6, d, None)
        capi.sync()
        got.append([b.to_array(npd(d), sh) for b, sh in ((dq, q.shape), (dk, k.shape), (kc, (pos + S, KVH, D)),
                                                        (vc, (pos + S, KVH, D)))])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
