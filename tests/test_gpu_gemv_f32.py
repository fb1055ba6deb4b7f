"""k_gemv_f32 (fp32 activations, fewer than 16 rows or K % 64 != 0) against
64-bit sums, alone and in a plan: every body of a pass (1, 2, 4, 6 and 8 rows,
and each as the last pass of a longer call), every depth of the weight ring
(2, 4 and 7 steps of 128 codes per wave), 1, 2 and 4 waves per tile of 16 channels
with tiles left over, fp32 and fp16 outputs, with bias and residual.

Tolerance per element: one rounding to the output type and the fp32 sums (no
product passes through more than K / 8 + 32 additions of partial sums of at most
sum |x w|: a lane adds 16 products of each 128, then 8 lanes and 4 waves).
"""
import ctypes

import numpy as np
import pytest

from vvllm_amd import capi

pytestmark = pytest.mark.gpu

F16, F32 = capi.F16, capi.F32


def run(rng, M, Ns, K, outd, plan):
    dt = np.float32 if outd == F32 else np.float16
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    dx = capi.DevBuf.from_array(x)
    probs, keep, refs = [], [dx], []
    for N in Ns:
        q, s = rng.integers(-127, 128, (N, K)).astype(np.int8), rng.uniform(1e-4, 3e-4, N).astype(np.float32)
        b, r = rng.normal(0, 1, N).astype(np.float32), rng.normal(0, 1, (M, N)).astype(dt)
        bufs = [capi.DevBuf.from_array(a) for a in (q, s, b, r)]
        out = capi.DevBuf(M * N * r.itemsize)
        keep += bufs + [out]
        probs.append(capi.Q8Problem(out=out.ptr, inp=dx.ptr, residual=bufs[3].ptr, weight=bufs[0].ptr, scales=bufs[1].ptr,
                                    bias=bufs[2].ptr, M=M, N=N, K=K))
        w = q.astype(np.float32).astype(np.float64)
        y = x.astype(np.float64) @ w.T * s + b + r
        mag = np.abs(x).astype(np.float64) @ np.abs(w).T * s + np.abs(b) + np.abs(r)
        refs.append((out, y, mag))
        assert capi.kernel_choice(M, N, K, F32, outd) == "gemv_f32"
    if plan:
        h = ctypes.c_uint64()
        capi.call("vvh_plan_create", (capi.Q8Problem * len(Ns))(*probs), len(Ns), F32, outd, ctypes.byref(h))
        capi.call("vvh_plan_run", h.value, None)
        capi.sync()
        capi.call("vvh_plan_destroy", h.value)
    else:
        for p in probs:
            capi.linear_q8_dev(p.out, p.inp, p.weight, p.scales, p.bias, p.residual, M, p.N, K, F32, outd)
        capi.sync()
    ulp = 2.0 ** -24 if outd == F32 else 2.0 ** -11
    for out, y, mag in refs:
        got = out.to_array(dt, y.shape).astype(np.float64)
        assert (np.abs(got - y) <= ulp * np.abs(y) + (K / 8 + 32) * 2.0 ** -24 * mag).all()


@pytest.mark.parametrize("plan", [False, True])
@pytest.mark.parametrize("outd", [F32, F16])
@pytest.mark.parametrize("M,Ns,K", [
    (1, (17925, 16), 1536),     # 2 waves per tile, 6 steps each: the ring of 7
    (1, (33003, 20), 896),      # 1 wave per tile, 7 steps
    (1, (130, 100), 2816),      # 4 waves per tile, 6 steps
    (2, (17925, 16), 1536), (2, (33003, 17), 896), (1, (33003, 16400), 144),
    (3, (16421, 33), 528), (6, (16421, 33), 528), (5, (100, 4864), 896), (8, (17925,), 272),
    (9, (250, 60), 4864), (10, (250, 60), 1040), (12, (130, 17), 896), (14, (130, 17), 896), (15, (9728, 33), 896),
    (33, (130, 17), 272), (38, (130, 17), 1040),
])
def test_gemv_f32(gpu, M, Ns, K, outd, plan):
    print(f"[case] gemv f32 M={M} N={Ns} K={K} out={outd} plan={plan}", flush=True)
    run(np.random.default_rng(M * 7 + K), M, Ns, K, outd, plan)


def test_rows_of_the_largest_grid(gpu):
    """8 rows per pass and 65535 passes in a grid: one row more is refused by
    a plan as it is by a single call, before any launch."""
    print("[case] gemv f32 largest grid", flush=True)
    M, K, N = 8 * 65535, 16, 16
    rng = np.random.default_rng(3)
    x = rng.normal(0, 1, (M + 1, K)).astype(np.float32)
    q = rng.integers(-127, 128, (N, K)).astype(np.int8)
    dx, dq = capi.DevBuf.from_array(x), capi.DevBuf.from_array(q)
    ds = capi.DevBuf.from_array(np.ones(N, np.float32))
    outs = [capi.DevBuf((M + 1) * N * 4) for _ in range(2)]
    for rows in (M, M + 1):
        p = [capi.Q8Problem(out=o.ptr, inp=dx.ptr, residual=None, weight=dq.ptr, scales=ds.ptr, bias=None, M=rows, N=N, K=K)
             for o in outs]
        h = ctypes.c_uint64()
        capi.call("vvh_plan_create", (capi.Q8Problem * 2)(*p), 2, F32, F32, ctypes.byref(h))
        st = capi.status_of("vvh_plan_run", h.value, None)
        capi.sync()
        capi.call("vvh_plan_destroy", h.value)
        single = capi.status_of("vvh_linear_q8_dev", outs[0].ptr, dx.ptr, dq.ptr, ds.ptr, None, None, rows, N, K, F32, F32,
                                None)
        assert (capi.STATUS[st], st) == ("VVH_OK" if rows == M else "VVH_ERR_UNSUPPORTED", single)
        capi.sync()
    y, mag = x[:M].astype(np.float64) @ q.T.astype(np.float64), np.abs(x[:M]).astype(np.float64) @ np.abs(q.astype(np.float64)).T
    assert (np.abs(outs[1].to_array(np.float32, (M, N)) - y) <= 2.0 ** -24 * np.abs(y) + (K / 8 + 32) * 2.0 ** -24 * mag).all()
