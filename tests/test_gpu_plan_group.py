"""Plans that run as one grouped launch: problems that share their activations
on the GEMM (q/k/v, gate and up of a prompt; fp16, and fp32 split into fp16
halves once), and fp32 decode problems.  Against 64-bit sums, at group sizes
2-4, column counts that are no multiple of a tile or of 8, row counts at the
edges of the tiles and of the dispatch, k split or not.  (Captured and
replayed: test_gpu_capture_first.py.)

Tolerance per element: one rounding to the output type, the fp32 sums (no
product passes through more than K / 8 additions of partial sums of at most
sum |x w|, scaled), and for split fp32 activations 2^-21 of each |x w|.
"""
import ctypes

import numpy as np
import pytest

from vvllm_amd import capi

pytestmark = pytest.mark.gpu

F16, F32 = capi.F16, capi.F32


def npd(d):
    return np.float32 if d == F32 else np.float16


def build(rng, M, Ns, K, d, same_x=True, outlier=0.0, bare=False):
    dev, probs, refs = [], [], []
    x = rng.normal(0, 1, (M, K)).astype(npd(d))
    if outlier:
        x[:, K // 2] = outlier
    dx = capi.DevBuf.from_array(x)
    for i, N in enumerate(Ns):
        q = rng.integers(-127, 128, (N, K)).astype(np.int8)
        if outlier:
            q[:, K // 2] = 0
        s = rng.uniform(1e-4, 3e-4, N).astype(np.float32)
        b = rng.normal(0, 1, N).astype(np.float32) if i % 2 == 0 and not bare else None
        r = rng.normal(0, 1, (M, N)).astype(npd(d)) if i == 1 and not bare else None
        xi, dxi = (x, dx) if same_x else (lambda a: (a, capi.DevBuf.from_array(a)))(rng.normal(0, 1, (M, K)).astype(npd(d)))
        do = capi.DevBuf(M * N * x.itemsize)
        bufs = [capi.DevBuf.from_array(a) if a is not None else None for a in (q, s, b, r)]
        dev += bufs + [do, dxi]
        p = [t.ptr if t is not None else None for t in bufs]
        probs.append(capi.Q8Problem(out=do.ptr, inp=dxi.ptr, residual=p[3], weight=p[0], scales=p[1], bias=p[2], M=M, N=N,
                                    K=K))
        w = q.astype(np.float64) * s[:, None].astype(np.float64)
        y, mag = xi.astype(np.float64) @ w.T, np.abs(xi).astype(np.float64) @ np.abs(w).T
        for t in (b, r):
            if t is not None:
                y, mag = y + t, mag + np.abs(t)
        refs.append((do, y, mag))
    h = ctypes.c_uint64()
    capi.call("vvh_plan_create", (capi.Q8Problem * len(Ns))(*probs), len(Ns), d, d, ctypes.byref(h))
    return h.value, refs, dev


def check(refs, M, K, d):
    for do, y, mag in refs:
        got = do.to_array(npd(d), y.shape).astype(np.float64)
        ulp = 2.0 ** -11 if d == F16 else 2.0 ** -24
        assert (np.abs(got - y) <= ulp * np.abs(y) + (K / 8 * 2.0 ** -24 + (2.0 ** -21 if d == F32 else 0)) * mag).all()


def launches(plan):
    n = ctypes.c_int()
    capi.call("vvh_plan_launches", plan, ctypes.byref(n))
    return n.value


GEMM = [(17, (896, 128, 128), 896), (33, (200, 72), 512), (64, (256, 256, 1536), 1536), (130, (100, 129, 64, 1000), 576),
        (333, (896, 128, 128), 896), (512, (4864, 4864), 896), (700, (1536, 256, 256), 1536), (1500, (8960, 8960), 256),
        (40, (128, 64), 8960)]


@pytest.mark.parametrize("d", [F32, F16])
@pytest.mark.parametrize("M,Ns,K", GEMM)
def test_gemm_group(gpu, M, Ns, K, d):
    print(f"[case] gemm group M={M} N={Ns} K={K} dtype={d}", flush=True)
    plan, refs, dev = build(np.random.default_rng(M + K), M, Ns, K, d)
    assert launches(plan) == 1
    for _ in range(2):
        capi.call("vvh_plan_run", plan, None)
    capi.sync()
    check(refs, M, K, d)
    capi.call("vvh_plan_destroy", plan)


@pytest.mark.parametrize("M,Ns,K,same_x", [(1, (896, 128, 128), 896, True), (1, (4864, 4864), 896, False),
                                           (2, (100, 17, 16, 33), 4864, False), (15, (896, 128), 1000 - 8, True),
                                           (20, (64, 48), 208, True)])
def test_gemv_f32_group(gpu, M, Ns, K, same_x):
    print(f"[case] gemv group M={M} N={Ns} K={K}", flush=True)
    plan, refs, dev = build(np.random.default_rng(M + K), M, Ns, K, F32, same_x)
    assert launches(plan) == 1
    capi.call("vvh_plan_run", plan, None)
    capi.sync()
    check(refs, M, K, F32)
    capi.call("vvh_plan_destroy", plan)


@pytest.mark.parametrize("M,N,K", [(1, 33, 16), (2, 896, 4864), (3, 1000, 144), (4, 17, 8960), (5, 1536, 1536),
                                   (7, 50, 4096), (8, 9728, 896), (15, 130, 1024), (9, 260, 560), (3, 64, 4160)])
def test_f32_few_rows(gpu, M, N, K):
    print(f"[case] f32 few rows M={M} N={N} K={K}", flush=True)
    plan, refs, dev = build(np.random.default_rng(M + K), M, (N, N), K, F32, same_x=False)  # one by one, or k_gemv_f32
    capi.call("vvh_plan_run", plan, None)
    capi.sync()
    check(refs, M, K, F32)
    capi.call("vvh_plan_destroy", plan)


@pytest.mark.parametrize("M,Ns,K", [(3, (896, 128), 4864), (5, (1536, 256, 256), 1536), (6, (4864, 4864), 896),
                                    (15, (896, 128, 128), 4096), (8, (130,), 8960), (4, (9000, 9000), 1152)])
def test_f32_few_rows_keep_small_activations(gpu, M, Ns, K):
    """Fewer than 16 fp32 rows are used as they are: an activation 2^36 times
    the others, under codes of 0, costs the others no bits."""
    print(f"[case] f32 few rows, one large activation M={M} N={Ns} K={K}", flush=True)
    plan, refs, dev = build(np.random.default_rng(M + K), M, Ns, K, F32, outlier=2.0 ** 36)
    capi.call("vvh_plan_run", plan, None)
    capi.sync()
    check(refs, M, K, F32)
    capi.call("vvh_plan_destroy", plan)
    for N in Ns:
        assert capi.kernel_choice(M, N, K, F32, F32) == "gemv_f32"


@pytest.mark.parametrize("M,Ns,K", [(100, (896, 128, 128), 896), (64, (1536, 256, 256), 1536), (39, (1362, 1362), 512),
                                    (333, (896, 128, 128), 896), (16, (256, 256), 8960)])
def test_f32_group_error(gpu, M, Ns, K):
    """A plan's fp32 sums are as close to 64 bits as those of its problems one by
    one, which few columns split over k into chains of a few stages (0.9e-7 to
    1.26e-7 of the result, 2-norm, at these sizes; in chains of 8 stages 1.17e-7
    to 1.35e-7).  With a fold every 2 stages 0.8e-7 to 1.08e-7."""
    print(f"[case] gemm group error M={M} N={Ns} K={K}", flush=True)
    plan, refs, dev = build(np.random.default_rng(M + K), M, Ns, K, F32, bare=True)
    capi.call("vvh_plan_run", plan, None)
    capi.sync()
    for do, y, mag in refs:
        got = do.to_array(np.float32, y.shape).astype(np.float64)
        e = np.linalg.norm(got - y) / np.linalg.norm(y)
        print(f"error {e:.3e}")
        assert e <= (1.14e-7 if K == 8960 else 1.03e-7)
    capi.call("vvh_plan_destroy", plan)


@pytest.mark.parametrize("M,Ns,K", [(59, (1600, 64, 384), 960), (847, (448, 256, 64), 1728), (41, (1362, 1362), 512)])
def test_fp16_to_fp32_runs_one_by_one(gpu, M, Ns, K):
    """fp16 activations with fp32 outputs keep the sums, and the bits, of a
    problem alone: a group's fewer k splits would show in 32 bits."""
    print(f"[case] fp16 to fp32 M={M} N={Ns} K={K}", flush=True)
    rng = np.random.default_rng(M)
    dx = capi.DevBuf.from_array(rng.normal(0, 1, (M, K)).astype(np.float16))
    dev = [(capi.DevBuf.from_array(rng.integers(-127, 128, (N, K)).astype(np.int8)),
            capi.DevBuf.from_array(rng.uniform(1e-4, 3e-4, N).astype(np.float32)), capi.DevBuf(M * N * 4), capi.DevBuf(M * N * 4))
           for N in Ns]
    probs = [capi.Q8Problem(out=o.ptr, inp=dx.ptr, residual=None, weight=q.ptr, scales=s.ptr, bias=None, M=M, N=N, K=K)
             for (q, s, o, _), N in zip(dev, Ns)]
    h = ctypes.c_uint64()
    capi.call("vvh_plan_create", (capi.Q8Problem * len(Ns))(*probs), len(Ns), F16, F32, ctypes.byref(h))
    assert launches(h.value) == len(Ns)
    capi.call("vvh_plan_run", h.value, None)
    for (q, s, _, o), N in zip(dev, Ns):
        capi.linear_q8_dev(o, dx, q, s, None, None, M, N, K, F16, F32)
    capi.sync()
    capi.call("vvh_plan_destroy", h.value)
    for (_, _, a, b), N in zip(dev, Ns):
        assert np.array_equal(a.to_array(np.float32, (M, N)), b.to_array(np.float32, (M, N)))


def test_different_inputs_run_one_by_one(gpu):
    plan, refs, dev = build(np.random.default_rng(9), 100, (128, 192), 512, F16, same_x=False)
    assert launches(plan) == 2
    capi.call("vvh_plan_run", plan, None)
    capi.sync()
    check(refs, 100, 512, F16)
    capi.call("vvh_plan_destroy", plan)
