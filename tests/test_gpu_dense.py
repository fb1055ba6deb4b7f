"""vvh_dense on the matrix cores (more than 4 rows, fp16 or fp32 throughout)
against 64-bit products (backend_naive.cc:139-156, :302-320), at the edges of its
tiles (32 and 64 rows, 64 columns), k stages (64 fp16 or 32 fp32
values) and k splits.

Tolerance per element: one rounding to the output type, and the fp32 sums: no
product passes through more than 48 + K / 128 additions (fp16: K / 16 + 16),
each rounding a partial sum of at most sum |x w|.
"""
import numpy as np
import pytest

from vvllm_amd import capi

pytestmark = pytest.mark.gpu

F16, F32 = capi.F16, capi.F32


def npd(d):
    return np.float32 if d == F32 else np.float16


def reference(x, w, b, r):
    y = x.astype(np.float64) @ w.astype(np.float64).T
    mag = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T
    if b is not None:
        y, mag = y + b.astype(np.float64), mag + np.abs(b)
    if r is not None:
        y, mag = y + r.astype(np.float64), mag + np.abs(r.astype(np.float64))
    return y, mag


CASES = [(5, 64, 8), (9, 64, 8), (6, 70, 2052 * 4), (31, 63, 64), (32, 65, 72), (33, 130, 896), (64, 896, 4864), (65, 200, 2056), (128, 128, 32),
         (129, 1000, 1000), (5, 512, 512), (7, 1100, 896), (10, 1024, 1024), (300, 9728, 136), (512, 8200, 896), (7, 40, 4864), (100, 33, 8960),
         # both sides of the lines where a k split gives way to a wave per weight row (its longest chain, K / 64 + 6, is shorter here)
         (9, 130, 1968), (9, 130, 1984), (8, 100, 2672), (8, 100, 2688), (16, 70, 856), (16, 70, 872), (12, 2100, 640), (5, 4000, 1536)]


@pytest.mark.parametrize("d", [F32, F16])
@pytest.mark.parametrize("M,N,K", CASES)
@pytest.mark.parametrize("bias,res", [(False, False), (True, True)])
def test_dense_rows(gpu, M, N, K, bias, res, d):
    print(f"[case] dense M={M} N={N} K={K} bias={bias} res={res} dtype={d}", flush=True)
    rng = np.random.default_rng(M * N + K)
    x, w = rng.normal(0, 1, (M, K)).astype(npd(d)), rng.normal(0, 0.1, (N, K)).astype(npd(d))
    b = rng.normal(0, 1, N).astype(np.float32) if bias else None
    r = rng.normal(0, 1, (M, N)).astype(npd(d)) if res else None
    dx, dw = capi.DevBuf.from_array(x), capi.DevBuf.from_array(w)
    db = capi.DevBuf.from_array(b) if bias else None
    do = capi.DevBuf.from_array(r if res else np.zeros((M, N), npd(d)))  # the residual in place
    capi.call("vvh_dense", do.ptr, dx.ptr, dw.ptr, d, db.ptr if bias else None, do.ptr if res else None, M, N, K, d, None)
    capi.sync()
    y, mag = reference(x, w, b, r)
    got = do.to_array(npd(d), (M, N)).astype(np.float64)
    adds = K / 16 + 16 if d == F16 else 48 + K / 128
    assert (np.abs(got - y) <= (2.0 ** -11 if d == F16 else 2.0 ** -24) * np.abs(y) + adds * 2.0 ** -24 * mag).all()


@pytest.mark.parametrize("d", [F32, F16])
def test_dense_rows_nonfinite(gpu, d):
    """An infinity or NaN of one row or weight reaches that row's or column's
    outputs only, also past K's last whole stage and past M's last whole tile."""
    M, N, K = 70, 130, 1000
    rng = np.random.default_rng(5)
    x, w = rng.normal(0, 1, (M, K)).astype(npd(d)), rng.normal(0, 0.1, (N, K)).astype(npd(d))
    x[M - 1, K - 1], w[N - 1, K - 8] = np.inf, np.nan
    dx, dw, do = capi.DevBuf.from_array(x), capi.DevBuf.from_array(w), capi.DevBuf(M * N * x.itemsize)
    capi.call("vvh_dense", do.ptr, dx.ptr, dw.ptr, d, None, None, M, N, K, d, None)
    capi.sync()
    fin = np.isfinite(do.to_array(npd(d), (M, N)))
    assert not fin[M - 1].any() and not fin[:, N - 1].any() and fin[:M - 1, :N - 1].all()


@pytest.mark.parametrize("M,N,K,bound", [(200, 256, 256, 7.95e-8), (306, 1536, 432, 8.4e-8), (64, 512, 512, 8.4e-8),
                                         (128, 1000, 896, 8.7e-8)])
def test_dense_f32_error(gpu, M, N, K, bound):
    """Closer to 64 bits (2-norm) than a wave per weight row with 64 lanes and
    a butterfly: at these sizes 8.16e-8, 8.68e-8, 8.64e-8 and 8.93e-8 with the
    waves' sums added in 32 bits (the butterfly 1 to 2% less up to K = 512),
    7.63e-8, 8.20e-8, 8.17e-8 and 8.45e-8 in 64."""
    rng = np.random.default_rng(M + K)
    x, w = rng.normal(0, 1, (M, K)).astype(np.float32), rng.normal(0, 0.1, (N, K)).astype(np.float32)
    dx, dw, do = capi.DevBuf.from_array(x), capi.DevBuf.from_array(w), capi.DevBuf(M * N * 4)
    capi.call("vvh_dense", do.ptr, dx.ptr, dw.ptr, F32, None, None, M, N, K, F32, None)
    capi.sync()
    y = x.astype(np.float64) @ w.astype(np.float64).T
    e = np.linalg.norm(do.to_array(np.float32, (M, N)) - y) / np.linalg.norm(y)
    print(f"error {e:.3e}")
    assert e <= bound
