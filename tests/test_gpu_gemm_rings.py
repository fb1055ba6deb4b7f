"""k_gemm3's 128-row tiles with rings of 2 and 3 stages: every stage count
around the ring and its unrolled round (shorter than the ring, the tails, one
and two rounds), tiles wholly inside the problem and edge tiles, with bias and
with the residual separate or in place.  Small integers: every product and sum
is exact in fp32, so the output is the exact value rounded once.
"""
import numpy as np
import pytest

from vvllm_amd import capi

pytestmark = pytest.mark.gpu

F16, F32 = capi.F16, capi.F32


@pytest.mark.parametrize("M,N,variant", [(2100, 1104, "k_gemm3 128x128"), (1030, 2203, "k_gemm3 128x128"),
                                         (2048, 2304, "k_gemm3 128x192"), (1930, 2411, "k_gemm3 128x192")])
@pytest.mark.parametrize("outd", [F16, F32])
def test_ring_lengths(gpu, M, N, variant, outd):
    rng = np.random.default_rng(M + N)
    dt = np.float16 if outd == F16 else np.float32
    x = rng.integers(-8, 9, (M, 14 * 64)).astype(np.float16)
    q = rng.integers(-127, 128, (N, 14 * 64)).astype(np.int8)
    s = (2.0 ** rng.integers(-8, -5, N)).astype(np.float32)
    b = rng.integers(-50, 50, N).astype(np.float32)
    r = rng.integers(-50, 50, (M, N)).astype(dt)
    ds, db = capi.DevBuf.from_array(s), capi.DevBuf.from_array(b)
    y = np.zeros((M, N), np.float32)
    for n in range(1, 15):
        K = 64 * n
        print(f"[case] gemm ring M={M} N={N} K={K} out={outd}", flush=True)
        assert capi.gemm_variant(M, N, K) == variant
        y += x[:, K - 64:K].astype(np.float32) @ q[:, K - 64:K].T.astype(np.float32)
        dx, dq = capi.DevBuf.from_array(np.ascontiguousarray(x[:, :K])), capi.DevBuf.from_array(np.ascontiguousarray(q[:, :K]))
        dr = capi.DevBuf.from_array(r)
        do = dr if n % 2 else capi.DevBuf(M * N * r.itemsize)
        capi.call("vvh_linear_q8_dev", do.ptr, dx.ptr, dq.ptr, ds.ptr, db.ptr, dr.ptr, M, N, K, F16, outd, None)
        want = (y * s + b + r.astype(np.float32)).astype(dt)
        assert np.array_equal(do.to_array(dt, (M, N)), want), K
