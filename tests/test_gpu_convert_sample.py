"""vvh_convert in 8-element chunks (remainders, aligned and not) and sampling at
the edges of its blocks: one block up to 2048 logits, then blocks of 512, from
2^18 logits on of 2048 and more, at most 1024 of them.  Conversions are exact or one rounding; the first index of the
maximum is exact.
"""
import numpy as np
import pytest

from vvllm_amd import capi

pytestmark = pytest.mark.gpu

F16, F32 = capi.F16, capi.F32
DT = {F16: np.float16, F32: np.float32}


@pytest.mark.parametrize("dst", [F16, F32])
@pytest.mark.parametrize("src", [F16, F32])
@pytest.mark.parametrize("n,off", [(1, 0), (7, 0), (8, 0), (2047, 0), (2049, 0), (151936, 0), (5000, 1), (5000, 8)])
def test_convert(gpu, n, off, src, dst):
    x = np.random.default_rng(n).normal(0, 100, n + off).astype(DT[src])
    x[n // 2 + off] = np.inf
    dx, do = capi.DevBuf.from_array(x), capi.DevBuf((n + 16) * DT[dst]().itemsize)
    guard = np.full(n + 16, 7, DT[dst])
    do = capi.DevBuf.from_array(guard)
    capi.call("vvh_convert", do.ptr, dst, dx.addr(off * x.itemsize), src, n, None)
    got = do.to_array(DT[dst], (n + 16,))
    assert np.array_equal(got[:n], x[off:].astype(DT[dst])) and (got[n:] == 7).all()


@pytest.mark.parametrize("d", [F16, F32])
@pytest.mark.parametrize("n", [1, 2048, 2049, 2560, 2561, 151936, 1 << 18, (1 << 18) + 1, 512 * 1024 + 1, (1 << 21) + 1])
def test_argmax_first_index(gpu, n, d):
    x = np.random.default_rng(n).integers(-100, 50, n).astype(DT[d])
    for at in ([0], [n - 1], [n // 3, n - 1], [min(n - 1, 511), min(n - 1, 512)]):
        y = x.copy()
        y[at] = 60
        dx, di = capi.DevBuf.from_array(y), capi.DevBuf(4)
        capi.call("vvh_sample", dx.ptr, d, n, 0.0, 1.0, 0, 0, di.ptr, None)
        assert di.to_array(np.int32, (1,))[0] == min(at)
