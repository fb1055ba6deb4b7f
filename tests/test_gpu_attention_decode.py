"""vvh_attention of one query whose span is split over blocks, or over two chunks
per wave of one (fp16, head_dim 64 and 128), against attention in 64 bits
(backend_naive.cc:344-378): the shortest such spans, ends of chunks, both sides of
the lines between one block, a block per chunk and blocks of four waves, and spans
of several chunks per wave.

Tolerance per element: the output's rounding (half an ulp, 2^-11 of the value)
and the fp32 scores and sums and the weights' 22 bits, below 1e-5 of the
largest |v|.
"""
import numpy as np
import pytest

from vvllm_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,H,KVH,D", [(513, 14, 2, 64), (576, 1, 1, 128), (577, 32, 2, 64), (1023, 16, 16, 64),
                                       (1025, 16, 16, 128), (4096, 14, 2, 64), (4097, 14, 2, 64), (4096, 12, 4, 128),
                                       (4095, 20, 5, 128), (9000, 12, 2, 128), (20001, 7, 1, 64), (1400, 100, 50, 64),
                                       (1024, 14, 2, 64), (1025, 14, 2, 64), (1000, 256, 128, 64), (700, 129, 129, 64), (513, 12, 2, 128)])
def test_split_span(gpu, n, H, KVH, D):
    print(f"[case] decode attention n={n} H={H} KVH={KVH} D={D}", flush=True)
    rng = np.random.default_rng(n + H)
    q, k, v = (rng.normal(0, s, sh).astype(np.float16) for s, sh in ((2, (H, D)), (1, (n, KVH, D)), (1, (n, KVH, D))))
    ref = np.empty((H, D))
    for h in range(H):
        g = h // (H // KVH)
        s = k[:, g].astype(np.float64) @ q[h].astype(np.float64) / np.sqrt(D)
        p = np.exp(s - s.max())
        ref[h] = p @ v[:, g].astype(np.float64) / p.sum()
    dq, dk, dv, do = *(capi.DevBuf.from_array(a) for a in (q, k, v)), capi.DevBuf(q.nbytes)
    for _ in range(2):
        capi.call("vvh_attention", do.ptr, dq.ptr, dk.ptr, dv.ptr, 1, n, H, KVH, D, float(1 / np.sqrt(D)), capi.F16, None)
        got = do.to_array(np.float16, (H, D)).astype(np.float64)
        assert (np.abs(got - ref) <= 2.0 ** -11 * np.abs(ref) + 1e-5 * np.abs(v).max()).all()
