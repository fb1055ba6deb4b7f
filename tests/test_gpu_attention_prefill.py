"""vvh_attention of several queries on the matrix cores (head_dim 64 and 128)
against causal attention in 64 bits (backend_naive.cc:344-378), at the edges of
its tiles: rows of 32 and 64 (query, head) pairs, stages of 64 and 128 keys, one
query more or less than they hold, keys split over blocks or not.

Tolerance per element: the output's rounding (fp16: half an ulp, 2^-11 of the
value), plus the scores' fp32 sums (|score| up to about 8, so 2e-6 of each
weight) and the weights' 22 bits or more, together below 1e-5 of the largest
|v|.
"""
import time

import numpy as np
import pytest

from vvllm_amd import capi

pytestmark = pytest.mark.gpu

F16, F32 = capi.F16, capi.F32
ULP = {F16: 2.0 ** -11, F32: 0.0}


def npd(d):
    return np.float32 if d == F32 else np.float16


def reference(q, k, v, len0, scale):
    n_q, H, D = q.shape
    T, KVH, _ = k.shape
    out = np.empty((n_q, H, D))
    seen = np.arange(T)[None, :] < len0 + np.arange(n_q)[:, None]
    for h in range(H):
        kh, vh = k[:, h // (H // KVH)].astype(np.float64), v[:, h // (H // KVH)].astype(np.float64)
        s = np.where(seen, q[:, h].astype(np.float64) @ kh.T * scale, -np.inf)
        p = np.exp(s - s.max(axis=1, keepdims=True))
        out[:, h] = (p / p.sum(axis=1, keepdims=True)) @ vh
    return out


def run(q, k, v, len0, scale, d):
    n_q, H, D = q.shape
    dq, dk, dv = (capi.DevBuf.from_array(a) for a in (q, k, v))
    do = capi.DevBuf(q.nbytes)
    capi.call("vvh_attention", do.ptr, dq.ptr, dk.ptr, dv.ptr, n_q, len0, H, k.shape[1], D, scale, d, None)
    capi.sync()
    return do.to_array(npd(d), (n_q, H, D)).astype(np.float64)


def draw(n_q, len0, H, KVH, D, d):
    rng = np.random.default_rng(n_q * 1000 + len0 + H)
    T = len0 + n_q - 1
    return (rng.normal(0, 2, (n_q, H, D)).astype(npd(d)), rng.normal(0, 1, (T, KVH, D)).astype(npd(d)),
            rng.normal(0, 1, (T, KVH, D)).astype(npd(d)), float(1 / np.sqrt(D)))


# G = H / KVH rows per query
CASES = [(2, 1, 14, 2, 64), (5, 1, 7, 1, 64), (33, 1, 1, 1, 64), (31, 97, 2, 2, 128), (64, 1, 12, 2, 128),
         (65, 64, 12, 2, 128), (129, 1, 8, 8, 64), (512, 1, 14, 2, 64), (7, 3000, 12, 2, 128), (3, 900, 40, 2, 64),
         (700, 200, 12, 2, 128), (1025, 1, 64, 8, 64), (1100, 60, 64, 8, 128)]


@pytest.mark.parametrize("d", [F32, F16])
@pytest.mark.parametrize("n_q,len0,H,KVH,D", CASES)
def test_prefill(gpu, n_q, len0, H, KVH, D, d):
    print(f"[case] prefill attention n_q={n_q} len0={len0} H={H} KVH={KVH} D={D} dtype={d}", flush=True)
    q, k, v, scale = draw(n_q, len0, H, KVH, D, d)
    got, ref = run(q, k, v, len0, scale, d), reference(q, k, v, len0, scale)
    assert (np.abs(got - ref) <= ULP[d] * np.abs(ref) + 1e-5 * np.abs(v).max()).all()


@pytest.mark.parametrize("n_q,len0,H,KVH,D", [(40, 3, 6, 2, 64), (70, 30, 12, 2, 128), (1100, 1, 64, 8, 64)])
@pytest.mark.parametrize("d", [F32, F16])
@pytest.mark.parametrize("bad", [np.inf, np.nan, 65504.0])
def test_prefill_unseen_rows(gpu, n_q, len0, H, KVH, D, d, bad):
    """A query's result does not depend on keys and values past its last
    visible position, whatever they hold; queries that see them carry them."""
    print(f"[case] unseen rows n_q={n_q} len0={len0} D={D} dtype={d} bad={bad}", flush=True)
    q, k, v, scale = draw(n_q, len0, H, KVH, D, d)
    t = len0 + n_q - 4  # visible to the last three queries only
    v[t, KVH - 1, 5] = bad
    k[t + 1, 0, 3] = bad
    got = run(q, k, v, len0, scale, d)
    clean_k, clean_v = k.copy(), v.copy()
    clean_v[t, KVH - 1, 5] = clean_k[t + 1, 0, 3] = 0
    ref = reference(q, clean_k, clean_v, len0, scale)
    early = slice(0, n_q - 3)
    assert (np.abs(got - ref)[early] <= ULP[d] * np.abs(ref)[early] + 1e-5 * np.abs(clean_v).max()).all()
    if not np.isfinite(bad):
        assert not np.isfinite(got[n_q - 3:, H - 1, 5]).any()


@pytest.mark.parametrize("n_q,len0,H,KVH,D,bound", [(333, 1, 14, 2, 64, 3.5e-7), (300, 67, 8, 8, 64, 4.2e-7),
                                                    (500, 1, 12, 2, 128, 5.5e-7), (126, 20, 8, 1, 128, 4.6e-7)])
def test_prefill_f32_error(gpu, n_q, len0, H, KVH, D, bound):
    """fp32 attention is closer to 64 bits (2-norm) than one block per head and
    query with a chain of head_dim products per score.  At these sizes 4.26e-7,
    5.14e-7, 6.45e-7 and 5.76e-7 in one chain per score and per lane's weights
    (that form: 0 to 3% less), 2.79e-7, 3.31e-7, 4.01e-7 and 3.52e-7 in two
    chains and with the weights summed by stages."""
    print(f"[case] fp32 error n_q={n_q} len0={len0} H={H} D={D}", flush=True)
    q, k, v, scale = draw(n_q, len0, H, KVH, D, F32)
    got, ref = run(q, k, v, len0, scale, F32), reference(q, k, v, len0, scale)
    e = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    print(f"error {e:.3e}")
    assert e <= bound


@pytest.mark.parametrize("n_q,len0,H,KVH,D", [(40, 1, 14, 2, 64), (700, 1, 12, 2, 128), (33, 3000, 12, 2, 128)])
@pytest.mark.parametrize("d", [F32, F16])
@pytest.mark.parametrize("gap", [12, 18, 22, 26])
def test_prefill_small_weights(gpu, n_q, len0, H, KVH, D, d, gap):
    """The keys a row attends to under a few with 2^gap times their weight and
    values of 0 (an attention sink) make up its whole output, so each weight
    has to keep its bits however far below the largest it is.  A key group of
    the tiles takes 32 keys at a time: one such key in each.  Per element, next
    to the output's rounding: scores of up to 26 in log2 units, summed in fp32
    (2e-5 of the value), and for fp16, weights in steps of 2^-34 of the largest
    (half of one for each key).
    """
    print(f"[case] small weights n_q={n_q} len0={len0} D={D} dtype={d} gap={gap}", flush=True)
    rng = np.random.default_rng(gap)
    T, scale = len0 + n_q - 1, float(1 / np.sqrt(D))
    q, k, v = np.zeros((n_q, H, D)), np.zeros((T, KVH, D)), rng.uniform(500, 1500, (T, KVH, D))
    q[..., 0] = 8.0
    sinks = [t for t in (0, 32, 64, 96) if t < T]
    k[sinks, :, 0], v[sinks] = gap / (8.0 * scale * np.log2(np.e)), 0.0
    q, k, v = (a.astype(npd(d)) for a in (q, k, v))
    got, ref = run(q, k, v, len0, scale, d), reference(q, k, v, len0, scale)
    tol = (ULP[d] + 2e-5) * np.abs(ref) + (2.0 ** -25 + T * 2.0 ** -35 * 1500.0 if d == F16 else 0.0)
    assert (np.abs(got - ref) <= tol).all()


NONFINITE = [(40, 3, 6, 2, 64), (90, 30, 12, 2, 128), (7, 700, 12, 2, 128), (500, 1, 14, 2, 64)]


@pytest.mark.parametrize("n_q,len0,H,KVH,D", NONFINITE)
@pytest.mark.parametrize("d", [F32, F16])
@pytest.mark.parametrize("where", ["v inf", "v nan", "k inf", "k nan", "v -inf and inf"])
@pytest.mark.parametrize("in_place", [False, True])
def test_prefill_nonfinite_rows(gpu, n_q, len0, H, KVH, D, d, where, in_place):
    """Queries that see a key or value that is not finite get what the sums
    give, infinities, NaN and the finite rest alike, also where out is q."""
    print(f"[case] nonfinite n_q={n_q} len0={len0} D={D} dtype={d} {where} in_place={in_place}", flush=True)
    q, k, v, scale = draw(n_q, len0, H, KVH, D, d)
    t = len0 // 2 + n_q // 3  # the queries from here on see it
    if where.startswith("v"):
        v[t, KVH - 1, 5] = {"inf": np.inf, "nan": np.nan, "-inf": -np.inf}[where.split()[1]]
        if "and" in where:
            v[t + 1, KVH - 1, 5], v[t, 0, 1] = np.inf, -np.inf
    else:
        k[t, KVH - 1] = np.inf if where == "k inf" else np.nan
        k[t, KVH - 1, 1:] = 0 if where == "k inf" else 1
    with np.errstate(invalid="ignore", over="ignore"):
        ref = reference(q, k, np.where(np.isfinite(v), v, 0), len0, scale)
        for s in range(n_q):  # dim 5 of kv head KVH - 1 (and dim 1 of kv head 0): sums of its values
            for kvh, dim in ((KVH - 1, 5), (0, 1)):
                seen = v[:len0 + s, kvh, dim].astype(np.float64)
                if not np.isfinite(seen).all():
                    ref[s, kvh * (H // KVH):(kvh + 1) * (H // KVH), dim] = seen[~np.isfinite(seen)].sum()
    if in_place:
        b = [capi.DevBuf.from_array(a) for a in (q, k, v)]
        capi.call("vvh_attention", b[0].ptr, b[0].ptr, b[1].ptr, b[2].ptr, n_q, len0, H, KVH, D, scale, d, None)
        capi.sync()
        got = b[0].to_array(npd(d), (n_q, H, D)).astype(np.float64)
    else:
        got = run(q, k, v, len0, scale, d)
    fin = np.isfinite(ref)
    assert fin.any() and not fin.all()
    assert np.array_equal(got[~fin], ref[~fin], equal_nan=True)
    vmax = np.abs(v[np.isfinite(v)]).max()
    assert (np.abs(got[fin] - ref[fin]) <= ULP[d] * np.abs(ref[fin]) + 1e-5 * vmax).all()


@pytest.mark.parametrize("d", [F32, F16])
@pytest.mark.parametrize("n_q,len0,H,KVH,D,ms", [(512, 1, 14, 2, 64, 0.6), (7, 4000, 12, 2, 128, 1.2)])
def test_prefill_nonfinite_time(gpu, n_q, len0, H, KVH, D, d, ms):
    """An infinity that every query sees does not leave the rows to one wave
    each (2.4 ms and more at these sizes; 0.07 to 0.5 with a block per row)."""
    q, k, v, scale = draw(n_q, len0, H, KVH, D, d)
    v[0] = np.inf
    b = [capi.DevBuf.from_array(a) for a in (q, k, v)] + [capi.DevBuf(q.nbytes)]
    best = np.inf
    for _ in range(5):
        t0 = time.perf_counter()
        capi.call("vvh_attention", b[3].ptr, b[0].ptr, b[1].ptr, b[2].ptr, n_q, len0, H, KVH, D, scale, d, None)
        capi.sync()
        best = min(best, time.perf_counter() - t0)
    print(f"error {best * 1e3:.3f} ms")
    assert best * 1e3 < ms
