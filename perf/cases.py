"""Performance cases: what a program that serves or evaluates a Qwen2-shaped
model has this library do, call by call through the C ABI
(include/vvllm_hip.h), over the range of sizes such a program meets.

Kinds of case, each one pass of a program's work:

  linear     one int8 per-channel linear (vvh_linear_q8_dev)
  decode     one token through decoder layers with a filled KV cache: in fp16
             the fused sequence of vvllm_amd/qwen2_decode.py (plans with their
             input stages and epilogues), in fp32 the operators one by one; a
             whole step embeds the token first and ends in the int8 LM head
  prefill    a prompt, or the next piece of one, through one decoder layer
  attention  the causal attention of such a piece alone
  head       the dense LM head (tied embedding) of one token and the sampler
  dense      a dense linear of the model run without quantization

Sizes come from Qwen2.5-0.5B (hidden 896, 14 heads, 2 kv heads of 64, MLP 4864,
24 layers, vocabulary 151936) and the 1.5B shapes of bench.py (hidden 1536, 12
heads, 2 kv heads of 128, MLP 8960), or are generic.  Weights are N(0, 0.02)
quantized per output channel, biases N(0, 0.01), norm weights 1 + N(0, 0.1),
hidden rows and cache rows N(0, 1), as in bench.py and the tests.
"""
from __future__ import annotations

import ctypes
import math

import torch

from vvllm_amd import capi

EPS = 1e-6
THETA = 1e6
ATTN_PARTS_MAX_SPAN = 512  # longest span vvh_attention_parts takes
DEV = "cuda"

M05 = dict(hidden=896, heads=14, kv_heads=2, inter=4864)
M15 = dict(hidden=1536, heads=12, kv_heads=2, inter=8960)


def listed() -> list[dict]:
    return [
        # the smallest call of a decode step: one token's o projection, added to the residual
        dict(name="linear_o_decode", kind="linear", M=1, N=896, K=896, act="f16", bias=False, residual=True),
        # eight sequences decoded together: the wide gate/up projection
        dict(name="linear_gate_up_batch8", kind="linear", M=8, N=17920, K=1536, act="f16", bias=False, residual=False),
        # a ragged prompt's down projection, added to the residual
        dict(name="linear_down_prompt", kind="linear", M=1000, N=896, K=4864, act="f16", bias=False, residual=True),
        # one generated token of Qwen2.5-0.5B, embedding to logits, 512 positions of context
        dict(name="decode_step_f16", kind="decode", **M05, layers=24, vocab=151936, pos=511, act="f16"),
        # one layer of a token generated far into a long context, 1.5B shape
        dict(name="decode_layer_long_f16", kind="decode", **M15, layers=1, vocab=0, pos=4095, act="f16"),
        # one layer of a token in fp32, the reference's default mode
        dict(name="decode_layer_f32", kind="decode", **M05, layers=1, vocab=0, pos=300, act="f32"),
        # an ordinary prompt through one layer
        dict(name="prefill_layer_f16", kind="prefill", **M05, tokens=512, past=0, act="f16"),
        # the largest: a long prompt through one 1.5B-shaped layer
        dict(name="prefill_layer_long_f16", kind="prefill", **M15, tokens=2048, past=0, act="f16"),
        # an odd-sized prompt in fp32
        dict(name="prefill_layer_f32", kind="prefill", **M05, tokens=333, past=0, act="f32"),
        # a piece of a long prompt against the positions before it
        dict(name="attention_chunk_f16", kind="attention", tokens=500, past=3500, heads=12, kv_heads=2, head_dim=128,
             act="f16"),
        # the logits of one token from the tied embedding, and the token drawn from them
        dict(name="lm_head_sample_f16", kind="head", vocab=151936, hidden=896, act="f16"),
        # the model without quantization, fp32: a prompt's gate projection
        dict(name="dense_prompt_f32", kind="dense", M=128, N=4864, K=896, act="f32", bias=False, residual=False),
    ]


# ---- drawn cases -----------------------------------------------------------
def _log(rng, lo: int, hi: int) -> int:
    """An integer spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _model(rng) -> dict:
    """A generic decoder shape, or one of the two named ones."""
    if rng.random() < 0.4:
        return dict(rng.choice([M05, M15]))
    while True:
        d, kv, g = rng.choice([64, 128]), rng.choice([1, 2, 4, 8]), rng.randint(1, 8)
        hidden = d * kv * g
        if 256 <= hidden <= 2048:
            return dict(hidden=hidden, heads=kv * g, kv_heads=kv, inter=64 * _log(rng, hidden // 32, 140))


def draw(rng) -> dict:
    kind = rng.choice(["linear", "linear", "linear", "decode", "decode", "prefill", "prefill", "attention", "head",
                       "dense", "dense"])
    act = rng.choice(["f16", "f16", "f32"])
    if kind == "linear":
        while True:
            m = _model(rng)
            h, kv, i = m["hidden"], m["kv_heads"] * m["hidden"] // m["heads"], m["inter"]
            N, K = rng.choice([(h, h), (kv, h), (i, h), (2 * i, h), (h, i),
                               (_log(rng, 128, 20000), 16 * _log(rng, 16, 560))])
            M = _log(rng, 1, 2048)
            if M * N * K <= 1.5e10:
                return dict(kind=kind, M=M, N=N, K=K, act=act, bias=rng.random() < 0.3, residual=rng.random() < 0.4)
    if kind == "decode":
        return dict(kind=kind, **_model(rng), layers=rng.choice([1, 1, 2]), vocab=0, pos=_log(rng, 1, 8000), act=act)
    if kind == "prefill":
        while True:
            tokens, past = _log(rng, 2, 1200), rng.choice([0, 0, _log(rng, 16, 2000)])
            c = dict(kind=kind, **_model(rng), tokens=tokens, past=past, act=act)
            if tokens * (past + tokens / 2) <= (5e5 if act == "f32" else 1e6):
                return c
    if kind == "attention":
        while True:
            m = _model(rng)
            tokens, past = _log(rng, 2, 1500), rng.choice([0, _log(rng, 1, 6000)])
            if tokens * (past + tokens / 2) * m["hidden"] <= (8e8 if act == "f32" else 1.6e9):
                return dict(kind=kind, tokens=tokens, past=past, heads=m["heads"], kv_heads=m["kv_heads"],
                            head_dim=m["hidden"] // m["heads"], act=act)
    if kind == "head":
        return dict(kind=kind, vocab=_log(rng, 16000, 151936), hidden=_model(rng)["hidden"], act=act)
    m = _model(rng)
    N, K = rng.choice([(m["hidden"], m["hidden"]), (m["inter"], m["hidden"]), (m["hidden"], m["inter"])])
    M = _log(rng, 1, max(1, min(512, int(1.2e9 / (N * K)))))
    return dict(kind=kind, M=M, N=N, K=K, act=act, bias=rng.random() < 0.5, residual=rng.random() < 0.3)


# ---- inputs -----------------------------------------------------------------
def _td(act: str):
    return torch.float16 if act == "f16" else torch.float32


def _cd(act: str) -> int:
    return capi.F16 if act == "f16" else capi.F32


class _Rng:
    """Seeded draws on the GPU."""

    def __init__(self, seed: int):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def normal(self, shape, std=1.0, mean=0.0, dtype=torch.float32):
        t = torch.randn(shape, generator=self.g, device=DEV, dtype=torch.float32)
        return (t * std + mean).to(dtype)

    def integer(self, n: int) -> int:
        return int(torch.randint(n, (1,), generator=self.g, device=DEV).item())


def _quantize(w: torch.Tensor):
    """Per-row int8 codes and fp32 scales (scale = absmax / 127)."""
    scales = w.abs().amax(dim=1) / 127.0
    q = w / scales[:, None]
    codes = torch.clamp(torch.trunc(q + torch.copysign(torch.full_like(q, 0.5), q)), -127, 127).to(torch.int8)
    return codes, scales


class _Q8:
    def __init__(self, rng: _Rng, N: int, K: int, bias: bool = False, src=None):
        self.N, self.K = N, K
        self.q, self.s = _quantize(rng.normal((N, K), 0.02) if src is None else src)
        self.b = rng.normal((N,), 0.01) if bias else None

    def exact(self, x):
        y = x @ (self.q.double() * self.s.double()[:, None]).T
        return y if self.b is None else y + self.b.double()


class _Layer:
    def __init__(self, rng: _Rng, c: dict, rows: int):
        h, kv, i, dt = c["hidden"], c["kv_heads"] * c["hidden"] // c["heads"], c["inter"], _td(c["act"])
        self.ln1, self.ln2 = rng.normal((h,), 0.1, 1.0), rng.normal((h,), 0.1, 1.0)
        self.q, self.k, self.v = _Q8(rng, h, h, True), _Q8(rng, kv, h, True), _Q8(rng, kv, h, True)
        self.o, self.gu, self.down = _Q8(rng, h, h), _Q8(rng, 2 * i, h), _Q8(rng, h, i)
        self.kc, self.vc = rng.normal((rows, kv), dtype=dt), rng.normal((rows, kv), dtype=dt)


class _State:
    """What a program keeps between calls; its plans end with it."""

    def __init__(self, case: dict, seed: int):
        capi.init(torch.cuda.current_device())
        self.case, self.rng, self.plans = case, _Rng(seed), []
        self.act, self.dt = _cd(case["act"]), _td(case["act"])

    def empty(self, *shape, dtype=None):
        return torch.empty(shape, device=DEV, dtype=dtype or self.dt)

    def plan(self, problems) -> int:
        """problems: (out, inp, weight, first row of the weight, rows, M)"""
        arr = (capi.Q8Problem * len(problems))()
        for p, (out, inp, w, r0, n, M) in zip(arr, problems):
            p.out, p.inp, p.residual = out.data_ptr(), inp.data_ptr(), None
            p.weight, p.scales = w.q.data_ptr() + r0 * w.K, w.s.data_ptr() + 4 * r0
            p.bias = w.b.data_ptr() + 4 * r0 if w.b is not None else None
            p.M, p.N, p.K = M, n, w.K
        h = ctypes.c_uint64()
        capi.call("vvh_plan_create", arr, len(problems), self.act, self.act, ctypes.byref(h))
        self.plans.append(h.value)
        return h.value

    def __del__(self):
        for h in getattr(self, "plans", []):
            capi.load().vvh_plan_destroy(h)


def _linear_state(c, seed):
    st = _State(c, seed)
    st.w = _Q8(st.rng, c["N"], c["K"], c["bias"])
    st.x = st.rng.normal((c["M"], c["K"]), dtype=st.dt)
    st.res = st.rng.normal((c["M"], c["N"]), dtype=st.dt) if c["residual"] else None
    st.out = st.empty(c["M"], c["N"])
    return st


def _decode_state(c, seed):
    st = _State(c, seed)
    h, i, D = c["hidden"], c["inter"], c["hidden"] // c["heads"]
    kv, rows = c["kv_heads"] * D, c["pos"] + 1
    st.x = [st.rng.normal((1, h), dtype=st.dt)]
    st.table = st.head = None
    if c["vocab"]:
        st.table = st.rng.normal((c["vocab"], h), 0.02)
        st.head = _Q8(st.rng, c["vocab"], h, src=st.table)
        st.token = st.rng.integer(c["vocab"])
        st.final_ln = st.rng.normal((h,), 0.1, 1.0)
        st.final, st.logits = st.empty(1, h), st.empty(1, c["vocab"], dtype=torch.float32)
    st.layers = [_Layer(st.rng, c, rows) for _ in range(c["layers"])]
    st.x += [st.empty(1, h) for _ in st.layers]
    st.mid = [st.empty(1, h) for _ in st.layers]
    st.norm, st.q, st.k, st.v = st.empty(1, h), st.empty(1, h), st.empty(1, kv), st.empty(1, kv)
    st.attn, st.gu, st.gate = st.empty(1, h), st.empty(1, 2 * i), st.empty(1, i)
    st.fused = c["act"] == "f16"
    st.qkv, st.mlp = [], []
    for n, L in enumerate(st.layers):
        src = st.x[n] if st.fused else st.norm
        p = st.plan([(st.q, src, L.q, 0, h, 1), (st.k, src, L.k, 0, kv, 1), (st.v, src, L.v, 0, kv, 1)])
        st.qkv.append(p)
        if not st.fused:
            continue
        capi.call("vvh_plan_set_input_op", p, capi.IN_RMS_NORM, L.ln1.data_ptr(), EPS)
        capi.call("vvh_plan_set_rope", p, 0, 1, 2, D, THETA, L.kc.data_ptr(), L.vc.data_ptr())
        capi.call("vvh_plan_set_rope_table", p, rows)
        g = st.plan([(st.gate, st.mid[n], L.gu, 0, 2 * i, 1)])
        capi.call("vvh_plan_set_input_op", g, capi.IN_RMS_NORM, L.ln2.data_ptr(), EPS)
        capi.call("vvh_plan_set_glu", g, 0)
        st.mlp.append(g)
    st.nparts = ctypes.c_size_t()
    st.parts = None
    if st.fused and rows <= ATTN_PARTS_MAX_SPAN and h <= 1024 and c["heads"] // c["kv_heads"] <= 16:
        st.parts = st.empty(8 * c["heads"] * (D + 4), dtype=torch.float32)
    return st


def _prefill_state(c, seed):
    st = _State(c, seed)
    S, h, i, D = c["tokens"], c["hidden"], c["inter"], c["hidden"] // c["heads"]
    kv = c["kv_heads"] * D
    st.x = st.rng.normal((S, h), dtype=st.dt)
    st.layer = L = _Layer(st.rng, c, c["past"] + S)
    st.norm, st.q, st.k, st.v = st.empty(S, h), st.empty(S, h), st.empty(S, kv), st.empty(S, kv)
    st.attn, st.mid, st.out = st.empty(S, h), st.empty(S, h), st.empty(S, h)
    st.gate, st.up = st.empty(S, i), st.empty(S, i)
    st.qkv = st.plan([(st.q, st.norm, L.q, 0, h, S), (st.k, st.norm, L.k, 0, kv, S), (st.v, st.norm, L.v, 0, kv, S)])
    st.mlp = st.plan([(st.gate, st.norm, L.gu, 0, i, S), (st.up, st.norm, L.gu, i, i, S)])
    return st


def _attention_state(c, seed):
    st = _State(c, seed)
    rows, D = c["past"] + c["tokens"], c["head_dim"]
    # scores of a few units, so that a query weighs some positions above others
    st.q = st.rng.normal((c["tokens"], c["heads"] * D), 2.0, dtype=st.dt)
    st.kc = st.rng.normal((rows, c["kv_heads"] * D), dtype=st.dt)
    st.vc = st.rng.normal((rows, c["kv_heads"] * D), dtype=st.dt)
    st.out = st.empty(c["tokens"], c["heads"] * D)
    return st


def _head_state(c, seed):
    st = _State(c, seed)
    st.w = st.rng.normal((c["vocab"], c["hidden"]), 0.02, dtype=st.dt)
    st.x = st.rng.normal((1, c["hidden"]), dtype=st.dt)
    st.out = st.empty(1, c["vocab"])
    st.logits = st.empty(1, c["vocab"], dtype=torch.float32) if c["act"] == "f16" else st.out
    st.token = torch.zeros(1, device=DEV, dtype=torch.int32)
    st.seed = seed & 0xFFFFFFFF
    return st


def _dense_state(c, seed):
    st = _State(c, seed)
    st.w = st.rng.normal((c["N"], c["K"]), 0.02, dtype=st.dt)
    st.b = st.rng.normal((c["N"],), 0.01) if c["bias"] else None
    st.x = st.rng.normal((c["M"], c["K"]), dtype=st.dt)
    st.res = st.rng.normal((c["M"], c["N"]), dtype=st.dt) if c["residual"] else None
    st.out = st.empty(c["M"], c["N"])
    return st


_STATES = dict(linear=_linear_state, decode=_decode_state, prefill=_prefill_state, attention=_attention_state,
               head=_head_state, dense=_dense_state)


def prepare(case: dict, seed: int):
    return _STATES[case["kind"]](case, seed)


# ---- one pass ---------------------------------------------------------------
def _p(t):
    return None if t is None else t.data_ptr()


def _linear(st, out, x, w, res, M, stream):
    capi.call("vvh_linear_q8_dev", out.data_ptr(), x.data_ptr(), w.q.data_ptr(), w.s.data_ptr(), _p(w.b), _p(res), M,
              w.N, w.K, st.act, st.act, stream)


def _run_linear(st, stream):
    _linear(st, st.out, st.x, st.w, st.res, st.case["M"], stream)
    return st.out


def _run_decode(st, stream):
    c, call, a = st.case, capi.call, st.act
    h, i, H, KVH, pos = c["hidden"], c["inter"], c["heads"], c["kv_heads"], c["pos"]
    D = h // H
    scale = 1.0 / math.sqrt(D)
    if st.table is not None:
        call("vvh_embedding", st.x[0].data_ptr(), st.table.data_ptr(), st.token, h, c["vocab"], a, stream)
    for n, L in enumerate(st.layers):
        x, mid, out = st.x[n], st.mid[n], st.x[n + 1]
        if st.fused:
            call("vvh_plan_run_pos", st.qkv[n], pos, stream)
        else:
            call("vvh_rms_norm", st.norm.data_ptr(), x.data_ptr(), L.ln1.data_ptr(), 1, h, EPS, a, stream)
            call("vvh_plan_run", st.qkv[n], stream)
            call("vvh_rope_append", st.q.data_ptr(), st.k.data_ptr(), st.v.data_ptr(), L.kc.data_ptr(),
                 L.vc.data_ptr(), 1, H, KVH, D, pos, THETA, a, stream)
        if st.parts is not None:
            call("vvh_attention_parts", st.parts.data_ptr(), st.parts.numel(), ctypes.byref(st.nparts),
                 st.q.data_ptr(), L.kc.data_ptr(), L.vc.data_ptr(), pos + 1, H, KVH, D, scale, a, stream)
            call("vvh_linear_q8_dev_attn", mid.data_ptr(), st.parts.data_ptr(), st.nparts.value, D, L.o.q.data_ptr(),
                 L.o.s.data_ptr(), None, x.data_ptr(), h, h, a, stream)
        else:
            call("vvh_attention", st.attn.data_ptr(), st.q.data_ptr(), L.kc.data_ptr(), L.vc.data_ptr(), 1, pos + 1,
                 H, KVH, D, scale, a, stream)
            _linear(st, mid, st.attn, L.o, x, 1, stream)
        if st.fused:
            call("vvh_plan_run", st.mlp[n], stream)
        else:
            call("vvh_rms_norm", st.norm.data_ptr(), mid.data_ptr(), L.ln2.data_ptr(), 1, h, EPS, a, stream)
            _linear(st, st.gu, st.norm, L.gu, None, 1, stream)
            call("vvh_eltwise", capi.OP_SILU_MUL, st.gate.data_ptr(), st.gu.data_ptr(),
                 st.gu.data_ptr() + i * st.gu.element_size(), i, a, stream)
        _linear(st, out, st.gate, L.down, mid, 1, stream)
    if st.table is None:
        return [st.x[-1]] + [t for L in st.layers for t in (L.kc, L.vc)]
    call("vvh_rms_norm", st.final.data_ptr(), st.x[-1].data_ptr(), st.final_ln.data_ptr(), 1, h, EPS, a, stream)
    call("vvh_linear_q8_dev", st.logits.data_ptr(), st.final.data_ptr(), st.head.q.data_ptr(), st.head.s.data_ptr(),
         None, None, 1, c["vocab"], h, a, capi.F32, stream)
    return [st.logits] + [t for L in st.layers for t in (L.kc, L.vc)]


def _run_prefill(st, stream):
    c, call, a, L = st.case, capi.call, st.act, st.layer
    S, past, h, H, KVH = c["tokens"], c["past"], c["hidden"], c["heads"], c["kv_heads"]
    D = h // H
    call("vvh_rms_norm", st.norm.data_ptr(), st.x.data_ptr(), L.ln1.data_ptr(), S, h, EPS, a, stream)
    call("vvh_plan_run", st.qkv, stream)
    call("vvh_rope_append", st.q.data_ptr(), st.k.data_ptr(), st.v.data_ptr(), L.kc.data_ptr(), L.vc.data_ptr(), S, H,
         KVH, D, past, THETA, a, stream)
    call("vvh_attention", st.attn.data_ptr(), st.q.data_ptr(), L.kc.data_ptr(), L.vc.data_ptr(), S, past + 1, H, KVH,
         D, 1.0 / math.sqrt(D), a, stream)
    _linear(st, st.mid, st.attn, L.o, st.x, S, stream)
    call("vvh_rms_norm", st.norm.data_ptr(), st.mid.data_ptr(), L.ln2.data_ptr(), S, h, EPS, a, stream)
    call("vvh_plan_run", st.mlp, stream)
    call("vvh_eltwise", capi.OP_SILU_MUL, st.gate.data_ptr(), st.gate.data_ptr(), st.up.data_ptr(), S * c["inter"], a,
         stream)
    _linear(st, st.out, st.gate, L.down, st.mid, S, stream)
    return [st.out, L.kc, L.vc]


def _run_attention(st, stream):
    c = st.case
    capi.call("vvh_attention", st.out.data_ptr(), st.q.data_ptr(), st.kc.data_ptr(), st.vc.data_ptr(), c["tokens"],
              c["past"] + 1, c["heads"], c["kv_heads"], c["head_dim"], 1.0 / math.sqrt(c["head_dim"]), st.act, stream)
    return st.out


def _run_head(st, stream):
    c, call = st.case, capi.call
    call("vvh_dense", st.out.data_ptr(), st.x.data_ptr(), st.w.data_ptr(), st.act, None, None, 1, c["vocab"],
         c["hidden"], st.act, stream)
    if st.logits is not st.out:
        call("vvh_convert", st.logits.data_ptr(), capi.F32, st.out.data_ptr(), capi.F16, c["vocab"], stream)
    call("vvh_sample", st.logits.data_ptr(), capi.F32, c["vocab"], 0.7, 1.0, st.seed, 1, st.token.data_ptr(), stream)
    return [st.logits, st.token]


def _run_dense(st, stream):
    c = st.case
    capi.call("vvh_dense", st.out.data_ptr(), st.x.data_ptr(), st.w.data_ptr(), st.act, _p(st.b), _p(st.res), c["M"],
              c["N"], c["K"], st.act, stream)
    return st.out


_RUNS = dict(linear=_run_linear, decode=_run_decode, prefill=_run_prefill, attention=_run_attention, head=_run_head,
             dense=_run_dense)


def run(state):
    return _RUNS[state.case["kind"]](state, torch.cuda.current_stream().cuda_stream or None)


# ---- the work of a pass ------------------------------------------------------
def _layer_work(c, S, past, es):
    h, i, D = c["hidden"], c["inter"], c["hidden"] // c["heads"]
    kv = c["kv_heads"] * D
    codes = 2 * h * h + 2 * kv * h + 3 * h * i
    rows = (h + 2 * kv) * 8 + (2 * h + 2 * i) * 4  # scales, and the biases of q, k and v
    cache = 2 * (past + S) * kv * es               # rows before read, new rows written
    pairs = S * past + S * (S + 1) // 2
    return codes + rows + 8 * h + cache, 2 * S * codes + 4 * c["heads"] * D * pairs


def work(case: dict) -> dict:
    c, es = case, 2 if case["act"] == "f16" else 4
    if c["kind"] in ("linear", "dense"):
        M, N, K = c["M"], c["N"], c["K"]
        wb = N * K + 4 * N if c["kind"] == "linear" else N * K * es
        b = wb + (4 * N if c["bias"] else 0) + M * K * es + M * N * es * (2 if c["residual"] else 1)
        return dict(bytes=b, flops=2 * M * N * K)
    if c["kind"] == "decode":
        b, f = _layer_work(c, 1, c["pos"], es)
        b, f = b * c["layers"] + 2 * c["hidden"] * es, f * c["layers"]
        if c["vocab"]:
            b += c["vocab"] * (c["hidden"] + 8) + 4 * c["hidden"]
            f += 2 * c["vocab"] * c["hidden"]
        return dict(bytes=b, flops=f)
    if c["kind"] == "prefill":
        b, f = _layer_work(c, c["tokens"], c["past"], es)
        return dict(bytes=b + 2 * c["tokens"] * c["hidden"] * es, flops=f)
    if c["kind"] == "attention":
        S, past, D = c["tokens"], c["past"], c["head_dim"]
        return dict(bytes=(2 * S * c["heads"] + 2 * (past + S) * c["kv_heads"]) * D * es,
                    flops=4 * c["heads"] * D * (S * past + S * (S + 1) // 2))
    return dict(bytes=c["vocab"] * c["hidden"] * es + c["hidden"] * es + 4 * c["vocab"] + 4,
                flops=2 * c["vocab"] * c["hidden"])


# ---- how far two correct implementations may be apart ------------------------
def tolerance(case: dict):
    if case["kind"] == "decode" and case["layers"] > 2:
        return {"rel": 1.6e-2}
    return {"rel": _REL[case["kind"], case["act"]]}


# About four times the largest distance from exact() over the listed cases and
# sixty drawn ones.  fp16: one rounding of each output (2e-4 of it), two or
# three where a layer rounds in between (4.6e-4); the 24 layers of a whole step
# hand their roundings on (3.9e-3 in the logits, above).  fp32: sums of up to
# 9000 products (2.9e-7), and of up to 7500 weighted rows of scores whose
# error the exponential magnifies (6.4e-7).
_REL = {
    ("linear", "f16"): 1e-3, ("linear", "f32"): 2e-6,
    ("decode", "f16"): 2e-3, ("decode", "f32"): 2e-6,
    ("prefill", "f16"): 2e-3, ("prefill", "f32"): 3e-6,
    ("attention", "f16"): 1e-3, ("attention", "f32"): 3e-6,
    ("head", "f16"): 1e-3, ("head", "f32"): 2e-6,
    ("dense", "f16"): 1e-3, ("dense", "f32"): 2e-6,
}


# ---- the same in 64 bits -------------------------------------------------------
def _rms(x, w):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + EPS) * w.double()


def _rope(x, heads, pos0):
    """Split-half RoPE of rows [S, heads * D] at positions pos0 ..; the
    exponent, frequency and angle are fp32 values, as the operator defines them."""
    S, D = x.shape[0], x.shape[1] // heads
    half = D // 2
    e = torch.arange(0, D, 2, device=x.device, dtype=torch.float32) / float(D)
    freq = 1.0 / torch.pow(torch.tensor(THETA, device=x.device, dtype=torch.float64), e.double()).float()
    angle = (torch.arange(pos0, pos0 + S, device=x.device, dtype=torch.float32)[:, None] * freq[None, :]).double()
    cos, sin = torch.cos(angle)[:, None, :], torch.sin(angle)[:, None, :]
    v = x.view(S, heads, D)
    a, b = v[..., :half], v[..., half:]
    return torch.cat([a * cos - b * sin, a * sin + b * cos], dim=-1).reshape(S, heads * D)


def _attention(q, k, v, heads, kv_heads, past):
    """Causal attention of rows q at positions past .., a block of queries at a time."""
    S, D = q.shape[0], q.shape[1] // heads
    g, T = heads // kv_heads, k.shape[0]
    out = torch.empty_like(q)
    for h in range(heads):
        kh, vh = k[:, (h // g) * D:(h // g + 1) * D], v[:, (h // g) * D:(h // g + 1) * D]
        for s0 in range(0, S, 1024):
            s1 = min(S, s0 + 1024)
            sc = (q[s0:s1, h * D:(h + 1) * D] @ kh.T) / math.sqrt(D)
            seen = torch.arange(T, device=q.device)[None, :] <= past + torch.arange(s0, s1, device=q.device)[:, None]
            p = torch.softmax(sc.masked_fill(~seen, -math.inf), dim=-1)
            out[s0:s1, h * D:(h + 1) * D] = p @ vh
    return out


def _exact_layer(c, L, x, past):
    S, i = x.shape[0], c["inter"]
    n = _rms(x, L.ln1)
    q = _rope(L.q.exact(n), c["heads"], past)
    kc, vc = L.kc.double(), L.vc.double()
    kc[past:past + S] = _rope(L.k.exact(n), c["kv_heads"], past)
    vc[past:past + S] = L.v.exact(n)
    x = x + L.o.exact(_attention(q, kc, vc, c["heads"], c["kv_heads"], past))
    gu = L.gu.exact(_rms(x, L.ln2))
    gate, up = gu[:, :i], gu[:, i:]
    return x + L.down.exact(gate * torch.sigmoid(gate) * up), kc, vc


def exact(case: dict, seed: int):
    c, st = case, prepare(case, seed)
    if c["kind"] == "linear":
        y = st.w.exact(st.x.double())
        return y if st.res is None else y + st.res.double()
    if c["kind"] == "dense":
        y = st.x.double() @ st.w.double().T
        y = y if st.b is None else y + st.b.double()
        return y if st.res is None else y + st.res.double()
    if c["kind"] == "head":
        return [st.x.double() @ st.w.double().T, None]
    if c["kind"] == "attention":
        return _attention(st.q.double(), st.kc.double(), st.vc.double(), c["heads"], c["kv_heads"], c["past"])
    if c["kind"] == "prefill":
        return list(_exact_layer(c, st.layer, st.x.double(), c["past"]))
    x, caches = st.x[0].double(), []
    if st.table is not None:
        x = st.table[st.token:st.token + 1].to(st.dt).double()
    for L in st.layers:
        x, kc, vc = _exact_layer(c, L, x, c["pos"])
        caches += [kc, vc]
    if st.table is not None:
        x = st.head.exact(_rms(x, st.final_ln))
    return [x] + caches
