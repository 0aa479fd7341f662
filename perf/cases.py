"""Timed workloads of rrr_hip: what a user of the library has it do, through its public calls.

Every case is a dict of plain values with a "kind":

  token      one decode step at a position (a recorded graph of fused calls, as a serving loop replays it)
  rows       a few token rows through whole layers with the batched calls (several sequences decoded
             together, or a very short prompt), f32 rows, a recorded graph
  prompt     a prompt's rows through whole layers with the fused f16 prefill calls, issued call by call
             (prompt lengths differ from request to request)
  gemm       bf16 rows times one weight matrix
  logits     final norm + F32 logits over the transposed vocabulary chunks + argmax
  dequant    a K-quant tensor expanded to f32
  roundtrip  host vector in, one GEMV, host vector out (the reference's gpu_matmul_kquant)

Weights are random super-blocks whose dequantized values have mean about 0 and a standard deviation of
1/sqrt(K), as trained matrices have; hidden rows are N(0, 1) with a few large channels.  Layers take the
mix of a Q4_K_M file: Q5_K for QKV, Q4_K for the attention output and gate/up, Q6_K / Q4_K by turns for
the down matrix.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "recursive-routing-racer-rs_amd"))
import rrr_hip as rrr  # noqa: E402

HEAD_DIM, ROPE_DIM, THETA, ATTN_FACTOR, EPS = 128, 96, 10000.0, 1.190238, 1e-5
MAX_SEQ, CHUNK = 2048, 8192
Q4, Q5, Q6 = rrr.Q4_K, rrr.Q5_K, rrr.Q6_K

# The shape of the repository's own configuration (hidden 3072, FFN 8192, 24 query heads on 8 KV heads).
MAIN = {"heads": 24, "kv": 8, "ffn": 8192}


def listed():
    return [
        # The smallest model calls: a small model's step early in a text, 41 launches of a few microseconds.
        {"name": "token_small", "kind": "token", "heads": 8, "kv": 2, "ffn": 2816, "layers": 8, "vocab": 32064,
         "pos": 37},
        # The headline step: all 32 layers deep into the context, logits on the tied Q6_K embedding (2.5 GB).
        {"name": "token_deep", "kind": "token", **MAIN, "layers": 32, "vocab": 200064, "pos": 1900},
        # Sequences decoded together: few, some, many.  Four layers each, so weights come from HBM and not a cache.
        {"name": "rows_3", "kind": "rows", **MAIN, "layers": 4, "rows": 3},
        {"name": "rows_8", "kind": "rows", **MAIN, "layers": 4, "rows": 8},
        {"name": "rows_27", "kind": "rows", **MAIN, "layers": 4, "rows": 27},
        # A short question, an ordinary prompt behind a cached prefix, and a prompt that nearly fills the cache.
        {"name": "prompt_75", "kind": "prompt", **MAIN, "layers": 4, "rows": 75, "pos": 0},
        {"name": "prompt_512", "kind": "prompt", **MAIN, "layers": 4, "rows": 512, "pos": 256},
        {"name": "prompt_2000", "kind": "prompt", **MAIN, "layers": 2, "rows": 2000, "pos": 0},
        # One bf16 GEMM with a ragged row count (a batch of prompts' rows through the down matrix).
        {"name": "gemm_1111", "kind": "gemm", "type": Q6, "K": 8192, "N": 3072, "rows": 1111},
        # The reference's F32 logits over the full vocabulary (2.46 GB), whose last chunk is ragged.
        {"name": "logits_f32", "kind": "logits", "K": 3072, "vocab": 200064},
        # A weight tensor expanded to f32, as a host that needs float weights has it done.
        {"name": "dequant_q4k", "kind": "dequant", "type": Q4, "K": 3072, "N": 16384},
        # The smallest call: one vector in from the host, one GEMV, one vector back.
        {"name": "roundtrip_q6k", "kind": "roundtrip", "type": Q6, "K": 8192, "N": 3072},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))


def _shape(rng):
    heads, kv = rng.choice([(8, 2), (8, 8), (12, 4), (16, 8), (20, 10), (24, 8), (24, 8), (32, 8)])
    return {"heads": heads, "kv": kv, "ffn": 256 * max(4, round(heads * HEAD_DIM * rng.uniform(2.0, 3.6) / 256))}


def draw(rng):
    kind = rng.choice(["token", "token", "rows", "rows", "rows", "prompt", "prompt", "prompt", "gemm", "logits",
                       "dequant", "roundtrip"])
    if kind == "token":
        s = _shape(rng)
        return {"kind": kind, **s, "layers": rng.randint(2, 12), "vocab": int(_log(rng, 4000, 130000)),
                "pos": int(_log(rng, 1, MAX_SEQ - 1))}
    if kind == "rows":
        return {"kind": kind, **_shape(rng), "layers": 3, "rows": int(_log(rng, 2, 64))}
    if kind == "prompt":
        rows = int(_log(rng, 5, 1900))
        return {"kind": kind, **_shape(rng), "layers": 2 if rows > 600 else 3, "rows": rows,
                "pos": rng.choice([0, rng.randint(0, MAX_SEQ - 1 - rows)])}
    t = rng.choice([Q4, Q5, Q6])
    if kind == "gemm":
        return {"kind": kind, "type": t, "K": 256 * rng.randint(4, 40), "N": 64 * int(_log(rng, 8, 256)),
                "rows": int(_log(rng, 17, 2048))}
    if kind == "logits":
        return {"kind": kind, "K": 256 * rng.randint(2, 12), "vocab": int(_log(rng, 3000, 200000))}
    if kind == "dequant":
        return {"kind": kind, "type": t, "K": 256 * rng.randint(4, 32), "N": int(_log(rng, 64, 16000))}
    return {"kind": kind, "type": t, "K": 256 * rng.randint(2, 40), "N": int(_log(rng, 200, 17000))}


# ---- inputs ----------------------------------------------------------------

BLOCK = {Q4: 144, Q5: 176, Q6: 210}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _weight(g, qtype, K, N):
    """N x K random super-blocks (uint8, one block a row)."""
    nb = N * K // 256
    b = torch.randint(0, 256, (nb, BLOCK[qtype]), dtype=torch.uint8, device="cuda", generator=g)
    step = 0.5 + torch.rand(nb, device="cuda", generator=g)
    # rms of the sub-block scales times the standard deviation of the quants
    spread, mid = {Q4: (36.6 * 4.61, 7.5), Q5: (36.6 * 9.23, 15.5), Q6: (73.9 * 18.5, 0.0)}[qtype]
    d = (step / (spread * math.sqrt(K))).half()
    if qtype == Q6:
        b[:, 208:210] = d[:, None].view(torch.uint8)
    else:
        b[:, 0:2] = d[:, None].view(torch.uint8)
        b[:, 2:4] = (d.float() * mid).half()[:, None].view(torch.uint8)
        b[:, 8:12] = b[:, 4:8]                      # each sub-block's min code equals its scale code: mean 0
        low = b[:, 12:16] & 15
        b[:, 12:16] = low | (low << 4)
    return b


def _rows(g, rows, d):
    x = torch.randn(rows, d, device="cuda", generator=g)
    x[:, torch.randperm(d, device="cuda", generator=g)[: max(1, d // 500)]] *= 20.0
    return x


def _gamma(g, d):
    return 1.0 + 0.1 * torch.randn(d, device="cuda", generator=g)


def _matrices(case, i):
    d, kvd, f = case["heads"] * HEAD_DIM, case["kv"] * HEAD_DIM, case["ffn"]
    return [("qkv", Q5, d, d + 2 * kvd), ("o", Q4, d, d), ("up", Q4, d, 2 * f),
            ("down", Q6 if i % 2 == 0 else Q4, f, d)]


def _layers(g, case):
    for i in range(case["layers"]):
        d = case["heads"] * HEAD_DIM
        layer = {"n1": _gamma(g, d), "n2": _gamma(g, d)}
        for name, t, K, N in _matrices(case, i):
            layer[name] = _weight(g, t, K, N)
        if case["kind"] != "rows":      # the rows of the cache before this call
            for c in ("k", "v"):
                layer[c] = torch.randn(case["pos"], case["kv"] * HEAD_DIM, device="cuda", generator=g).half()
        else:                           # the sequences' attention outputs
            layer["att"] = _rows(g, case["rows"], d)
        yield layer


def _factors(g):
    return 1.0 + torch.randn(ROPE_DIM // 2, device="cuda", generator=g).abs()


# ---- the library's side ----------------------------------------------------

_CTX = None


def _ctx():
    """One context for the process, as a program keeps one engine; calls are queued and not waited for."""
    global _CTX
    if _CTX is None:
        _CTX = rrr.Context(0)
        _CTX.set_async(True)
    return _CTX


class _State:
    """Device buffers (freed with the state) and what a pass issues."""

    def __init__(self):
        self.ctx, self.bufs, self.graph = _ctx(), [], None

    def alloc(self, nbytes):
        self.bufs.append(self.ctx.alloc(max(int(nbytes), 256)))
        return self.bufs[-1]

    def put(self, t):
        b = self.alloc(t.numel() * t.element_size())
        self.ctx.upload(b, t.contiguous().view(torch.uint8).cpu().numpy())
        return b

    def weight(self, qtype, K, N, raw):
        self.bufs.append(self.ctx.weight_upload(qtype, K, N, raw.cpu().numpy()))
        return self.bufs[-1]

    def cache(self, t):
        b = self.alloc(MAX_SEQ * t.shape[1] * 2)
        self.ctx.fill_u32(b, 0)
        if t.shape[0]:
            self.ctx.upload(b, t.contiguous().view(torch.uint8).cpu().numpy())
        return b

    def record(self, issue):
        self.ctx.graph_begin()
        issue()
        self.graph = self.ctx.graph_end()

    def __del__(self):
        if self.graph is not None:
            self.graph.destroy()
        for b in self.bufs:
            b.free()


class _Results(dict):
    """A pass's outputs by name.  They stay in their device buffers (which live as long as this), where the
    program's next call finds them; reading an entry copies it to the host."""

    def __init__(self, state):
        super().__init__(state.out)
        self.state = state

    def __getitem__(self, name):
        buf, dtype, offset, shape = super().__getitem__(name)
        return self.state.ctx.download(buf, dtype, int(np.prod(shape)), offset).reshape(shape)


def _prepare_token(case, seed):
    s, g = _State(), _gen(seed)
    c, heads, kv, f, pos, V = s.ctx, case["heads"], case["kv"], case["ffn"], case["pos"], case["vocab"]
    d, kvd = heads * HEAD_DIM, kv * HEAD_DIM
    x, factors, norm = s.put(_rows(g, 1, d)), s.put(_factors(g)), s.put(_gamma(g, d))
    zero, hid, qkv, att = s.put(torch.zeros(d)), s.alloc(d * 4), s.alloc((d + 2 * kvd) * 4), s.alloc(d * 4)
    mid, logits, token = s.alloc(f * 4), s.alloc(V * 4), s.alloc(4)
    layers = []
    for i, L in enumerate(_layers(g, case)):
        dev = {n: s.weight(t, K, N, L[n]) for n, t, K, N in _matrices(case, i)}
        layers.append((dev, s.put(L["n1"]), s.put(L["n2"]), s.cache(L["k"]), s.cache(L["v"])))
    emb = s.weight(Q6, d, V, _weight(g, Q6, d, V))

    def issue():
        c.residual_add(x, zero, hid, d)
        for i, (w, n1, n2, kc, vc) in enumerate(layers):
            c.gemv_rmsnorm_rope_kv(hid, n1, EPS, w["qkv"], Q5, qkv, d, factors, ROPE_DIM // 2, kc, vc, pos, heads, kv,
                                   HEAD_DIM, ROPE_DIM, d, kvd, THETA, ATTN_FACTOR)
            c.attention(qkv, kc, vc, att, pos + 1, kv, heads // kv, HEAD_DIM)
            c.gemv_residual(att, rrr.ACT_IDENTITY, 0, w["o"], Q4, hid, d, d)
            c.gemv_rmsnorm_silu(hid, n2, EPS, w["up"], Q4, mid, d, f)
            c.gemv_residual(mid, rrr.ACT_IDENTITY, 0, w["down"], Q6 if i % 2 == 0 else Q4, hid, f, d)
        c.logits_rmsnorm_argmax(hid, norm, EPS, emb, logits, d, V, token, rrr.LOGITS_Q6K, 0)

    s.record(issue)
    kc, vc = layers[-1][3:]
    s.out = {"hidden": (hid, np.float32, 0, (d,)), "logits": (logits, np.float32, 0, (V,)),
             "token": (token, np.uint32, 0, (1,)), "k": (kc, np.float16, pos * kvd * 2, (kvd,)),
             "v": (vc, np.float16, pos * kvd * 2, (kvd,))}
    return s


def _prepare_rows(case, seed):
    s, g = _State(), _gen(seed)
    c, M, f = s.ctx, case["rows"], case["ffn"]
    d, kvd = case["heads"] * HEAD_DIM, case["kv"] * HEAD_DIM
    x, zero = s.put(_rows(g, M, d)), s.put(torch.zeros(M, d))
    hid, nrm, qkv = s.alloc(M * d * 4), s.alloc(M * d * 4), s.alloc(M * (d + 2 * kvd) * 4)
    tmp, gu, mid = s.alloc(M * d * 4), s.alloc(M * 2 * f * 4), s.alloc(M * f * 4)
    layers = []
    for i, L in enumerate(_layers(g, case)):
        dev = {n: s.weight(t, K, N, L[n]) for n, t, K, N in _matrices(case, i)}
        layers.append((dev, s.put(L["n1"]), s.put(L["n2"]), s.put(L["att"])))

    def issue():
        c.residual_add(x, zero, hid, M * d)
        for i, (w, n1, n2, att) in enumerate(layers):
            c.rmsnorm(hid, n1, nrm, M, d, EPS)
            c.gemv(nrm, w["qkv"], Q5, qkv, d, d + 2 * kvd, M)
            c.gemv(att, w["o"], Q4, tmp, d, d, M)
            c.residual_add(hid, tmp, hid, M * d)
            c.rmsnorm(hid, n2, nrm, M, d, EPS)
            c.gemv(nrm, w["up"], Q4, gu, d, 2 * f, M)
            c.silu_gate(gu, mid, M, f)
            c.gemv(mid, w["down"], Q6 if i % 2 == 0 else Q4, tmp, f, d, M)
            c.residual_add(hid, tmp, hid, M * d)

    s.record(issue)
    s.out = {"hidden": (hid, np.float32, 0, (M, d)), "qkv": (qkv, np.float32, 0, (M, d + 2 * kvd))}
    return s


def _prepare_prompt(case, seed):
    s, g = _State(), _gen(seed)
    c, heads, kv, f, M, pos = s.ctx, case["heads"], case["kv"], case["ffn"], case["rows"], case["pos"]
    d, kvd = heads * HEAD_DIM, kv * HEAD_DIM
    Mp = -(-M // 128) * 128                     # the GEMMs take whole row blocks: zero rows fill the last
    rows = torch.zeros(Mp, d, device="cuda")
    rows[:M] = _rows(g, M, d)
    x, zero, factors = s.put(rows), s.put(torch.zeros(Mp, d)), s.put(_factors(g))
    hid, n16, qkv = s.alloc(Mp * d * 4), s.alloc(Mp * d * 2), s.alloc(Mp * (d + 2 * kvd) * 4)
    att, gu, mid, scale = s.alloc(Mp * d * 2), s.alloc(Mp * 2 * f * 4), s.alloc(Mp * f * 2), s.alloc(Mp * 4)
    for b in (n16, qkv, att, gu, mid, scale):
        c.fill_u32(b, 0)
    layers = []
    for i, L in enumerate(_layers(g, case)):
        dev = {n: s.weight(t, K, N, L[n]) for n, t, K, N in _matrices(case, i)}
        layers.append((dev, s.put(L["n1"]), s.put(L["n2"]), s.cache(L["k"]), s.cache(L["v"])))
    fused_silu = Mp % 256 == 0 and f % 64 == 0 and (f // 64) * (Mp // 256) >= 128 and Mp * f * 4 <= (48 << 20)

    def issue():
        c.residual_add(x, zero, hid, Mp * d)
        for i, (w, n1, n2, kc, vc) in enumerate(layers):
            if i == 0:
                c.rmsnorm_f16(hid, n1, n16, Mp, d, EPS)
            c.gemm_f16_rope_kv_rows(n16, w["qkv"], Q5, qkv, d, Mp, M, factors, ROPE_DIM // 2, kc, vc, pos, heads, kv,
                                    HEAD_DIM, ROPE_DIM, d, kvd, THETA, ATTN_FACTOR)
            c.attention_prefill(qkv, M, kc, vc, att, pos, kv, heads // kv, HEAD_DIM, out_type=rrr.F16)
            c.gemm_f16_rmsnorm(att, w["o"], Q4, hid, d, d, Mp, n2, n16, EPS, accumulate=True)
            if fused_silu:
                c.gemm_f16_silu_gate_f16(n16, w["up"], Q4, mid, scale, d, f, Mp)
            else:
                c.gemm_f16(n16, w["up"], Q4, gu, d, 2 * f, Mp)
                c.silu_gate_f16(gu, mid, scale, Mp, f)
            t = Q6 if i % 2 == 0 else Q4
            if i + 1 < len(layers):
                c.gemm_f16_rmsnorm(mid, w["down"], t, hid, f, d, Mp, layers[i + 1][1], n16, EPS, accumulate=True,
                                   row_scale=scale)
            else:
                c.gemm_f16(mid, w["down"], t, hid, f, d, Mp, accumulate=True, row_scale=scale)

    s.issue = issue
    kc, vc = layers[-1][3:]
    s.out = {"hidden": (hid, np.float32, 0, (M, d)), "k": (kc, np.float16, pos * kvd * 2, (M, kvd)),
             "v": (vc, np.float16, pos * kvd * 2, (M, kvd))}
    return s


def _prepare_gemm(case, seed):
    s, g = _State(), _gen(seed)
    c = s.ctx
    K, N, M, t = case["K"], case["N"], case["rows"], case["type"]
    x, w, y = s.put(_rows(g, M, K).bfloat16()), s.weight(t, K, N, _weight(g, t, K, N)), s.alloc(M * N * 4)
    s.issue = lambda: c.gemm_bf16(x, w, t, y, K, N, M)
    s.out = {"y": (y, np.float32, 0, (M, N))}
    return s


def _embedding(g, case):
    """The F32 logits matrix in the reference's transposed chunks: chunk c holds B_c[k * n + v]."""
    return torch.randn(case["vocab"] * case["K"], device="cuda", generator=g) * 0.02


def _prepare_logits(case, seed):
    s, g = _State(), _gen(seed)
    c = s.ctx
    K, V = case["K"], case["vocab"]
    x, gamma, emb = s.put(_rows(g, 1, K)), s.put(_gamma(g, K)), s.put(_embedding(g, case))
    y, token = s.alloc(V * 4), s.alloc(4)
    s.issue = lambda: c.logits_rmsnorm_argmax(x, gamma, EPS, emb, y, K, V, token, rrr.LOGITS_CHUNKED, CHUNK)
    s.out = {"logits": (y, np.float32, 0, (V,)), "token": (token, np.uint32, 0, (1,))}
    return s


def _prepare_dequant(case, seed):
    s, g = _State(), _gen(seed)
    c = s.ctx
    K, N, t = case["K"], case["N"], case["type"]
    w, y = s.weight(t, K, N, _weight(g, t, K, N)), s.alloc(K * N * 4)
    s.issue = lambda: c.dequant(t, w, y, K * N)
    s.out = {"w": (y, np.float32, 0, (N, K))}
    return s


def _prepare_roundtrip(case, seed):
    s, g = _State(), _gen(seed)
    K, N, t = case["K"], case["N"], case["type"]
    x = _rows(g, 1, K)[0].cpu().numpy()
    c, w, a, y = s.ctx, s.weight(t, K, N, _weight(g, t, K, N)), s.alloc(K * 4), s.alloc(N * 4)
    s.call = lambda: c.matmul_kquant(a, w, y, t, x, K, N)
    return s


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    if hasattr(state, "call"):
        return state.call()
    if state.graph is not None:
        state.graph.launch()
    else:
        state.issue()
    return _Results(state)


# ---- what a pass cannot do without -----------------------------------------

def work(case):
    kind = case["kind"]
    if kind in ("token", "rows", "prompt"):
        d, kvd = case["heads"] * HEAD_DIM, case["kv"] * HEAD_DIM
        M = case.get("rows", 1)
        nbytes, weights = 0, 0
        for i in range(case["layers"]):
            for _, t, K, N in _matrices(case, i):
                nbytes += rrr.tensor_bytes(t, K, N)
                weights += K * N
            nbytes += 2 * d * 4
        nbytes += 2 * M * d * 4                                    # hidden rows in and out
        flops = 2 * M * weights
        if kind == "rows":
            nbytes += case["layers"] * M * (d + d + 2 * kvd) * 4   # attention outputs in, qkv rows out
            return {"bytes": nbytes, "flops": flops}
        pos = case["pos"]
        nbytes += case["layers"] * 2 * (pos + M) * kvd * 2         # the cache: earlier rows read, new ones written
        flops += case["layers"] * 4 * d * (M * pos + M * (M + 1) // 2)
        if kind == "token":
            nbytes += rrr.tensor_bytes(Q6, d, case["vocab"]) + case["vocab"] * 4
            flops += 2 * d * case["vocab"]
        return {"bytes": nbytes, "flops": flops}
    if kind == "logits":
        K, V = case["K"], case["vocab"]
        return {"bytes": V * K * 4 + 2 * K * 4 + V * 4, "flops": 2 * K * V}
    K, N, w = case["K"], case["N"], rrr.tensor_bytes(case["type"], case["K"], case["N"])
    if kind == "gemm":
        return {"bytes": w + case["rows"] * (2 * K + 4 * N), "flops": 2 * case["rows"] * K * N}
    if kind == "dequant":
        return {"bytes": w + 4 * K * N, "flops": 2 * K * N}
    return {"bytes": w + 4 * (K + N), "flops": 2 * K * N}


def tolerance(case):
    """About four times what the library's results differ from exact() by, for each kind's arithmetic."""
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    if kind == "token":          # f32 rows (1e-5 off after the layers); new cache rows are f16, angles f32 (9e-5)
        return {"rel": 4e-4, "max": 5e-3}
    if kind == "rows":           # to 16 rows f32 results (4e-7 to 3e-6 off), above f16 operands (8e-4)
        return {"rel": 1.5e-5, "max": 2e-4} if case["rows"] <= 16 else {"rel": 3e-3, "max": 2e-2}
    if kind == "prompt":         # f16 operands through every layer (1.3e-3 off)
        return {"rel": 5e-3, "max": 5e-2}
    if kind == "gemm":           # f16 operands (2.9e-4 off)
        return {"rel": 1.2e-3, "max": 8e-3}
    return {"rel": 1e-5, "max": 1e-4}    # f32 sums, 20-bit activation digits (2e-7 to 2e-6 off)


# ---- the same results in 64 bits -------------------------------------------

def _dequant(b, qtype):
    """Super-blocks (uint8 rows) as f64 rows of 256."""
    nb = b.shape[0]

    def f16(lo):
        return b[:, lo:lo + 2].contiguous().view(torch.float16).double().view(nb, 1, 1)

    if qtype == Q6:
        ql, qh = b[:, :128].reshape(nb, 2, 2, 32), b[:, 128:192].reshape(nb, 2, 32)
        quarters = []
        for q in range(4):           # 32 values each: ql half q % 2, its low or high nibble, qh bits 2q
            nib = ql[:, :, q % 2] & 15 if q < 2 else ql[:, :, q % 2] >> 4
            quarters.append((nib | (((qh >> (2 * q)) & 3) << 4)).double() - 32.0)
        q = torch.stack(quarters, 2).reshape(nb, 16, 16)
        sc = b[:, 192:208].contiguous().view(torch.int8).double().view(nb, 16, 1)
        return (f16(208) * sc * q).reshape(nb, 256)
    s = b[:, 4:16].int()
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
    qs = (b[:, 16:144] if qtype == Q4 else b[:, 48:176]).reshape(nb, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], 2).reshape(nb, 8, 32)
    if qtype == Q5:
        bit = torch.arange(8, device=b.device, dtype=torch.uint8).view(1, 8, 1)
        q = q + (((b[:, 16:48].reshape(nb, 1, 32) >> bit) & 1) << 4)
    return (f16(0) * sc.double()[:, :, None] * q.double() - f16(2) * mn.double()[:, :, None]).reshape(nb, 256)


def _times(x, raw, qtype, K):
    """x (rows x K, f64) times the transposed matrix of `raw`, in slices of its rows."""
    per = K // 256
    step = max(1, (1 << 25) // K) * per
    return torch.cat([x @ _dequant(raw[i:i + step], qtype).view(-1, K).T for i in range(0, raw.shape[0], step)], 1)


def _norm(x, gamma):
    return x * gamma.double() / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def _rope(x, positions, factors):
    """x: rows x heads x HEAD_DIM; interleaved pairs over the first ROPE_DIM dims."""
    i = torch.arange(ROPE_DIM // 2, device="cuda", dtype=torch.float64)
    angle = positions.double()[:, None] * (THETA ** (-2.0 * i / ROPE_DIM) / factors.double())[None]
    cos, sin = (ATTN_FACTOR * f(angle)[:, None] for f in (torch.cos, torch.sin))
    a, b = x[..., 0:ROPE_DIM:2], x[..., 1:ROPE_DIM:2]
    out = x.clone()
    out[..., 0:ROPE_DIM:2], out[..., 1:ROPE_DIM:2] = a * cos - b * sin, a * sin + b * cos
    return out


def _half(x):
    """As the f16 cache holds it."""
    return x.half().double()


def _attention(q, k, v, pos):
    """q: rows x heads x HEAD_DIM at positions pos ..; k, v: cache rows x KV heads x HEAD_DIM."""
    M, heads = q.shape[:2]
    per = heads // k.shape[1]
    seen = torch.arange(k.shape[0], device="cuda")[None] <= pos + torch.arange(M, device="cuda")[:, None]
    out = torch.empty_like(q)
    for h in range(heads):
        p = (q[:, h] @ k[:, h // per].T) / math.sqrt(HEAD_DIM)
        out[:, h] = torch.softmax(p.masked_fill(~seen, -math.inf), 1) @ v[:, h // per]
    return out.reshape(M, -1)


def _silu_gate(gu):
    a, b = gu.chunk(2, -1)
    return a / (1 + torch.exp(-a)) * b


def _exact_layers(g, case, x, factors):
    """(hidden rows, last layer's qkv, its new K rows, its new V rows)."""
    heads, kv = case["heads"], case["kv"]
    d, kvd, M, pos = heads * HEAD_DIM, kv * HEAD_DIM, x.shape[0], case.get("pos", 0)
    h, k, v = x.double(), None, None
    for i, L in enumerate(_layers(g, case)):
        qkv = _times(_norm(h, L["n1"]), L["qkv"], Q5, d)
        if case["kind"] == "rows":
            att = L["att"].double()
        else:
            at = pos + torch.arange(M, device="cuda")
            q = _rope(qkv[:, :d].reshape(M, heads, HEAD_DIM), at, factors)
            k = _half(_rope(qkv[:, d:d + kvd].reshape(M, kv, HEAD_DIM), at, factors))
            v = _half(qkv[:, d + kvd:].reshape(M, kv, HEAD_DIM))
            kk, vv = (torch.cat([L[n].double().view(pos, kv, HEAD_DIM), new]) for n, new in (("k", k), ("v", v)))
            att = _attention(q, kk, vv, pos)
        h = h + _times(att, L["o"], Q4, d)
        mid = _silu_gate(_times(_norm(h, L["n2"]), L["up"], Q4, d))
        h = h + _times(mid, L["down"], Q6 if i % 2 == 0 else Q4, case["ffn"])
    return h, qkv, k, v


def exact(case, seed):
    g, kind = _gen(seed), case["kind"]

    def host(t):
        return t.cpu().numpy()

    if kind in ("token", "rows", "prompt"):
        M, d, kvd = case.get("rows", 1), case["heads"] * HEAD_DIM, case["kv"] * HEAD_DIM
        x = _rows(g, M, d)
        factors = _factors(g) if kind != "rows" else None
        norm = _gamma(g, d) if kind == "token" else None
        h, qkv, k, v = _exact_layers(g, case, x, factors)
        if kind == "rows":
            return {"hidden": host(h), "qkv": host(qkv)}
        if kind == "prompt":
            return {"hidden": host(h), "k": host(k.reshape(M, kvd)), "v": host(v.reshape(M, kvd))}
        logits = _times(_norm(h, norm), _weight(g, Q6, d, case["vocab"]), Q6, d)
        return {"hidden": host(h[0]), "logits": host(logits[0]), "token": None, "k": host(k.reshape(-1)),
                "v": host(v.reshape(-1))}
    K = case["K"]
    if kind == "logits":
        x, gamma = _rows(g, 1, K), _gamma(g, K)
        e, x, out = _embedding(g, case), _norm(x.double(), gamma), []
        for v0 in range(0, case["vocab"], CHUNK):
            n = min(CHUNK, case["vocab"] - v0)
            out.append(x @ e[v0 * K:(v0 + n) * K].view(K, n).double())
        return {"logits": host(torch.cat(out, 1)[0]), "token": None}
    N, t = case["N"], case["type"]
    if kind == "gemm":
        x = _rows(g, case["rows"], K).bfloat16().double()
        return {"y": host(_times(x, _weight(g, t, K, N), t, K))}
    if kind == "dequant":
        return {"w": host(_dequant(_weight(g, t, K, N), t).view(N, K))}
    x = _rows(g, 1, K).double()
    return host(_times(x, _weight(g, t, K, N), t, K)[0])
