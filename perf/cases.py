"""Performance cases of the verify path: what a program that uses this
library has it compute, through its public entry points (the plan API, the
direct calls and the qwen35 engine), over the sizes they are used at.

A case is a dict; "kind" names the part of the path:

  proj    one packed projection of a few rows through yuuka_lm_head: the
          matvec of a plain decode step (1 row), a verify projection, the
          LM head over the vocabulary
  ffn     RMSNorm + gate/up + SwiGLU and the down projection + residual as a
          captured plan: 1-8 rows of one request's verify step, up to a few
          hundred rows of a batch or of prefill chunks
  gdn     a Gated DeltaNet block: norm + input projections, the deferred
          scan of every request's rows, gated out projection + residual,
          and the commit of the accepted rows into the recurrent state
  attn    a gated attention block: norm + q|gate, k, v projections, rotation
          table, paged verify attention with the KV write, out projection
  moe     an MoE FFN block: norm, router, top-k routing, grouped expert
          SwiGLU and down projection with the shared expert, combine
  accept  fused acceptance over the logits of a step (greedy, stochastic,
          top-k / top-p)
  model   whole engine calls: a new request's prompt, then verify steps,
          and the last step's logits

Weights are packed Q4_K / Q6_K super-blocks of random quants whose
dequantized spread is about 0.02, activations are normal; `exact` computes
the same in float64 with torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from yuuka_amd import hip, model

Q4_K, Q6_K, F16, F32 = hip.Q4_K, hip.Q6_K, hip.F16, hip.F32
BLOCK_BYTES = {Q4_K: 144, Q6_K: 210}
DTYPES = {"q4_k": Q4_K, "q6_k": Q6_K, "f16": F16, "f32": F32}

# flags of include/yuuka_hip.h that hip.py does not name
FLAG_DEFER, FLAG_RAW_OUT, FLAG_GDN_COEF, FLAG_OWN_POS, FLAG_MOE_SHARED = 0x100, 0x200, 0x400, 0x1000, 0x4000

EPS = 1e-6
STATE = 128          # GDN head width
CONV = 4             # GDN conv taps
HEAD_DIM, ROPE_DIM, ROPE_BASE, BLOCK = 256, 64, 1e7, 16
VOCAB = 151936


def listed():
    return [
        # one plain decode matvec (an out projection): launch latency
        dict(name="proj_decode", kind="proj", rows=1, n_in=2560, n_out=2560, dtype="q4_k"),
        # the LM head of a verify step, k = 4 drafts
        dict(name="proj_head", kind="proj", rows=5, n_in=2560, n_out=VOCAB, dtype="q6_k"),
        # FFN of a single request's verify step, k = 4
        dict(name="ffn_verify", kind="ffn", rows=5, hidden=2560, ffn=9216),
        # FFN of four requests with k = 16 (the 9B-like widths)
        dict(name="ffn_batch4", kind="ffn", rows=68, hidden=4096, ffn=12288),
        # FFN of sixteen requests with k = 8
        dict(name="ffn_batch16", kind="ffn", rows=144, hidden=2560, ffn=9216),
        # Gated DeltaNet layer, one request, k = 4
        dict(name="gdn_verify", kind="gdn", requests=1, rows=5, hidden=2560, heads=16),
        # Gated DeltaNet layer, sixteen requests, k = 8
        dict(name="gdn_batch16", kind="gdn", requests=16, rows=9, hidden=2560, heads=16),
        # attention layer early in a conversation, one request, k = 4
        dict(name="attn_verify", kind="attn", requests=1, rows=5, context=517, hidden=2560, heads=16, kv_heads=4,
             kv="f16"),
        # attention layer, sixteen requests with 4k contexts, k = 8
        dict(name="attn_batch16", kind="attn", requests=16, rows=9, context=4096, hidden=2560, heads=16, kv_heads=4,
             kv="f16"),
        # MoE FFN of eight requests, k = 4: 256 experts, top 8
        dict(name="moe_batch8", kind="moe", rows=40, hidden=2048, expert_ffn=512, experts=256, used=8),
        # acceptance of sixteen requests, k = 8, sampled with top-p
        dict(name="accept_topp", kind="accept", requests=16, drafts=8, vocab=VOCAB, mode="stochastic",
             temperature=0.7, top_k=0, top_p=0.9),
        # a new request on the 4B-like decoder: prompt of 77 tokens, eight verify steps of k = 4
        dict(name="model_request", kind="model", layers=32, prompt=77, steps=8, rows=5),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _blocks(rng, lo, hi):
    """A width in whole 256-element super-blocks, spread over its logarithm."""
    return 256 * _log_int(rng, lo // 256, hi // 256)


def draw(rng):
    kind = rng.choice(["proj", "proj", "ffn", "ffn", "ffn", "gdn", "gdn", "attn", "attn", "moe", "accept", "model"])
    if kind == "proj":
        n_in = _blocks(rng, 1024, 12288)
        return dict(kind=kind, rows=rng.randint(1, 16), n_in=n_in,
                    n_out=_log_int(rng, 256, min(VOCAB, 2560 * VOCAB // n_in)), dtype=rng.choice(["q4_k", "q6_k"]))
    if kind == "ffn":
        return dict(kind=kind, rows=_log_int(rng, 1, 256), hidden=_blocks(rng, 1024, 4096),
                    ffn=_blocks(rng, 2048, 12288))
    if kind == "gdn":
        return dict(kind=kind, requests=_log_int(rng, 1, 16), rows=rng.randint(1, 17),
                    hidden=_blocks(rng, 1024, 4096), heads=rng.choice([8, 16, 16, 32]))
    if kind == "attn":
        requests = _log_int(rng, 1, 16)
        kv = rng.choice(["f16", "f16", "f16", "f32"])
        heads, kv_heads = rng.choice([(16, 4), (16, 4), (8, 2), (16, 2)])
        rows = rng.randint(1, 17) if kv == "f16" else rng.randint(1, 8)
        # the float32 pool's kernel holds rows x heads / kv_heads <= 40 query rows
        rows = rows if kv == "f16" else min(rows, 40 * kv_heads // heads)
        return dict(kind=kind, requests=requests, rows=rows,
                    context=_log_int(rng, 1, min(16384, (65536 if kv == "f16" else 16384) // requests)),
                    hidden=_blocks(rng, 1024, 4096), heads=heads, kv_heads=kv_heads, kv=kv)
    if kind == "moe":
        return dict(kind=kind, rows=_log_int(rng, 1, 160), hidden=256 * rng.randint(4, 8),
                    expert_ffn=rng.choice([256, 512]), experts=rng.choice([16, 64, 128, 256]), used=rng.randint(2, 8))
    if kind == "accept":
        mode = rng.choice(["greedy", "stochastic", "stochastic", "stochastic"])
        return dict(kind=kind, requests=_log_int(rng, 1, 16), drafts=rng.randint(0, 8),
                    vocab=_log_int(rng, 8192, VOCAB), mode=mode, temperature=round(rng.uniform(0.5, 1.2), 2),
                    top_k=rng.choice([0, 0, 40, 200]) if mode != "greedy" else 0,
                    top_p=rng.choice([1.0, 0.8, 0.9, 0.95]) if mode != "greedy" else 1.0)
    return dict(kind=kind, layers=4 * rng.randint(1, 3), prompt=_log_int(rng, 16, 77), steps=rng.randint(1, 8),
                rows=rng.randint(2, 9))


# ------------------------------------------------------------ device memory

_device = _stream = None


def _open():
    """The device and the stream that every case runs on."""
    global _device, _stream
    if _device is None:
        torch.cuda.init()
        _device = hip.Device(0)
        _stream = hip.Stream(_device)
    return _device, _stream


class _Memory:
    """A library buffer as torch sees it."""

    def __init__(self, buf, shape, typestr):
        self.buf = buf
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=typestr, data=(buf.device_ptr, False),
                                             version=2)


_TYPESTR = {torch.float32: "<f4", torch.float16: "<f2", torch.int32: "<i4", torch.uint8: "|u1"}


def _view(buf, shape, dtype=torch.float32):
    return torch.as_tensor(_Memory(buf, shape, _TYPESTR[dtype]), device="cuda")


def _upload(t):
    """A library buffer that holds t."""
    dev, _ = _open()
    buf = dev.alloc(max(4, t.numel() * t.element_size()))
    if t.numel():
        _view(buf, t.shape, t.dtype).copy_(t)
    return buf


def _empty(*shape):
    dev, _ = _open()
    return dev.alloc(4 * math.prod(shape))


class _Captured:
    """A plan recorded once and captured into a graph, replayed by every pass."""

    def __init__(self, build):
        dev, stream = _open()
        torch.cuda.synchronize()
        self.stream = stream
        self.plan = hip.Plan(dev)
        build(self.plan)
        self.graph = hip.Graph(self.plan, stream, None)

    def replay(self):
        self.graph.replay(self.stream)

    def __del__(self):
        try:
            self.graph.destroy()
            self.plan.destroy()
        except Exception:
            pass


# ------------------------------------------------------------------- inputs

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 % (1 << 62) + 17)


def _normal(g, *shape, sigma=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * sigma


def _norm_weight(g, n):
    return 1.0 + _normal(g, n, sigma=0.05)


def _packed(g, rows, cols, dtype=Q4_K):
    """Random super-blocks [rows][cols / 256][block bytes], dequantized spread about 0.02."""
    nb = rows * cols // 256
    b = torch.randint(0, 256, (nb, BLOCK_BYTES[dtype]), generator=g, device="cuda", dtype=torch.uint8)

    def put(at, values):
        b[:, at:at + 2] = values.to(torch.float16).view(torch.uint8).reshape(nb, 2)

    if dtype == Q4_K:
        d = _normal(g, nb, sigma=1.4e-4).abs()
        put(0, d)
        put(2, 3.75 * d)
    else:
        b[:, 192:208] = torch.randint(-31, 32, (nb, 16), generator=g, device="cuda", dtype=torch.int8).view(torch.uint8)
        put(208, _normal(g, nb, sigma=1.0e-4).abs())
    return b.reshape(rows, cols // 256, BLOCK_BYTES[dtype])


def _dequant(b, dtype=Q4_K):
    """Packed rows in float64 [rows][cols]."""
    rows, nsb, nbytes = b.shape
    b = b.reshape(-1, nbytes)

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).to(torch.float64)

    if dtype == Q4_K:
        s = b[:, 4:16].to(torch.int32)
        lo, mid, hi = s[:, 0:4], s[:, 4:8], s[:, 8:12]
        sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1)
        mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1)
        q = b[:, 16:144].reshape(-1, 4, 32)
        q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32)
        w = (half(0) * sc).unsqueeze(2) * q - (half(2) * mn).unsqueeze(2)
    else:
        ql, qh = b[:, 0:128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)
        high = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
        q = (low | (high << 4)).to(torch.int32) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8)
        w = (half(208) * sc).unsqueeze(2) * q.reshape(-1, 16, 16)
    return w.reshape(rows, nsb * 256)


def _inputs(case, seed):
    """Everything a case's program has in hand, as torch tensors on the GPU."""
    g = _generator(seed)
    c, kind = case, case["kind"]
    if kind == "proj":
        return dict(x=_normal(g, c["rows"], c["n_in"]), w=_packed(g, c["n_out"], c["n_in"], DTYPES[c["dtype"]]))
    if kind == "ffn":
        h, f = c["hidden"], c["ffn"]
        return dict(x=_normal(g, c["rows"], h), norm=_norm_weight(g, h), gate=_packed(g, f, h), up=_packed(g, f, h),
                    down=_packed(g, h, f))
    if kind == "gdn":
        h, n, req, rows = c["hidden"], c["heads"], c["requests"], c["rows"]
        groups = min(n, 16)
        inner, cd = n * STATE, (2 * groups + n) * STATE
        accepted = torch.randint(0, rows, (req,), generator=g, device="cuda", dtype=torch.int32)
        result = torch.zeros(req, 4, device="cuda", dtype=torch.int32)
        result[:, 0] = accepted
        return dict(x=_normal(g, req * rows, h), norm=_norm_weight(g, h), qkv=_packed(g, cd, h),
                    z=_packed(g, inner, h), beta=_packed(g, n, h), alpha=_packed(g, n, h), out=_packed(g, h, inner),
                    conv=_normal(g, cd, CONV, sigma=0.3), dt=_normal(g, n, sigma=0.5),
                    a=-(0.2 + 1.8 * torch.rand(n, generator=g, device="cuda")), head_norm=_norm_weight(g, STATE),
                    conv_state=_normal(g, req, cd, CONV - 1), state=_normal(g, req, n, STATE, STATE, sigma=0.1),
                    result=result)
    if kind == "attn":
        h, nh, nk, req, rows, ctx = c["hidden"], c["heads"], c["kv_heads"], c["requests"], c["rows"], c["context"]
        kvd, blocks = nk * HEAD_DIM, -(-(ctx + rows) // BLOCK)
        pool_type = torch.float16 if c["kv"] == "f16" else torch.float32
        # the requests' contexts differ by a few tokens, the last one is whole
        pos = ctx - torch.randint(0, max(1, min(ctx, 64)), (req,), generator=g, device="cuda", dtype=torch.int32)
        pos[-1] = ctx
        dyn = torch.stack([torch.zeros_like(pos), pos], 1).contiguous()
        table = torch.randperm(req * blocks, generator=g, device="cuda").to(torch.int32).reshape(req, blocks)
        return dict(x=_normal(g, req * rows, h), norm=_norm_weight(g, h), q=_packed(g, nh * HEAD_DIM * 2, h),
                    k=_packed(g, kvd, h), v=_packed(g, kvd, h, Q6_K), o=_packed(g, h, nh * HEAD_DIM),
                    q_norm=_norm_weight(g, HEAD_DIM), k_norm=_norm_weight(g, HEAD_DIM), dyn=dyn, table=table,
                    kpool=_normal(g, req * blocks * BLOCK, kvd).to(pool_type),
                    vpool=_normal(g, req * blocks * BLOCK, kvd).to(pool_type))
    if kind == "moe":
        h, f, e = c["hidden"], c["expert_ffn"], c["experts"]
        return dict(x=_normal(g, c["rows"], h), norm=_norm_weight(g, h), router=_normal(g, e, h, sigma=h ** -0.5),
                    shared_gate=_normal(g, h, sigma=h ** -0.5), gate=_packed(g, (e + 1) * f, h),
                    up=_packed(g, (e + 1) * f, h), down=_packed(g, (e + 1) * h, f))
    if kind == "accept":
        req, k, v = c["requests"], c["drafts"], c["vocab"]
        logits = _normal(g, req, k + 1, v, sigma=3.0)
        guess = torch.randint(0, v, (req, k), generator=g, device="cuda", dtype=torch.int32)
        hit = torch.rand(req, k, generator=g, device="cuda") < 0.7
        return dict(logits=logits, drafts=torch.where(hit, logits[:, :k].argmax(2).to(torch.int32), guess))
    raise ValueError(kind)


# -------------------------------------------------------------------- model

_host = {}


def _model(layers, rows):
    """The 4B-like decoder's configuration and host weights: four layers of bytes, repeated to the depth."""
    cfg = model.replace(model.QWEN35_4B_LIKE, n_layers=layers, capacity=256, max_rows=max(16, rows))
    if "weights" not in _host:
        _host["weights"] = model.make_weights(model.replace(cfg, n_layers=4), seed=1)
    w = dict(_host["weights"])
    w["layers"] = (w["layers"] * -(-layers // 4))[:layers]
    return cfg, w


class _Request:
    """An engine and one request's prompt, drafts and accepted lengths."""

    def __init__(self, case, seed):
        dev, _ = _open()
        cfg, weights = _model(case["layers"], case["rows"])
        self.prompt, self.tokens, self.accepted = _request_tokens(case, seed)
        self.accept = model.accept_struct()
        self.engine = model.Engine(dev, cfg, weights)

    def run(self):
        e = self.engine
        e.reset()
        e.prefill(self.prompt, want_logits=False)
        for tokens, accepted in zip(self.tokens, self.accepted):
            e.step_batch(tokens[None], accept=self.accept, forced=accepted[None])
        return e.logits(self.tokens.shape[1])

    def __del__(self):
        try:
            self.engine.close()
        except Exception:
            pass


def _request_tokens(case, seed):
    rng = np.random.default_rng(seed)
    return (rng.integers(0, VOCAB, case["prompt"], dtype=np.int32),
            rng.integers(0, VOCAB, (case["steps"], case["rows"]), dtype=np.int32),
            rng.integers(0, case["rows"], case["steps"], dtype=np.int32))


# ------------------------------------------------------------------ prepare

def _fused(plan, x, n_in, rows, segments, epilogue=0, norm=None, out_map=0, gate=None, head_norm=None):
    """One GEMM_FUSED op; segments: (weight, dtype, n_out, out, residual)."""
    bufs = [x, norm] + [None] * 14
    n = [n_in, rows, 0, 0, 0, 0]
    types = 0
    for i, (w, dtype, n_out, out, res) in enumerate(segments):
        bufs[2 + i], bufs[6 + i], bufs[10 + i] = w, out, res
        n[2 + i] = n_out
        types |= dtype << (8 * i)
    bufs[14], bufs[15] = gate, head_norm
    plan.add(hip.OP["GEMM_FUSED"], bufs, n=n, u=[types, epilogue, out_map], f=[EPS])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "model":
        return _Request(case, seed)
    dev, stream = _open()
    t = _inputs(case, seed)
    state = dict(kind=kind, case=case)
    if kind == "moe":  # the packed expert layout, rewritten once at load
        raw = {n: _upload(t.pop(n)) for n in ("gate", "up", "down")}
        torch.cuda.synchronize()
        b = {n: dev.alloc(r.nbytes) for n, r in raw.items()}
        h, f, e = case["hidden"], case["expert_ffn"], case["experts"] + 1
        for n, (rows, cols) in dict(gate=(e * f, h), up=(e * f, h), down=(e * h, f)).items():
            hip.moe_pack_q4k(stream, b[n], raw[n], rows, cols)
        stream.sync()
        b.update({n: _upload(v) for n, v in t.items()})
    else:
        b = {n: _upload(v) for n, v in t.items()}
    globals()["_prepare_" + kind](state, b)
    torch.cuda.synchronize()
    return state


def _prepare_proj(state, b):
    c = state["case"]
    out = _empty(c["rows"], c["n_out"])
    state.update(b, out=out, outputs=_view(out, (c["rows"], c["n_out"])), dtype=DTYPES[c["dtype"]])


def _prepare_ffn(state, b):
    c = state["case"]
    rows, h, f = c["rows"], c["hidden"], c["ffn"]
    act, out = _empty(rows, f), _empty(rows, h)

    def build(plan):
        _fused(plan, b["x"], h, rows, [(b["gate"], Q4_K, f, act, None), (b["up"], Q4_K, f, None, None)], epilogue=2,
               norm=b["norm"])
        _fused(plan, act, f, rows, [(b["down"], Q4_K, h, out, b["x"])], epilogue=1)

    state.update(graph=_Captured(build), outputs=[_view(act, (rows, f)), _view(out, (rows, h))])


def _prepare_gdn(state, b):
    c = state["case"]
    req, rows, h, n = c["requests"], c["rows"], c["hidden"], c["heads"]
    groups, r = min(n, 16), req * rows
    inner, cd = n * STATE, (2 * groups + n) * STATE
    qkv, conv, z, raw = _empty(r, cd), _empty(r, cd), _empty(r, inner), _empty(r, inner)
    alpha, beta, out = _empty(r, n), _empty(r, n), _empty(r, h)
    dt_a = _upload(torch.cat([_view(b["dt"], (n,)), _view(b["a"], (n,))]))
    dims = [rows, groups, n, STATE, cd, inner]

    def build(plan):
        _fused(plan, b["x"], h, r, [(b["qkv"], Q4_K, cd, qkv, None), (b["z"], Q4_K, inner, z, None),
                                    (b["beta"], Q4_K, n, beta, None), (b["alpha"], Q4_K, n, alpha, dt_a)],
               norm=b["norm"], out_map=(1 << 4) | (2 << 8) | (3 << 12))
        plan.add(hip.OP["RECURRENT_CHUNK"],
                 [b["conv_state"], b["state"], qkv, z, alpha, beta, b["conv"], b["dt"], b["a"], b["head_norm"], raw,
                  conv], n=dims, u=[CONV, req], f=[EPS, STATE ** -0.5], flags=FLAG_DEFER | FLAG_RAW_OUT | FLAG_GDN_COEF)
        _fused(plan, raw, inner, r, [(b["out"], Q4_K, h, out, b["x"])], epilogue=1, gate=z, head_norm=b["head_norm"])
        plan.add(hip.OP["GDN_COMMIT"], [b["conv_state"], b["state"], qkv, conv, alpha, beta, b["dt"], b["a"],
                                        b["result"]], n=dims, u=[CONV, req], flags=FLAG_GDN_COEF)

    state.update(graph=_Captured(build),
                 outputs=[_view(out, (r, h)), _view(b["state"], (req, n, STATE, STATE)),
                          _view(b["conv_state"], (req, cd, CONV - 1))])


def _prepare_attn(state, b):
    c = state["case"]
    req, rows, h, nh, nk, ctx = c["requests"], c["rows"], c["hidden"], c["heads"], c["kv_heads"], c["context"]
    r, kvd, kv = req * rows, nk * HEAD_DIM, DTYPES[c["kv"]]
    blocks = -(-(ctx + rows) // BLOCK)
    q, k, v = _empty(r, nh * HEAD_DIM * 2), _empty(r, kvd), _empty(r, kvd)
    rope, attn, out = _empty(r, ROPE_DIM), _empty(r, nh * HEAD_DIM), _empty(r, h)

    def build(plan):
        plan.add(hip.OP["ROPE_TABLE"], [rope] + [None] * 14 + [b["dyn"]], n=[rows, ROPE_DIM, 0, req, rows],
                 f=[ROPE_BASE], flags=FLAG_OWN_POS)
        _fused(plan, b["x"], h, r, [(b["q"], Q4_K, nh * HEAD_DIM * 2, q, None), (b["k"], Q4_K, kvd, k, None),
                                    (b["v"], Q6_K, kvd, v, None)], norm=b["norm"])
        plan.add(hip.OP["ATTN_VERIFY"],
                 [q, k, v, b["kpool"], b["vpool"], attn, b["table"], b["q_norm"], b["k_norm"], rope] + [None] * 5 +
                 [b["dyn"]], n=[nk, nh, HEAD_DIM, kvd, rows, 0],
                 u=[BLOCK, blocks * BLOCK, kv, ROPE_DIM | (req << 8) | (rows << 20)], f=[HEAD_DIM ** -0.5, EPS],
                 flags=FLAG_OWN_POS)
        _fused(plan, attn, nh * HEAD_DIM, r, [(b["o"], Q4_K, h, out, b["x"])], epilogue=1)

    pool = (req * blocks * BLOCK, kvd), torch.float16 if c["kv"] == "f16" else torch.float32
    state.update(graph=_Captured(build), keep=b, outputs=[_view(out, (r, h)), _view(b["kpool"], *pool),
                                                          _view(b["vpool"], *pool)])


def _prepare_moe(state, b):
    c = state["case"]
    rows, h, f, e, used = c["rows"], c["hidden"], c["expert_ffn"], c["experts"], c["used"]
    y, xn, logits, sg = _empty(rows, h), _empty(rows, h), _empty(rows, e), _empty(rows)
    ids, w, counts = _empty(rows, used), _empty(rows, used), _empty(e)
    a_rows, a_slots, a_w = (_empty(e, rows * used) for _ in range(3))
    act, eo = _empty(rows, used + 1, f), _empty(rows, used + 1, h)
    flags = hip.FLAG_MOE_PACKED | FLAG_MOE_SHARED

    def build(plan):
        plan.add(hip.OP["COPY"], [y, b["x"]], n=[rows * h])  # the residual stream, added to in place
        plan.add(hip.OP["RMSNORM_BATCH"], [y, b["norm"], xn], n=[h, rows, h, h], f=[EPS])
        plan.add(hip.OP["MOE_ROUTER"], [xn, b["router"], logits, b["shared_gate"], sg], n=[h, e, rows])
        plan.add(hip.OP["MOE_ROUTE"], [logits, ids, w, counts, a_rows, a_slots, a_w], n=[rows, e, used])
        plan.add(hip.OP["MOE_GATE_UP"], [xn, b["gate"], b["up"], counts, a_rows, a_slots, act, None],
                 n=[h, f, rows, e, used], u=[Q4_K], flags=hip.FLAG_MOE_SWIGLU | flags)
        plan.add(hip.OP["MOE_DOWN"], [act, b["down"], counts, a_rows, a_slots, eo], n=[f, h, rows, e, used],
                 u=[Q4_K], flags=flags)
        plan.add(hip.OP["MOE_COMBINE"], [y, eo, w, None, sg], n=[h, rows, used], flags=FLAG_MOE_SHARED)

    state.update(graph=_Captured(build), outputs=[_view(y, (rows, h)), _view(logits, (rows, e))])


def _prepare_accept(state, b):
    c = state["case"]
    result = _upload(torch.zeros(c["requests"], 4, device="cuda", dtype=torch.int32))
    params = hip.accept_params(hip.ACCEPT_GREEDY if c["mode"] == "greedy" else hip.ACCEPT_STOCHASTIC, c["requests"],
                               c["drafts"], c["vocab"], temperature=c["temperature"], top_k=c["top_k"],
                               top_p=c["top_p"], seed=7, step=3)
    state.update(b, result=result, params=params, outputs=_view(result, (c["requests"], 4), torch.int32))


# ---------------------------------------------------------------------- run

def run(state):
    if isinstance(state, _Request):
        return state.run()
    kind = state["kind"]
    if kind == "proj":
        c = state["case"]
        hip.lm_head(_stream, state["out"], state["x"], state["w"], c["n_in"], c["n_out"], c["rows"], state["dtype"])
    elif kind == "accept":
        hip.verify_accept(_stream, state["logits"], state["drafts"], state["result"], state["params"])
    else:
        state["graph"].replay()
    return state["outputs"]


# --------------------------------------------------------------------- work

def _weights(rows, cols, dtype=Q4_K):
    return rows * cols // 256 * BLOCK_BYTES[dtype]


def work(case):
    c, kind = case, case["kind"]
    if kind == "proj":
        n = c["n_in"] * c["n_out"]
        return dict(bytes=_weights(c["n_out"], c["n_in"], DTYPES[c["dtype"]]) + 4 * c["rows"] * (c["n_in"] + c["n_out"]),
                    flops=2 * c["rows"] * n)
    if kind == "ffn":
        h, f, r = c["hidden"], c["ffn"], c["rows"]
        return dict(bytes=3 * _weights(f, h) + 4 * (r * (2 * h + f) + h), flops=6 * r * h * f)
    if kind == "gdn":
        h, n, req, rows = c["hidden"], c["heads"], c["requests"], c["rows"]
        inner, cd = n * STATE, (2 * min(n, 16) + n) * STATE
        proj = cd + inner + 2 * n
        state = req * (n * STATE * STATE + cd * (CONV - 1))
        return dict(bytes=_weights(proj, h) + _weights(h, inner) + 4 * (2 * req * rows * h + 2 * state + cd * CONV),
                    flops=2 * req * rows * (proj * h + inner * h + 4 * n * STATE * STATE))
    if kind == "attn":
        h, nh, nk, req, rows, ctx = c["hidden"], c["heads"], c["kv_heads"], c["requests"], c["rows"], c["context"]
        kvd, od = nk * HEAD_DIM, nh * HEAD_DIM
        weights = _weights(2 * od + kvd, h) + _weights(kvd, h, Q6_K) + _weights(h, od)
        cache = 2 * req * (ctx + rows) * kvd * (2 if c["kv"] == "f16" else 4)
        return dict(bytes=weights + cache + 8 * req * rows * h,
                    flops=2 * req * rows * ((3 * od + 2 * kvd) * h + 2 * od * (ctx + rows)))
    if kind == "moe":
        r, h, f, e, used = c["rows"], c["hidden"], c["expert_ffn"], c["experts"], c["used"]
        touched = e * (1 - (1 - used / e) ** r) + 1
        return dict(bytes=touched * 3 * _weights(f, h) + 4 * (e * h + r * (2 * h + e)),
                    flops=2 * r * ((used + 1) * 3 * f * h + (e + 1) * h))
    if kind == "accept":
        n = c["requests"] * (c["drafts"] + 1) * c["vocab"]
        return dict(bytes=4 * n, flops=2 * n)
    cfg = model.replace(model.QWEN35_4B_LIKE, n_layers=c["layers"])
    h, od, kvd = cfg.hidden, cfg.heads * HEAD_DIM, cfg.kv_heads * HEAD_DIM
    full = c["layers"] // cfg.full_interval
    gdn = _weights(cfg.conv_dim + cfg.inner + 2 * cfg.rank, h) + _weights(h, cfg.inner)
    attn = _weights(2 * od + kvd, h) + _weights(kvd, h, Q6_K) + _weights(h, od)
    weights = c["layers"] * 3 * _weights(cfg.ffn, h) + full * attn + (c["layers"] - full) * gdn
    # the prompt's tokens share one pass over the layers' weights; every step reads them and the head again
    per_row = 2 * (weights * 256 // 144)
    head = _weights(VOCAB, h, Q6_K)
    return dict(bytes=(1 + c["steps"]) * weights + c["steps"] * head + 4 * c["rows"] * VOCAB,
                flops=per_row * (c["prompt"] + c["steps"] * c["rows"]) + 2 * c["steps"] * c["rows"] * VOCAB * h)


def tolerance(case):
    kind = case["kind"]
    if kind == "accept":
        return "exact"
    if kind == "model":
        return {"rel": 1e-3}
    # up to 8 rows a projection's activations are rounded to 16-bit integers
    # (3e-5 to 6e-5 from the exact result; a softmax over few keys takes that
    # to 1.6e-4), beyond that to FP16 (up to 3e-4); the grouped expert
    # projections always take the integers
    rows = case["rows"] * case.get("requests", 1)
    if rows > 8 and kind != "moe":
        return {"rel": 1.2e-3}
    return {"rel": 6e-4 if kind == "attn" else 2.5e-4}


# -------------------------------------------------------------------- exact

def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _silu(x):
    return x * torch.sigmoid(x)


def _times(x, w, dtype=Q4_K):
    return x @ _dequant(w, dtype).T


def _exact_ffn(x, t):
    y = _rms(x, t["norm"])
    act = _silu(_times(y, t["gate"])) * _times(y, t["up"])
    return act, x + _times(act, t["down"])


def _exact_gdn(x, t, heads, conv_state, state, accepted):
    """x [requests][rows][hidden]; both states after accepted + 1 rows."""
    groups = min(heads, 16)
    kd = groups * STATE
    y = _rms(x, t["norm"])
    qkv, z = _times(y, t["qkv"]), _silu(_times(y, t["z"]))
    beta = torch.sigmoid(_times(y, t["beta"]))
    decay = torch.exp(torch.nn.functional.softplus(_times(y, t["alpha"]) + t["dt"], threshold=100) * t["a"])
    line = torch.cat([conv_state.transpose(1, 2), qkv], 1)
    rows = x.shape[1]
    cv = _silu(sum(line[:, i:i + rows] * t["conv"][:, i] for i in range(CONV)))

    def unit(v):
        v = v.reshape(*v.shape[:2], groups, STATE)
        v = v / torch.sqrt((v * v).sum(-1, keepdim=True) + EPS)
        return v.repeat(1, 1, heads // groups, 1)

    q, k = unit(cv[..., :kd]) * STATE ** -0.5, unit(cv[..., kd:2 * kd])
    v = cv[..., 2 * kd:].reshape(*cv.shape[:2], heads, STATE)
    kept = state.clone()
    outs = []
    for r in range(rows):
        state = state * decay[:, r, :, None, None]
        d = (v[:, r] - (state * k[:, r, :, :, None]).sum(2)) * beta[:, r, :, None]
        state = state + k[:, r, :, :, None] * d[:, :, None, :]
        outs.append((state * q[:, r, :, :, None]).sum(2))
        kept = torch.where((accepted >= r)[:, None, None, None], state, kept)
    raw = _rms(torch.stack(outs, 1), t["head_norm"]).flatten(2) * z
    window = torch.stack([line[i, a + 1:a + CONV] for i, a in enumerate(accepted.tolist())]).transpose(1, 2)
    return x + _times(raw, t["out"]), kept, window.contiguous()


def _rotate(x, pos):
    """x [rows][heads][HEAD_DIM]: the first ROPE_DIM dimensions, in halves."""
    half = ROPE_DIM // 2
    freq = ROPE_BASE ** (-2.0 * torch.arange(half, device="cuda", dtype=torch.float64) / ROPE_DIM)
    th = pos.to(torch.float64)[:, None] * freq
    co, si = torch.cos(th)[:, None], torch.sin(th)[:, None]
    a, b = x[..., :half], x[..., half:ROPE_DIM]
    return torch.cat([a * co - b * si, a * si + b * co, x[..., ROPE_DIM:]], -1)


def _exact_attn(x, t, heads, kv_heads, pos, past_k, past_v):
    """x [rows][hidden] at positions pos, pos + 1, ...; also the rows' keys and values."""
    rows, hd = x.shape[0], HEAD_DIM
    at = pos + torch.arange(rows, device="cuda")
    y = _rms(x, t["norm"])
    q, gate = _times(y, t["q"]).reshape(rows, heads, 2, hd).unbind(2)
    k = _rotate(_rms(_times(y, t["k"]).reshape(rows, kv_heads, hd), t["k_norm"]), at)
    v = _times(y, t["v"], Q6_K).reshape(rows, kv_heads, hd)
    q = _rotate(_rms(q, t["q_norm"]), at)
    keys, values = torch.cat([past_k, k]), torch.cat([past_v, v])
    out = torch.empty(rows, heads, hd, device="cuda", dtype=torch.float64)
    unseen = torch.arange(keys.shape[0], device="cuda")[None] > at[:, None]
    for h in range(heads):
        j = h * kv_heads // heads
        s = (q[:, h] @ keys[:, j].T * hd ** -0.5).masked_fill(unseen, -math.inf)
        out[:, h] = torch.softmax(s, 1) @ values[:, j]
    return x + _times((out * torch.sigmoid(gate)).flatten(1), t["o"]), k, v


def _exact_moe(x, t, c):
    h, f, e, used = c["hidden"], c["expert_ffn"], c["experts"], c["used"]
    y = _rms(x, t["norm"])
    logits = y @ t["router"].T
    top, ids = logits.topk(used, 1)
    share = torch.softmax(top, 1)
    out = x.clone()

    def expert(i, rows):
        act = _silu(_times(rows, t["gate"][i * f:(i + 1) * f])) * _times(rows, t["up"][i * f:(i + 1) * f])
        return _times(act, t["down"][i * h:(i + 1) * h])

    for i in ids.unique().tolist():
        r, s = (ids == i).nonzero(as_tuple=True)
        out.index_add_(0, r, share[r, s, None] * expert(i, y[r]))
    return out + torch.sigmoid(y @ t["shared_gate"])[:, None] * expert(e, y), logits


def _exact_model(case, seed):
    cfg, w = _model(case["layers"], case["rows"])
    prompt, steps, accepted = _request_tokens(case, seed)
    kept = [prompt] + [s[:a + 1] for s, a in zip(steps[:-1], accepted[:-1])] + [steps[-1]]
    tokens = torch.from_numpy(np.concatenate(kept)).cuda()
    zero = torch.zeros(1, device="cuda", dtype=torch.int64)

    def tensor(v):
        if not isinstance(v, dict):
            return torch.from_numpy(v).cuda().to(torch.float64)
        return torch.from_numpy(v["data"]).cuda().reshape(v["rows"], v["cols"] // 256, BLOCK_BYTES[v["dtype"]])

    x = _dequant(tensor(w["embedding"])[tokens])
    for i in range(case["layers"]):
        t = {n: tensor(v) for n, v in w["layers"][i].items()}
        if cfg.is_recurrent(i):
            t.update(norm=t["attn_norm"], z=t["gate"], head_norm=t["ssm_norm"], conv=t["conv"].reshape(-1, CONV))
            empty = dict(device="cuda", dtype=torch.float64)
            x = _exact_gdn(x[None], t, cfg.rank, torch.zeros(1, cfg.conv_dim, CONV - 1, **empty),
                           torch.zeros(1, cfg.rank, STATE, STATE, **empty), zero)[0][0]
        else:
            t.update(norm=t["attn_norm"])
            none = torch.zeros(0, cfg.kv_heads, HEAD_DIM, device="cuda", dtype=torch.float64)
            x = _exact_attn(x, t, cfg.heads, cfg.kv_heads, 0, none, none)[0]
        x = _exact_ffn(x, dict(norm=t["post_norm"], gate=t["ffn_gate"], up=t["ffn_up"], down=t["ffn_down"]))[1]
    y = _rms(x[-case["rows"]:], tensor(w["output_norm"]))
    return _times(y, tensor(w["output"]), Q6_K).cpu().numpy()


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "accept":
        return None
    if kind == "model":
        return _exact_model(case, seed)
    t = {n: v.to(torch.float64) if v.dtype == torch.float32 else v for n, v in _inputs(case, seed).items()}
    if kind == "proj":
        return _times(t["x"], t["w"], DTYPES[c["dtype"]])
    if kind == "ffn":
        return list(_exact_ffn(t["x"], t))
    if kind == "gdn":
        x = t["x"].reshape(c["requests"], c["rows"], c["hidden"])
        y, state, conv = _exact_gdn(x, t, c["heads"], t["conv_state"], t["state"], t["result"][:, 0])
        return [y.flatten(0, 1), state, conv]
    if kind == "attn":
        kpool, vpool = t["kpool"].to(torch.float64), t["vpool"].to(torch.float64)
        shape, outs = (-1, c["kv_heads"], HEAD_DIM), []
        for r in range(c["requests"]):
            pos = int(t["dyn"][r, 1])
            at = torch.arange(pos + c["rows"], device="cuda")
            at = t["table"][r, at // BLOCK].to(torch.int64) * BLOCK + at % BLOCK
            y, k, v = _exact_attn(t["x"][r * c["rows"]:(r + 1) * c["rows"]], t, c["heads"], c["kv_heads"], pos,
                                  kpool[at[:pos]].reshape(shape), vpool[at[:pos]].reshape(shape))
            kpool[at[pos:]], vpool[at[pos:]] = k.flatten(1), v.flatten(1)
            outs.append(y)
        return [torch.cat(outs), kpool, vpool]
    y, logits = _exact_moe(t["x"], t, c)
    return [y, logits]
