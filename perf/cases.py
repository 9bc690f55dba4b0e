"""The work a user of this library has it do, as cases that can be timed.

A case is a dict of plain values; `kind` names the path and the rest its
sizes:

  linear     one Q4_0 projection of m positions: the Q8_0 quantiser and the
             product, as an engine calls a bare Linear (rows x cols)
  head       the output head of m hidden states: the Q8_K quantiser and the
             Q6_K product, logits out
  ffn        the feed-forward half of a Qwen3 block for m positions: pre-norm,
             Gate|Up with SwiGLU, Down
  attention  the attention half of a Qwen3 block for m new positions after
             `prefix` cached ones: pre-norm, Q|K|V, head norms, RoPE, cache
             stores, attention, O.  slots > 0: one new position in each of
             m = slots conversations (a server's lock-step batch)
  moe        the mixture layer of m positions: router, choice, experts
  model      one decode token of a Qwen3 decoder: embedding, blocks, final
             norm and head (QwenModel.forward and .logits)

The calls of each kind are those golem_amd/qwen.py makes for these sizes (a
single position takes the fused entry points).  Weights, norms and
activations have the distributions of golem_amd/synth.py, drawn on the GPU.
"""
import ctypes
import math

import torch

from golem_amd import capi, qwen, synth

EPS = 1e-6
ROPE_BASE = 1e6
FUSED_MAX = 767     # prefixes the one-kernel decode attention takes
Q4_BYTES = 18 / 32  # bytes a Q4_0 weight
Q6_BYTES = 210 / 256
MOE = {"dim": 2816, "ffn": 704, "experts": 128, "top_k": 8}


def listed():
    qwen_dims = {"dim": 2560, "heads": 32, "kv_heads": 8, "head_dim": 128}
    return [
        # one K or V projection of a decode step: the smallest call there is
        {"name": "linear_one", "kind": "linear", "m": 1, "rows": 1024, "cols": 2560},
        # a long prompt through an FFN projection
        {"name": "linear_prompt", "kind": "linear", "m": 2048, "rows": 9728, "cols": 2560},
        # the logits of a decode step
        {"name": "head_one", "kind": "head", "m": 1, "rows": 151936, "cols": 2560},
        # the logits of six conversations decoded in lock step
        {"name": "head_slots", "kind": "head", "m": 6, "rows": 151936, "cols": 2560},
        # a decode step's feed forward
        {"name": "ffn_one", "kind": "ffn", "m": 1, "dim": 2560, "ffn": 9728},
        # eight conversations' feed forward
        {"name": "ffn_slots", "kind": "ffn", "m": 8, "dim": 2560, "ffn": 9728},
        # a prompt of ordinary length, not a multiple of any tile
        {"name": "ffn_prompt", "kind": "ffn", "m": 500, "dim": 2560, "ffn": 9728},
        # a decode step far into a conversation
        dict(qwen_dims, name="attention_one_long", kind="attention", m=1, prefix=3000, slots=0),
        # a document read in one batch
        dict(qwen_dims, name="attention_prompt_long", kind="attention", m=1500, prefix=0, slots=0),
        # a decode step of the mixture layer
        dict(MOE, name="moe_one", kind="moe", m=1),
        # a prompt's positions grouped by expert
        dict(MOE, name="moe_prompt", kind="moe", m=256),
        # a whole decode token, four blocks deep, in mid-conversation
        {"name": "model_one", "kind": "model", "layers": 4, "prefix": 600, "context": 768},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "head", "ffn", "ffn", "attention", "attention", "attention", "moe",
                       "model"])
    if kind == "linear":
        return {"kind": kind, "m": _log(rng, 1, 1024), "rows": _log(rng, 512, 9728),
                "cols": 32 * rng.choice([22, 32, 65, 80, 88, 128, 304])}
    if kind == "head":
        return {"kind": kind, "m": rng.randint(1, 16), "rows": _log(rng, 4096, 151936),
                "cols": 256 * rng.choice([4, 10, 11])}
    if kind == "ffn":
        dim, ffn = rng.choice([(2560, 9728), (1024, 2816), (512, 1024)])
        return {"kind": kind, "m": _log(rng, 1, 700), "dim": dim, "ffn": ffn}
    if kind == "attention":
        dim, heads, kv, hd = rng.choice([(2560, 32, 8, 128), (2560, 32, 8, 128), (1024, 16, 8, 128),
                                         (512, 8, 2, 64)])
        c = {"kind": kind, "dim": dim, "heads": heads, "kv_heads": kv, "head_dim": hd}
        form = rng.choice(["one", "one", "prompt", "prompt", "slots"])
        if form == "one":
            return dict(c, m=1, prefix=_log(rng, 1, 4000), slots=0)
        if form == "prompt":
            return dict(c, m=_log(rng, 5, 1400), prefix=rng.choice([0, 0, _log(rng, 1, 1500)]), slots=0)
        n = rng.randint(2, 8)
        return dict(c, m=n, prefix=_log(rng, 1, FUSED_MAX - 2), slots=n)
    if kind == "moe":
        dims = rng.choice([MOE, MOE, {"dim": 1024, "ffn": 704, "experts": 64, "top_k": 4}])
        return dict(dims, kind=kind, m=_log(rng, 1, 255) if dims is not MOE else rng.choice([2, 3, _log(rng, 4, 255)]))
    return {"kind": kind, "layers": rng.randint(1, 4), "prefix": _log(rng, 1, 700), "context": 768}


# ---- inputs -------------------------------------------------------------------


def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + salt)
    return g


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _half_bytes(x):
    return x.to(torch.float16).view(torch.uint8)


def _q4_bytes(g, rows, cols):
    """GGUF Q4_0 rows: fp16 |N(0,1)| * 0.02, then 16 random nibble bytes."""
    n = rows * cols // 32
    out = torch.empty((n, 18), dtype=torch.uint8, device="cuda")
    out[:, :2] = _half_bytes(_normal(g, n, 1).abs() * 0.02)
    out[:, 2:] = torch.randint(0, 256, (n, 16), generator=g, device="cuda", dtype=torch.uint8)
    return out


def _q6_bytes(g, rows, cols):
    """GGUF Q6_K rows: ql and qh random, sub-scales -64..63, fp16 d."""
    n = rows * cols // 256
    out = torch.empty((n, 210), dtype=torch.uint8, device="cuda")
    out[:, :192] = torch.randint(0, 256, (n, 192), generator=g, device="cuda", dtype=torch.uint8)
    out[:, 192:208] = torch.randint(-64, 64, (n, 16), generator=g, device="cuda", dtype=torch.int8).view(torch.uint8)
    out[:, 208:] = _half_bytes(_normal(g, n, 1).abs() * 0.002)
    return out


def _gains(g, n):
    return 1.0 + 0.02 * _normal(g, n)


def _rope(context, head_dim):
    """cos and sin of pos * base^(-2i/head_dim), rounded to float32."""
    half = head_dim // 2
    freq = ROPE_BASE ** (-2.0 * torch.arange(half, dtype=torch.float64, device="cuda") / head_dim)
    theta = torch.arange(context, dtype=torch.float64, device="cuda")[:, None] * freq[None, :]
    return theta.cos().float(), theta.sin().float()


def _context_of(case):
    return (case["prefix"] + (1 if case["slots"] else case["m"]) + 7) // 8 * 8


def _cached(g, case):
    """The cached keys and values of `prefix` positions a conversation, in the
    library's cache layouts (fp16 bits); the rest of a cache is zero."""
    n, kv, hd, ctx = max(case["slots"], 1), case["kv_heads"], case["head_dim"], _context_of(case)
    kc = torch.zeros((n, kv, hd // 8, ctx, 8), dtype=torch.float16, device="cuda")
    vc = torch.zeros((n, kv, hd, ctx), dtype=torch.float16, device="cuda")
    p = case["prefix"]
    kc[:, :, :, :p] = _normal(g, n, kv, hd // 8, p, 8).half()
    vc[:, :, :, :p] = (4.0 * _normal(g, n, kv, hd, p)).half()
    return kc, vc


def _inputs(case, seed):
    """The tensors of a case, from the seed alone: what prepare() lays out for
    the library and exact() computes with."""
    g = _gen(seed, 17)
    k = case["kind"]
    if k == "linear":
        return {"w": _q4_bytes(g, case["rows"], case["cols"]), "x": _normal(g, case["m"], case["cols"])}
    if k == "head":
        return {"w": _q6_bytes(g, case["rows"], case["cols"]), "x": _normal(g, case["m"], case["cols"])}
    if k == "ffn":
        return {"gu": _q4_bytes(g, 2 * case["ffn"], case["dim"]), "down": _q4_bytes(g, case["dim"], case["ffn"]),
                "gain": _gains(g, case["dim"]), "x": _normal(g, case["m"], case["dim"]),
                "add": _normal(g, case["m"], case["dim"])}
    if k == "attention":
        qd, kvd = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
        i = {"qkv": _q4_bytes(g, qd + 2 * kvd, case["dim"]), "o": _q4_bytes(g, case["dim"], qd),
             "gain": _gains(g, case["dim"]), "q_norm": _gains(g, case["head_dim"]),
             "k_norm": _gains(g, case["head_dim"]), "x": _normal(g, case["m"], case["dim"])}
        i["cos"], i["sin"] = _rope(_context_of(case), case["head_dim"])
        i["kc"], i["vc"] = _cached(g, case)
        return i
    if k == "moe":
        e, d, f = case["experts"], case["dim"], case["ffn"]
        return {"router": 0.02 * _normal(g, e, d), "router_scale": _gains(g, d), "down_scale": _gains(g, e),
                "gu": _q4_bytes(g, e * 2 * f, d), "down": _q4_bytes(g, e * d, f),
                "x": _normal(g, case["m"], d)}
    cfg = _model_config(case)
    qd, kvd = cfg.heads * cfg.head_dim, cfg.kv_heads * cfg.head_dim
    blocks, caches = [], []
    half = {"kv_heads": cfg.kv_heads, "head_dim": cfg.head_dim, "slots": 0, "m": case["context"] - case["prefix"],
            "prefix": case["prefix"]}
    for _ in range(cfg.layers):
        blocks.append({
            "attn_norm": _gains(g, cfg.dim), "q": _q4_bytes(g, qd, cfg.dim), "q_norm": _gains(g, cfg.head_dim),
            "k": _q4_bytes(g, kvd, cfg.dim), "k_norm": _gains(g, cfg.head_dim), "v": _q4_bytes(g, kvd, cfg.dim),
            "o": _q4_bytes(g, cfg.dim, qd), "ffn_norm": _gains(g, cfg.dim),
            "gate": _q4_bytes(g, cfg.ffn, cfg.dim), "up": _q4_bytes(g, cfg.ffn, cfg.dim),
            "down": _q4_bytes(g, cfg.dim, cfg.ffn)})
        caches.append(_cached(g, half))
    return {"blocks": blocks, "caches": caches, "output_norm": _gains(g, cfg.dim),
            "token_embd": _q6_bytes(g, cfg.vocab, cfg.dim),
            "token": torch.randint(0, cfg.vocab, (1,), generator=g, device="cuda", dtype=torch.int32)}


def _model_config(case):
    c = synth.qwen3_4b(case["context"])
    c.layers = case["layers"]
    return c


# ---- what a program holds before the call ---------------------------------------


class _State:
    """A case's device buffers and weights; the weights go with it."""

    def __init__(self, case):
        self.case = case
        self.ctx = capi.Context(0, stream=torch.cuda.current_stream().cuda_stream)
        self.weights = []
        self.model = None

    def weight(self, data, quant, rows, cols, count=1):
        torch.cuda.current_stream().synchronize()
        w = capi.Weight(self.ctx, (data.data_ptr(), data.numel() * data.element_size()), quant, rows, cols, count)
        self.ctx.sync()
        self.weights.append(w)
        return w

    def __del__(self):
        try:
            torch.cuda.synchronize()
            if self.model is not None:
                self.model.free()
            for w in self.weights:
                w.free()
            self.ctx.close()
        except Exception:  # the interpreter is going down
            pass


def _empty(shape, dtype):
    return torch.empty(shape, dtype=dtype, device="cuda")


def _q8(m, k):
    return _empty((m, k), torch.int8), _empty((m, k // 32), torch.float32), _empty((m, k // 32), torch.int32)


def prepare(case, seed):
    i, s = _inputs(case, seed), _State(case)
    k, m = case["kind"], case.get("m", 1)
    if k == "linear":
        s.x, s.act, s.y = i["x"], _q8(m, case["cols"]), _empty((m, case["rows"]), torch.float32)
        s.w = s.weight(i["w"], capi.Q4_0, case["rows"], case["cols"])
    elif k == "head":
        s.x, s.y = i["x"], _empty((m, case["rows"]), torch.float32)
        s.act = (_empty((m, case["cols"]), torch.int8), _empty((m, case["cols"] // 256), torch.float32),
                 _empty((m, case["cols"] // 16), torch.int16))
        s.w = s.weight(i["w"], capi.Q6_K, case["rows"], case["cols"])
    elif k == "ffn":
        d, f = case["dim"], case["ffn"]
        s.x, s.add, s.gain = i["x"], i["add"], i["gain"]
        s.normed, s.mid = _q8(m, d), _q8(m, f)
        s.x_out, s.y = _empty((m, d), torch.float32), _empty((m, d), torch.float32)
        s.gu = s.weight(i["gu"], capi.Q4_0, 2 * f, d)
        s.down = s.weight(i["down"], capi.Q4_0, d, f)
    elif k == "attention":
        d, hd = case["dim"], case["head_dim"]
        qd, kvd = case["heads"] * hd, case["kv_heads"] * hd
        for n in ("x", "gain", "q_norm", "k_norm", "cos", "sin", "kc", "vc"):
            setattr(s, n, i[n])
        s.context = _context_of(case)
        s.qkv, s.o = s.weight(i["qkv"], capi.Q4_0, qd + 2 * kvd, d), s.weight(i["o"], capi.Q4_0, d, qd)
        s.normed, s.set8 = _q8(m, d), _q8(m, qd)
        s.rows, s.qh = _empty((m, qd + 2 * kvd), torch.float32), _empty((m, qd), torch.int16)
        s.y = _empty((m, d), torch.float32)
        first = case["prefix"]
        s.max_pos = first + (0 if case["slots"] else m - 1)
        s.positions = torch.full((m,), first, dtype=torch.int32, device="cuda") if case["slots"] else torch.arange(
            first, first + m, dtype=torch.int32, device="cuda")
        s.slots = torch.arange(m, dtype=torch.int32, device="cuda") if case["slots"] else None
        n = capi.size_out("gx_qwen_attention_workspace_bytes", m, case["heads"], s.max_pos)
        s.ws = _empty(((n + 255) // 256 * 256,), torch.uint8)
    elif k == "moe":
        e, d, f, tk = case["experts"], case["dim"], case["ffn"], case["top_k"]
        for n in ("x", "router_scale", "down_scale"):
            setattr(s, n, i[n])
        s.router = s.weight(i["router"], capi.F32, e, d)
        s.gu = s.weight(i["gu"], capi.Q4_0, 2 * f, d, e)
        s.down = s.weight(i["down"], capi.Q4_0, d, f, e)
        s.logits, s.ids = _empty((m, e), torch.float32), _empty((m, tk), torch.int32)
        s.route, s.y = _empty((m, tk), torch.float32), _empty((m, d), torch.float32)
        n = capi.size_out("gx_moe_workspace_bytes", m, tk, d, f, e)
        s.ws = _empty(((n + 255) // 256 * 256,), torch.uint8)
    else:
        def host(v):
            return [host(u) for u in v] if isinstance(v, list) else {n: host(u) for n, u in v.items()} if isinstance(
                v, dict) else v.cpu().numpy() if v.dtype == torch.float32 else v.reshape(-1).cpu().numpy()

        w = host({n: i[n] for n in ("blocks", "output_norm", "token_embd")})
        s.model = qwen.QwenModel(s.ctx, _model_config(case), w, max_batch=1)
        for at, (kc, vc) in enumerate(i["caches"]):
            s.model.kc[at].copy_(kc.view(torch.int16))
            s.model.vc[at].copy_(vc.view(torch.int16))
        s.token = i["token"]
    torch.cuda.synchronize()
    return s


# ---- one pass ---------------------------------------------------------------------


def run(s):
    case, vp, call, ctx = s.case, capi.vp, capi.call, s.ctx.ptr
    k, m, eps = case["kind"], case.get("m", 1), ctypes.c_float(EPS)
    if k == "linear":
        q, sc, qs = s.act
        rows, cols = case["rows"], case["cols"]
        call("gx_quantize_q8_0", ctx, vp(s.x), cols, m, cols, vp(q), vp(sc), vp(qs), None, None)
        call("gx_matmul_q4_0", ctx, s.w.ptr, vp(q), vp(sc), vp(qs), None, m, 0, rows, None, vp(s.y), rows)
        return s.y
    if k == "head":
        q, ks, bs = s.act
        rows, cols = case["rows"], case["cols"]
        call("gx_quantize_q8_k", ctx, vp(s.x), cols, m, cols, vp(q), vp(ks), vp(bs))
        call("gx_matmul_q6_k", ctx, s.w.ptr, vp(q), vp(ks), vp(bs), m, 0, rows, None, vp(s.y), rows)
        return s.y
    if k == "ffn":
        d, mid = case["dim"], s.mid
        if m == 1:
            call("gx_norm_swiglu_q4_0", ctx, s.gu.ptr, vp(s.x), vp(s.add), vp(s.gain), eps, vp(s.x_out), vp(mid[0]),
                 vp(mid[1]), vp(mid[2]))
        else:
            q, sc, qs = s.normed
            call("gx_norm_quant", ctx, vp(s.x), d, None, d, vp(s.gain), m, d, eps, None, 0, vp(q), vp(sc), vp(qs))
            call("gx_matmul_swiglu_q4_0", ctx, s.gu.ptr, vp(q), vp(sc), vp(qs), m, vp(mid[0]), vp(mid[1]),
                 vp(mid[2]))
        call("gx_matmul_q4_0", ctx, s.down.ptr, vp(mid[0]), vp(mid[1]), vp(mid[2]), None, m, 0, d, None, vp(s.y), d)
        return {"y": s.y, "x": s.x_out} if m == 1 else {"y": s.y}
    if k == "attention":
        d, h, kv, hd = case["dim"], case["heads"], case["kv_heads"], case["head_dim"]
        q, sc, qs = s.set8
        nq, ns, nqs = s.normed
        width = (h + 2 * kv) * hd
        heads = (vp(s.positions), vp(s.q_norm), vp(s.k_norm), vp(s.cos), vp(s.sin), eps)
        caches = (vp(s.kc), vp(s.vc), s.context)
        out = (vp(q), vp(sc), vp(qs))
        if m == 1 and not case["slots"]:
            call("gx_norm_matmul_q4_0", ctx, s.qkv.ptr, vp(s.x), None, vp(s.gain), eps, None, 0, width, vp(s.rows))
            if s.max_pos < FUSED_MAX:
                call("gx_qwen_rope_attention_parallel", ctx, vp(s.rows), width, h, kv, hd, s.max_pos, *heads,
                     *caches, *out, None, 0)
            else:
                call("gx_qwen_qk_rope", ctx, vp(s.rows), width, 1, h, kv, hd, *heads, vp(s.qh), *caches, None, 0)
                call("gx_qwen_attention_parallel", ctx, vp(s.qh), 1, h, kv, hd, s.max_pos, vp(s.positions), *caches,
                     *out, vp(s.ws), s.ws.numel(), None, 0)
        else:
            call("gx_norm_quant", ctx, vp(s.x), d, None, d, vp(s.gain), m, d, eps, None, 0, vp(nq), vp(ns), vp(nqs))
            if case["slots"]:
                call("gx_matmul_q4_0", ctx, s.qkv.ptr, vp(nq), vp(ns), vp(nqs), None, m, 0, width, None, vp(s.rows),
                     width)
                call("gx_qwen_rope_attention_slots", ctx, vp(s.rows), width, m, h, kv, hd, s.max_pos, *heads,
                     *caches, *out, vp(s.slots), m, 1)
            else:
                call("gx_qwen_qkv_rope", ctx, s.qkv.ptr, vp(nq), vp(ns), vp(nqs), m, h, kv, hd, *heads, vp(s.qh),
                     *caches, None, 0, vp(s.rows))
                call("gx_qwen_attention_parallel", ctx, vp(s.qh), m, h, kv, hd, s.max_pos, vp(s.positions), *caches,
                     *out, vp(s.ws), s.ws.numel(), None, 0)
        call("gx_matmul_q4_0", ctx, s.o.ptr, vp(q), vp(sc), vp(qs), None, m, 0, d, None, vp(s.y), d)
        return {"y": s.y, "keys": s.kc, "values": s.vc}
    if k == "moe":
        d, tk = case["dim"], case["top_k"]
        call("gx_moe_route", ctx, s.router.ptr, vp(s.router_scale), vp(s.x), d, m, tk, eps, vp(s.logits), vp(s.ids),
             vp(s.route))
        call("gx_moe_experts", ctx, s.gu.ptr, s.down.ptr, vp(s.down_scale), vp(s.x), d, m, tk, vp(s.ids),
             vp(s.route), vp(s.y), d, vp(s.ws), s.ws.numel())
        return {"y": s.y, "logits": s.logits, "weights": s.route, "ids": s.ids}
    hidden = s.model.forward(s.token, case["prefix"])
    logits = s.model.logits(0)
    return {"logits": logits, "hidden": hidden, "keys": [c.view(torch.float16) for c in s.model.kc],
            "values": [c.view(torch.float16) for c in s.model.vc]}


# ---- what a pass cannot do without ---------------------------------------------------


def work(case):
    k, m = case["kind"], case.get("m", 1)
    if k == "linear":
        r, c = case["rows"], case["cols"]
        return {"bytes": r * c * Q4_BYTES + 4 * m * (r + c), "flops": 2 * m * r * c}
    if k == "head":
        r, c = case["rows"], case["cols"]
        return {"bytes": r * c * Q6_BYTES + 4 * m * (r + c), "flops": 2 * m * r * c}
    if k == "ffn":
        d, f = case["dim"], case["ffn"]
        return {"bytes": 3 * d * f * Q4_BYTES + 4 * d + 4 * m * d * (4 if m == 1 else 2), "flops": 6 * m * d * f}
    if k == "attention":
        return _attention_work(case, m, case["prefix"], case["slots"], case)
    if k == "moe":
        e, d, f, tk = case["experts"], case["dim"], case["ffn"], case["top_k"]
        touched = e * (1.0 - (1.0 - tk / e) ** m)  # experts that m positions choose, on average
        return {"bytes": touched * 3 * d * f * Q4_BYTES + 4 * (e * d + d + e) + 4 * m * (2 * d + e + 2 * tk),
                "flops": 2 * m * (e * d + tk * 3 * d * f)}
    c = _model_config(case)
    one = {"dim": c.dim, "heads": c.heads, "kv_heads": c.kv_heads, "head_dim": c.head_dim}
    a = _attention_work(one, 1, case["prefix"], 0, one)
    head = c.vocab * c.dim * Q6_BYTES + c.dim * Q6_BYTES + 4 * (c.vocab + c.dim)
    return {"bytes": c.layers * (a["bytes"] + 3 * c.dim * c.ffn * Q4_BYTES) + head,
            "flops": c.layers * (a["flops"] + 6 * c.dim * c.ffn) + 2 * c.vocab * c.dim}


def _attention_work(case, m, prefix, slots, dims):
    d, hd = dims["dim"], dims["head_dim"]
    qd, kvd = dims["heads"] * hd, dims["kv_heads"] * hd
    cached = (slots or 1) * prefix * 2 * kvd * 2
    pairs = m * (prefix + 1) if slots else m * prefix + m * (m + 1) / 2
    return {"bytes": (d * (qd + 2 * kvd) + d * qd) * Q4_BYTES + cached + m * 2 * kvd * 2 + 4 * m * 2 * d,
            "flops": 2 * m * (d * (qd + 2 * kvd) + d * qd) + 4 * pairs * qd}


def tolerance(case):
    # linear, head: 32-bit sums of exact block integers.  The others quantise
    # their own intermediate values: one that sits between two steps moves by
    # a step when a sum's last bit does.
    return {"linear": {"rel": 1e-6}, "head": {"rel": 1e-6}, "ffn": {"rel": 1e-3}, "attention": {"rel": 3e-3},
            "moe": {"rel": 1e-3, "differ": 0.002}, "model": {"rel": 1e-2}}[case["kind"]]


# ---- the same in 64 bits ---------------------------------------------------------------


def _deq4(b, rows, cols):
    d = b[:, :2].contiguous().view(torch.float16).double()
    n = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8.0
    return (d * n).reshape(rows, cols)


def _deq6(b, rows, cols):
    n = b.shape[0]
    ql, qh = b[:, :128].reshape(n, 2, 64), b[:, 128:192].reshape(n, 2, 32)
    lo = torch.cat([ql[:, :, :32] & 15, ql[:, :, 32:] & 15, ql[:, :, :32] >> 4, ql[:, :, 32:] >> 4], 2)
    hi = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
    q = (lo | (hi << 4)).double() - 32.0  # [n][2][128]
    sc = b[:, 192:208].contiguous().view(torch.int8).double().repeat_interleave(16, 1).reshape(n, 2, 128)
    d = b[:, 208:].contiguous().view(torch.float16).double()[:, :, None]
    return (d * sc * q).reshape(rows, cols)


def _q8_0(x):
    """The Q8_0 form of float32(x), expanded again: the format's own steps."""
    b = x.float().reshape(-1, 32)
    peak = b.abs().amax(1, keepdim=True)
    top = torch.full_like(peak, 127.0)  # tensors divided: torch takes a number's reciprocal first
    inv = torch.where(peak > 0, top / peak, torch.zeros_like(peak))
    n = (b * inv).round().clamp(-128, 127).double()
    return (n * (peak / top).half().double()).reshape(x.shape)


def _q8_k(x):
    b = x.float().reshape(-1, 256)
    ext = b.gather(1, b.abs().argmax(1, keepdim=True))
    inv = torch.where(ext != 0, torch.full_like(ext, -128.0) / ext, torch.zeros_like(ext))
    n = (b * inv).round().clamp(max=127).double()
    ks = torch.where(ext != 0, 1.0 / inv, torch.zeros_like(inv)).double()
    return (n * ks).reshape(x.shape)


def _rms(x, gain=None):
    x = x.double()
    y = x / (x.pow(2).mean(-1, keepdim=True) + EPS).sqrt()
    return y if gain is None else y * gain.double()


def _half(x):
    return x.float().half().double()


def _ffn64(x, gain, gu, down, dim, ffn):
    """Gate and up rows of gu interleaved by 32."""
    w = _deq4(gu, 2 * ffn, dim).reshape(ffn // 32, 2, 32, dim)
    a = _q8_0(_rms(x, gain))
    g, u = a @ w[:, 0].reshape(ffn, dim).T, a @ w[:, 1].reshape(ffn, dim).T
    return _q8_0(g * torch.sigmoid(g) * u) @ _deq4(down, dim, ffn).T


def _attention64(i, case, x, positions):
    """The attention half in 64 bits: (O's output, key cache, value cache).
    Queries, cache entries and probabilities are fp16, as they are stored."""
    h, kv, hd, d = case["heads"], case["kv_heads"], case["head_dim"], case["dim"]
    qd, kvd, m = h * hd, kv * hd, x.shape[0]
    rows = _q8_0(_rms(x, i["gain"])) @ _deq4(i["qkv"], qd + 2 * kvd, d).T
    cos, sin = i["cos"].double()[positions.long()][:, None], i["sin"].double()[positions.long()][:, None]

    def rope(v, gain):
        v = _rms(v, gain)
        a, b = v[..., : hd // 2], v[..., hd // 2:]
        return _half(torch.cat([a * cos - b * sin, a * sin + b * cos], -1))

    q = rope(rows[:, :qd].reshape(m, h, hd), i["q_norm"])
    k = rope(rows[:, qd:qd + kvd].reshape(m, kv, hd), i["k_norm"])
    v = _half(rows[:, qd + kvd:].reshape(m, kv, hd))
    kc, vc = i["kc"].double(), i["vc"].double()
    slot = torch.arange(m, device="cuda") if case.get("slots") else torch.zeros(m, dtype=torch.long, device="cuda")
    pos = positions.long()
    kc[slot, :, :, pos] = k.reshape(m, kv, hd // 8, 8)
    vc[slot, :, :, pos] = v
    heads = torch.empty((m, h, hd), dtype=torch.float64, device="cuda")
    top = int(pos.max()) + 1
    at = torch.arange(top, device="cuda")
    for j in range(h):
        if case.get("slots"):
            ks = kc[:, j * kv // h, :, :top].transpose(1, 2).reshape(m, top, hd)
            s = (q[:, j, None, :] * ks).sum(-1)
        else:
            ks = kc[0, j * kv // h, :, :top].transpose(0, 1).reshape(top, hd)
            s = q[:, j] @ ks.T
        s = (s / math.sqrt(hd)).masked_fill(at[None, :] > pos[:, None], float("-inf"))
        p = _half(torch.softmax(s, -1))
        if case.get("slots"):
            heads[:, j] = (p[:, None, :] * vc[:, j * kv // h, :, :top]).sum(-1)
        else:
            heads[:, j] = p @ vc[0, j * kv // h, :, :top].T
    y = _q8_0(heads.reshape(m, qd)) @ _deq4(i["o"], d, qd).T
    return y, kc, vc


def _moe64(i, case):
    e, d, f, tk, m = case["experts"], case["dim"], case["ffn"], case["top_k"], case["m"]
    r = _rms(i["x"]) / math.sqrt(d) * i["router_scale"].double()
    logits = r @ i["router"].double().T
    ids = logits.float().sort(dim=1, descending=True, stable=True).indices[:, :tk]
    w = torch.softmax(logits.gather(1, ids), 1)
    y = torch.zeros((m, d), dtype=torch.float64, device="cuda")
    x8 = _q8_0(i["x"])
    gub, dnb = i["gu"].reshape(e, -1, 18), i["down"].reshape(e, -1, 18)
    for ex in ids.unique().tolist():
        t, s = (ids == ex).nonzero(as_tuple=True)
        gu = x8[t] @ _deq4(gub[ex], 2 * f, d).T
        g, u = _half(gu[:, :f]), gu[:, f:]  # the GELU table's input and output are fp16
        a = _half(0.5 * g * (1 + torch.tanh(0.79788456080286535588 * g * (1 + 0.044715 * g * g))))
        a = torch.where(gu[:, :f] <= -10, 0.0, torch.where(gu[:, :f] >= 10, gu[:, :f], a))
        part = _q8_0(a * u) @ _deq4(dnb[ex], d, f).T
        y.index_add_(0, t, part * (w[t, s] * i["down_scale"].double()[ex])[:, None])
    return {"y": y, "logits": logits, "weights": w, "ids": ids.int()}


def _model64(i, case):
    c = _model_config(case)
    one = {"dim": c.dim, "heads": c.heads, "kv_heads": c.kv_heads, "head_dim": c.head_dim}
    per = c.dim // 256
    tok = int(i["token"][0])
    x = _deq6(i["token_embd"][tok * per:(tok + 1) * per], 1, c.dim)
    cos, sin = _rope(case["context"], c.head_dim)
    pos = torch.tensor([case["prefix"]], device="cuda")
    keys, values = [], []
    for b, (kc, vc) in zip(i["blocks"], i["caches"]):
        a = {"qkv": torch.cat([b["q"], b["k"], b["v"]]), "o": b["o"], "gain": b["attn_norm"], "q_norm": b["q_norm"],
             "k_norm": b["k_norm"], "cos": cos, "sin": sin, "kc": kc, "vc": vc}
        y, k64, v64 = _attention64(a, one, x, pos)
        keys.append(k64)
        values.append(v64)
        x = x + y
        gu = torch.stack([b["gate"].reshape(c.ffn // 32, -1, 18), b["up"].reshape(c.ffn // 32, -1, 18)], 1)
        x = x + _ffn64(x, b["ffn_norm"], gu.reshape(-1, 18), b["down"], c.dim, c.ffn)
    hidden = _rms(x, i["output_norm"])
    a = _q8_k(hidden)
    parts = i["token_embd"].reshape(8, -1, 210)
    logits = torch.cat([(a @ _deq6(p, c.vocab // 8, c.dim).T)[0] for p in parts])
    return {"logits": logits, "hidden": hidden, "keys": keys, "values": values}


def exact(case, seed):
    i, k = _inputs(case, seed), case["kind"]
    if k == "linear":
        return _q8_0(i["x"]) @ _deq4(i["w"], case["rows"], case["cols"]).T
    if k == "head":
        rows, cols = case["rows"], case["cols"]
        a, per = _q8_k(i["x"]), cols // 256
        step = 16384
        return torch.cat([a @ _deq6(i["w"][r * per:min(r + step, rows) * per], min(step, rows - r), cols).T
                          for r in range(0, rows, step)], 1)
    if k == "ffn":
        x = i["x"].double() + i["add"].double() if case["m"] == 1 else i["x"]
        y = _ffn64(x, i["gain"], i["gu"], i["down"], case["dim"], case["ffn"])
        return {"y": y, "x": x} if case["m"] == 1 else {"y": y}
    if k == "attention":
        first, m = case["prefix"], case["m"]
        pos = torch.full((m,), first, device="cuda") if case["slots"] else torch.arange(first, first + m,
                                                                                       device="cuda")
        y, kc, vc = _attention64(i, case, i["x"], pos)
        return {"y": y, "keys": kc, "values": vc}
    if k == "moe":
        return _moe64(i, case)
    return _model64(i, case)
