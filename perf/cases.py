"""Performance cases of the decode and prefill path.

Each case is one call (or one small block of calls) that a program serving an
INT8 model through this framework makes, at sizes of the model shapes the
framework is built for (hidden 1024 / 4096 / 5120, head dims 64 and 128, FFN 3072
to 25600) or at generic ones:

  linear        int8_linear, from one decode token to a 4096-token prompt
  mlp           norm + gate / up + SwiGLU, then down + residual, 1-16 tokens
  attn_decode   paged decode attention of a batch, equal or different lengths
  attn_prefill  prompt attention over pages: causal, continued, or padded
  kv_write      q / k norm + RoPE of a prompt and its K/V into the pages
  head          final norm + fp16 lm_head, 1-16 tokens
  step          one decode step of a whole model (DecodeEngine), graph replay

`exact` is the same computation in fp64 torch, from the prepared inputs.
"""
import math

import torch

from helm_amd import kernels as hk
from helm_amd.kernels import attention as ka
from helm_amd.kernels import fused
from helm_amd.runtime.decode_engine import DecodeEngine, Int8Qwen3Weights, Qwen3Shape

# hidden, q heads, kv heads, head dim, FFN width of the supported model shapes
SHAPES = [(1024, 16, 8, 64, 3072), (4096, 32, 8, 128, 12288), (5120, 40, 8, 128, 17408),
          (5120, 64, 8, 128, 25600)]
EPS = 1e-6
THETA = 1e6
W_LEVEL = 30.0      # standard deviation of the int8 weights (a normal matrix, 127 at ~4.2 sigma)


def listed():
    return [
        # the smallest call: one token through one 4096 x 4096 projection
        {"name": "linear_1_token", "kind": "linear", "m": 1, "k": 4096, "n": 4096, "bias": False},
        # batched decode: eight sequences through a 17408 -> 5120 down projection
        {"name": "linear_8_tokens_down", "kind": "linear", "m": 8, "k": 17408, "n": 5120, "bias": False},
        # a short prompt (or a handful of speculated tokens per sequence), odd length
        {"name": "linear_77_tokens", "kind": "linear", "m": 77, "k": 4096, "n": 12288, "bias": False},
        # a long prompt through a gate / up projection
        {"name": "linear_2048_tokens", "kind": "linear", "m": 2048, "k": 5120, "n": 17408, "bias": False},
        # batched decode: the MLP block of a layer for twelve sequences
        {"name": "mlp_12_tokens", "kind": "mlp", "m": 12, "h": 5120, "f": 17408},
        # single-stream decode attention, long context
        {"name": "attn_decode_16k", "kind": "attn_decode", "b": 1, "hq": 32, "hkv": 8, "d": 128,
         "page": 16, "ctx": 16384, "ragged": False},
        # a serving batch: sequences of different lengths, up to 12000 tokens
        {"name": "attn_decode_batch", "kind": "attn_decode", "b": 8, "hq": 40, "hkv": 8, "d": 128,
         "page": 16, "ctx": 12000, "ragged": True},
        # a whole prompt's attention
        {"name": "attn_prefill_2048", "kind": "attn_prefill", "t": 2048, "past": 0, "hq": 40, "hkv": 8,
         "d": 128, "page": 16, "mask": False},
        # a prompt continued in a chunk of odd length over cached tokens
        {"name": "attn_prefill_chunk", "kind": "attn_prefill", "t": 390, "past": 7000, "hq": 32, "hkv": 8,
         "d": 128, "page": 16, "mask": False},
        # the q / k norm, RoPE and page write between the projection and the attention
        {"name": "kv_write_2000", "kind": "kv_write", "t": 2000, "hq": 32, "hkv": 8, "d": 128, "page": 16},
        # the fp16 lm_head of a small batch
        {"name": "head_4_tokens", "kind": "head", "m": 4, "h": 4096, "vocab": 151936},
        # a whole decode step, batch 1 at 16K context
        {"name": "step_16k", "kind": "step", "layers": 36, "h": 4096, "hq": 32, "hkv": 8, "d": 128,
         "f": 12288, "vocab": 151936, "ctx": 16384},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "mlp", "attn_decode", "attn_decode",
                       "attn_prefill", "attn_prefill", "kv_write", "head", "step"])
    h, hq, hkv, d, f = rng.choice(SHAPES)
    page = rng.choice([16, 16, 32, 64])
    if kind == "linear":
        k, n = rng.choice([(h, hq * d), (h, hkv * d), (h, (hq + 2 * hkv) * d), (hq * d, h), (h, f), (f, h)])
        if rng.random() < 0.25:                     # odd output widths
            n = max(1, n - rng.randrange(1, 200))
        m = _log_int(rng, 1, min(4096, max(1, int(1.0e12 / (2 * n * k)))))
        return {"kind": kind, "m": m, "k": k, "n": n, "bias": rng.random() < 0.25}
    if kind == "mlp":
        return {"kind": kind, "m": rng.randrange(1, 17), "h": h, "f": f - 16 * rng.randrange(0, 8)}
    if kind == "attn_decode":
        b = _log_int(rng, 1, 16)
        return {"kind": kind, "b": b, "hq": hq, "hkv": hkv, "d": d, "page": page,
                "ctx": _log_int(rng, 128, min(32768, 131072 // b)), "ragged": b > 1 and rng.random() < 0.7}
    if kind == "attn_prefill":
        mask = rng.random() < 0.3
        t = _log_int(rng, 17, 2048 if mask else 4096)
        past = 0 if mask or rng.random() < 0.5 else _log_int(rng, 64, 12000)
        return {"kind": kind, "t": t, "past": past, "hq": hq, "hkv": hkv, "d": d, "page": page, "mask": mask}
    if kind == "kv_write":
        return {"kind": kind, "t": _log_int(rng, 1, 4096), "hq": hq, "hkv": hkv, "d": d, "page": page}
    if kind == "head":
        return {"kind": kind, "m": rng.randrange(1, 17), "h": h,
                "vocab": rng.choice([32000, 151936, rng.randrange(30000, 152000)])}
    h, hq, hkv, d, f = rng.choice(SHAPES[:3])
    return {"kind": "step", "layers": rng.randrange(12, 29), "h": h, "hq": hq, "hkv": hkv, "d": d, "f": f,
            "vocab": rng.choice([32000, 151936]), "ctx": _log_int(rng, 512, 16384)}


# ── inputs ───────────────────────────────────────────────────────────────────

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, std=1.0):
    return (torch.randn(*shape, generator=g, device="cuda") * std).half()


def _int8(g, n, k):
    q = torch.empty(n, k, dtype=torch.int8, device="cuda")
    for i in range(0, n, 16384):
        w = torch.randn(min(16384, n - i), k, generator=g, device="cuda") * W_LEVEL
        q[i:i + 16384] = w.round_().clamp_(-127, 127)
    return q


def _scale(g, n):
    """Per-channel scales giving weights of about N(0, 0.02)."""
    return ((0.75 + 0.5 * torch.rand(n, generator=g, device="cuda")) * (0.02 / W_LEVEL)).half()


def _norm_w(g, n):
    return (1.0 + 0.1 * torch.randn(n, generator=g, device="cuda")).half()


def _pages(g, tokens, hkv, d, page, fill=True):
    """K/V pools holding ceil(tokens / page) pages, their view, and the pages in a
    random order."""
    n = -(-tokens // page)
    k = torch.zeros(n, hkv, page, d, dtype=torch.float16, device="cuda")
    v = ka.alloc_v((n, hkv, page, d), device="cuda", zero=True)
    if fill:
        k.normal_(generator=g)
        v.transpose(-1, -2).normal_(generator=g)
    order = torch.randperm(n, generator=g, device="cuda").to(torch.int32)
    return k, v, ka.PoolView.of_pool(k, v), order


def _lengths(case, seed):
    """Sequence lengths of a decode batch: all `ctx`, or spread over ctx / 16 .. ctx
    with the longest `ctx`."""
    b, ctx = case["b"], case["ctx"]
    if not case["ragged"]:
        return [ctx] * b
    g = torch.Generator().manual_seed(int(seed))
    u = torch.rand(b, generator=g).tolist()
    lens = [max(1, int(ctx * 16.0 ** (x - 1.0))) for x in u]
    lens[int(seed) % b] = ctx
    return lens


def _step_weights(case, g):
    sh = Qwen3Shape(hidden=case["h"], n_heads=case["hq"], n_kv_heads=case["hkv"], head_dim=case["d"],
                    ffn=case["f"], n_layers=case["layers"], vocab=case["vocab"], eps=EPS, rope_theta=THETA)
    w = Int8Qwen3Weights(sh)
    h, nq, d, f = case["h"], case["hq"] * case["d"], case["d"], case["f"]
    for _ in range(case["layers"]):
        lay = {}
        for name, n, k in (("qkv", nq + 2 * case["hkv"] * d, h), ("o", h, nq), ("gate", f, h), ("up", f, h),
                           ("down", h, f)):
            lay[name + "_q"], lay[name + "_s"] = _int8(g, n, k), _scale(g, n)
        lay["in_ln"], lay["post_ln"] = _norm_w(g, h), _norm_w(g, h)
        lay["q_norm"], lay["k_norm"] = _norm_w(g, d), _norm_w(g, d)
        w.layers.append(lay)
    w.embed = _normal(g, case["vocab"], h, std=0.02)
    w.norm = _norm_w(g, h)
    w.lm_head = _normal(g, case["vocab"], h, std=0.02)
    return w


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "linear":
        n, k = case["n"], case["k"]
        s["x"] = _normal(g, case["m"], k)
        s["q"], s["s"] = _int8(g, n, k), _scale(g, n)
        s["b"] = _normal(g, n, std=0.1) if case["bias"] else None
    elif kind == "mlp":
        h, f = case["h"], case["f"]
        s["x"] = _normal(g, case["m"], h)
        s["norm"] = _norm_w(g, h)
        for name, n, k in (("gate", f, h), ("up", f, h), ("down", h, f)):
            s[name + "_q"], s[name + "_s"] = _int8(g, n, k), _scale(g, n)
    elif kind == "attn_decode":
        lens = _lengths(case, seed)
        page, hkv, d = case["page"], case["hkv"], case["d"]
        counts = [-(-n // page) for n in lens]
        s["k"], s["v"], s["pool"], order = _pages(g, sum(counts) * page, hkv, d, page)
        table = torch.full((len(lens), max(counts)), -1, dtype=torch.int32, device="cuda")
        at = 0
        for i, c in enumerate(counts):
            table[i, :c] = order[at:at + c]
            at += c
        s["table"], s["lens"] = table, torch.tensor(lens, dtype=torch.int32, device="cuda")
        s["host_lens"] = lens
        s["q"] = _normal(g, len(lens), case["hq"], d)
        s["ws"] = ka.AttnWorkspace(s["q"].device)
    elif kind == "attn_prefill":
        s["k"], s["v"], s["pool"], s["table"] = _pages(g, case["past"] + case["t"], case["hkv"], case["d"],
                                                       case["page"])
        s["q"] = _normal(g, case["t"], case["hq"], case["d"])
        s["mask"] = None
        if case["mask"]:      # the causal mask of a left-padded prompt
            t = case["t"]
            i = torch.arange(t, device="cuda")
            pad = 1 + int(seed) % max(1, t // 3)
            s["mask"] = ((i[None, :] <= i[:, None]) & (i[None, :] >= pad))[None]
    elif kind == "kv_write":
        t, d = case["t"], case["d"]
        s["qkv"] = _normal(g, t, (case["hq"] + 2 * case["hkv"]) * d)
        s["q_norm"], s["k_norm"] = _norm_w(g, d), _norm_w(g, d)
        s["k"], s["v"], s["pool"], order = _pages(g, t, case["hkv"], d, case["page"], fill=False)
        s["pos"] = torch.arange(t, dtype=torch.int32, device="cuda")
        s["slots"] = order.repeat_interleave(case["page"])[:t].contiguous()
        s["offs"] = s["pos"].remainder(case["page"])
        s["inv_freq"] = fused.rope_inv_freq(d, THETA, torch.device("cuda"))
        s["q_out"] = torch.zeros(t, case["hq"], d, dtype=torch.float16, device="cuda")
    elif kind == "head":
        s["x"] = _normal(g, case["m"], case["h"])
        s["norm"] = _norm_w(g, case["h"])
        s["w"] = _normal(g, case["vocab"], case["h"], std=0.02)
    else:
        w = _step_weights(case, g)
        eng = DecodeEngine(w, max_context=case["ctx"] + 12288, page_size=16, device="cuda")
        eng.fill_synthetic_context(case["ctx"], seed=int(seed))
        s["engine"] = eng
        s["token"] = torch.randint(case["vocab"], (1,), generator=g, device="cuda")
    return s


# ── one pass ─────────────────────────────────────────────────────────────────

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear":
        return hk.int8_linear(s["x"], s["q"], s["s"], s["b"])
    if kind == "mlp":
        act = fused.int8_gemv_swiglu(s["x"], s["gate_q"], s["gate_s"], s["up_q"], s["up_s"],
                                     norm_weight=s["norm"], eps=EPS)
        return act, fused.int8_gemv_fused(act, s["down_q"], s["down_s"], residual=s["x"])
    if kind == "attn_decode":
        return ka.paged_decode_attention(s["q"], s["pool"], s["table"], s["lens"], case["page"],
                                         workspace=s["ws"])
    if kind == "attn_prefill":
        return ka.prefill_attention(s["q"], s["pool"], s["table"], case["page"], q_start=case["past"],
                                    mask=s["mask"])
    if kind == "kv_write":
        fused.qk_norm_rope_append(s["qkv"], s["q_norm"], s["k_norm"], EPS, s["pos"], s["inv_freq"],
                                  s["q_out"], s["pool"], s["slots"], s["offs"], case["hq"], case["hkv"],
                                  case["d"], case["page"])
        return {"q": s["q_out"], "k": s["k"], "v": s["v"]}
    if kind == "head":
        return fused.fp16_gemv_rmsnorm(s["x"], s["norm"], EPS, s["w"])
    eng = s["engine"]
    eng.tok.copy_(s["token"])           # a given token (scoring), not the last greedy one
    eng.decode_step()
    return eng.step_logits()


# ── what a pass cannot do without ────────────────────────────────────────────

def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": n * k + 2 * n * (2 if case["bias"] else 1) + 2 * m * (k + n), "flops": 2 * m * n * k}
    if kind == "mlp":
        m, h, f = case["m"], case["h"], case["f"]
        return {"bytes": 3 * h * f + 2 * (2 * f + 2 * h) + 2 * m * (2 * h + 2 * f), "flops": 6 * m * h * f}
    if kind == "attn_decode":
        tokens = sum(_lengths(case, 0)) if not case["ragged"] else case["ctx"] * (1 + (case["b"] - 1) * 0.338)
        return {"bytes": tokens * case["hkv"] * case["d"] * 4 + case["b"] * case["hq"] * case["d"] * 4,
                "flops": 4 * tokens * case["hq"] * case["d"]}
    if kind == "attn_prefill":
        t, past = case["t"], case["past"]
        pairs = t * past + t * (t + 1) // 2
        if case["mask"]:      # a sixth of the prompt is padding, on average
            pairs = pairs * 25 // 36
        return {"bytes": 4 * (past + t) * case["hkv"] * case["d"] + 4 * t * case["hq"] * case["d"],
                "flops": 4 * pairs * case["hq"] * case["d"]}
    if kind == "kv_write":
        return {"bytes": 4 * case["t"] * (case["hq"] + 2 * case["hkv"]) * case["d"], "flops": 0}
    if kind == "head":
        m, h, v = case["m"], case["h"], case["vocab"]
        return {"bytes": 2 * v * h + 2 * h + 2 * m * (h + v), "flops": 2 * m * h * v}
    h, hq, hkv, d, f = (case[x] for x in ("h", "hq", "hkv", "d", "f"))
    per = (hq + 2 * hkv) * d * h + hq * d * h + 3 * h * f
    kv = case["ctx"] * hkv * d * 4
    return {"bytes": case["layers"] * (per + kv) + 2 * case["vocab"] * (h + 1),
            "flops": case["layers"] * (2 * per + 4 * case["ctx"] * hq * d) + 2 * case["vocab"] * h}


def tolerance(case):
    """About four times the error of the fp16 roundings each path ends in (a result
    rounded once to fp16 is 2e-4 off in the 2-norm, at most 2^-11 of its value)."""
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 1e-3, "max": 4e-3}
    if kind == "attn_decode":
        return {"rel": 1e-3, "max": 8e-3}
    if kind == "mlp":         # roundings of the normalised x, gate, up, SiLU and the product
        return {"rel": 2.6e-3, "max": 2e-2}
    if kind == "step":        # a rounding in one layer goes through all that follow
        return {"rel": 2e-2, "max": 2e-1}
    # fp16 intermediates: the normalised x, the probabilities of a prompt's attention,
    # the factors of RoPE
    return {"rel": 2e-3, "max": 2e-2}


# ── the same in 64 bits ──────────────────────────────────────────────────────

def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _mm(x, q, s):
    """x @ (q * s)^T in fp64, q in row blocks."""
    out = torch.empty(x.shape[0], q.shape[0], dtype=torch.float64, device=x.device)
    for i in range(0, q.shape[0], 16384):
        w = q[i:i + 16384].double()
        if s is not None:
            w *= s[i:i + 16384].double()[:, None]
        out[:, i:i + 16384] = torch.mm(x, w.t().contiguous())
    return out


def _rope(x, pos, d):
    """rotate_half RoPE of x [..., T, heads, d] at positions pos [T]."""
    inv = 1.0 / (THETA ** (torch.arange(0, d, 2, device=x.device, dtype=torch.float64) / d))
    ang = pos.double()[:, None] * inv[None]
    c = torch.cat([ang.cos(), ang.cos()], -1)[:, None]
    s = torch.cat([ang.sin(), ang.sin()], -1)[:, None]
    rot = torch.cat([-x[..., d // 2:], x[..., :d // 2]], -1)
    return x * c + rot * s


def _gather(pool, table, n):
    """Token rows [n, Hkv, D] of the pages `table` of a [slots, Hkv, P, D] pool."""
    p = pool.index_select(0, table.long())
    return p.transpose(1, 2).reshape(-1, pool.shape[1], pool.shape[3])[:n].double()


def _attend(q, k, v, visible=None):
    """softmax(q k^T / sqrt(d)) v; q [T, Hq, d], k / v [S, Hkv, d], visible [T, S]."""
    t, hq, d = q.shape
    grp = hq // k.shape[1]
    out = torch.empty(t, hq, d, dtype=torch.float64, device=q.device)
    for h in range(hq):
        sc = torch.mm(q[:, h].contiguous(), k[:, h // grp].t().contiguous()) / math.sqrt(d)
        if visible is not None:
            sc = sc.masked_fill(~visible, float("-inf"))
        p = torch.softmax(sc, -1).nan_to_num(0.0)       # a row that sees nothing gives zeros
        out[:, h] = torch.mm(p, v[:, h // grp].contiguous())
    return out


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "linear":
        y = _mm(s["x"].double(), s["q"], s["s"])
        return y if s["b"] is None else y + s["b"].double()
    if kind == "mlp":
        x = _rms(s["x"].double(), s["norm"])
        act = torch.nn.functional.silu(_mm(x, s["gate_q"], s["gate_s"])) * _mm(x, s["up_q"], s["up_s"])
        return act, s["x"].double() + _mm(act, s["down_q"], s["down_s"])
    if kind == "attn_decode":
        rows = []
        for i, n in enumerate(s["host_lens"]):
            table = s["table"][i, :-(-n // case["page"])]
            rows.append(_attend(s["q"][i:i + 1].double(), _gather(s["k"], table, n), _gather(s["v"], table, n))[0])
        return torch.stack(rows)
    if kind == "attn_prefill":
        t, past = case["t"], case["past"]
        k, v = (_gather(s[x], s["table"], past + t) for x in ("k", "v"))
        if case["mask"]:
            visible = s["mask"][0]
        else:
            visible = (torch.arange(past + t, device="cuda")[None, :]
                       <= torch.arange(past, past + t, device="cuda")[:, None])
        return _attend(s["q"].double(), k, v, visible)
    if kind == "kv_write":
        t, d, hq, hkv, page = (case[x] for x in ("t", "d", "hq", "hkv", "page"))
        x = s["qkv"].double().view(t, hq + 2 * hkv, d)
        q = _rope(_rms(x[:, :hq], s["q_norm"]), s["pos"], d)
        k = _rope(_rms(x[:, hq:hq + hkv], s["k_norm"]), s["pos"], d)
        ko, vo = s["k"].double(), s["v"].double().contiguous()
        ko[s["slots"].long(), :, s["offs"].long()] = k
        vo[s["slots"].long(), :, s["offs"].long()] = x[:, hq + hkv:]
        return {"q": q, "k": ko, "v": vo}
    if kind == "head":
        return _mm(_rms(s["x"].double(), s["norm"]), s["w"], None)
    eng = s["engine"]
    hq, hkv, d, n = case["hq"], case["hkv"], case["d"], case["ctx"]
    pos = torch.tensor([n], device="cuda")
    h = eng.w.embed[s["token"]].double()
    for li, lay in enumerate(eng.w.layers):
        x = _mm(_rms(h, lay["in_ln"]), lay["qkv_q"], lay["qkv_s"]).view(1, hq + 2 * hkv, d)
        q = _rope(_rms(x[:, :hq], lay["q_norm"]), pos, d)
        kn = _rope(_rms(x[:, hq:hq + hkv], lay["k_norm"]), pos, d)
        slots = torch.tensor([p.slot for p in eng.kvcm.layers[li].pages], device="cuda")
        k = torch.cat([_gather(eng.pool.k, slots, n), kn])
        v = torch.cat([_gather(eng.pool.v, slots, n), x[:, hq + hkv:]])
        h = h + _mm(_attend(q, k, v).view(1, hq * d), lay["o_q"], lay["o_s"])
        x = _rms(h, lay["post_ln"])
        act = torch.nn.functional.silu(_mm(x, lay["gate_q"], lay["gate_s"])) * _mm(x, lay["up_q"], lay["up_s"])
        h = h + _mm(act, lay["down_q"], lay["down_s"])
    return _mm(_rms(h, eng.w.norm), eng.w.lm_head, None)[0]
