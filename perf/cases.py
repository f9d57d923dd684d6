"""The timed work of this engine: what its callers have it do, through its
public entry points, with sizes of the Qwen2.5 presets the library ships.

Kinds of case:
  gemv     one weight-only-quantized projection (cq_gemv)
  layer    one decoder layer for one token through the op-level entry points
           over the head-major cache, the way a caller of the launch_* family
           chains them: embedding, norm + QKV + RoPE, cache store, attention,
           O-projection, MLP
  attn     decode attention of one layer over the engine's tiled cache, fp16,
           int8 or E4M3
  head     lm_head, repetition penalty and argmax of one token
  decode   one step of the chat loop (State.forward and its logits)
  prefill  a prompt or a chat turn (State.prefill and its logits), alone or
           on top of a cache that earlier turns have filled; `keep`: the
           caller also takes the last layer's K and V, to keep the prompt

Model-level cases but the two `decode` ones listed run a stack of a few
layers of the preset, so that an output's rounding is that of those layers
and not of a whole network.
"""
import math

import numpy as np
import torch

import cuqwen_amd as cq

GROUP = 128
KV = {"fp16": cq.KV_FP16, "int8": cq.KV_INT8, "fp8": cq.KV_FP8}
QUANT = cq.QUANT_NAMES
DEV = "cuda"
EPS = float(np.float16(1e-6))      # the norms add half(eps)
PENALTY = float(np.float16(1.1))   # the penalty is applied as half(1.1)


def listed():
    return [
        # the smallest call: the 0.5B model's down projection, one token
        dict(name="gemv-0.5B-int8", kind="gemv", quant="int8", rows=896, cols=4864),
        # an op-level caller's layer, middle of an 8K conversation
        dict(name="layer-7B-int4-8k", kind="layer", model="7B", quant="int4", ctx=8191),
        # decode attention at the longest context, and at a ragged medium one with the E4M3 cache
        dict(name="attn-7B-32k", kind="attn", model="7B", kv="fp16", ctx=32768),
        dict(name="attn-14B-fp8-3k", kind="attn", model="14B", kv="fp8", ctx=3001),
        # the tied fp16 head of the small model, 500 generated ids
        dict(name="head-0.5B", kind="head", model="0.5B", quant="int8", history=500),
        # chat steps: the small model (launch bound), the 7B model at the end of its context
        dict(name="decode-0.5B-int8-1k", kind="decode", model="0.5B", quant="int8", kv="fp16", layers=24, pos=1151,
             history=120),
        dict(name="decode-7B-int4-32k", kind="decode", model="7B", quant="int4", kv="fp16", layers=28, pos=32700,
             history=333),
        # a short user turn on top of an earlier conversation
        dict(name="turn-7B-int4-27", kind="prefill", model="7B", quant="int4", kv="fp16", layers=4, tokens=27, pos=1500,
             keep=False),
        # a prompt of ordinary length
        dict(name="prompt-7B-int4-1k", kind="prefill", model="7B", quant="int4", kv="fp16", layers=4, tokens=1024, pos=0,
             keep=False),
        # the last full pass of a 32K document
        dict(name="long-7B-int4-2k-at-30k", kind="prefill", model="7B", quant="int4", kv="fp16", layers=3, tokens=2048,
             pos=30720, keep=False),
        # a ragged document chunk over a quantized cache
        dict(name="chunk-1.5B-int8-kv8-777", kind="prefill", model="1.5B", quant="int8", kv="int8", layers=6, tokens=777,
             pos=3000, keep=False),
        # unquantized weights, a system prompt whose K and V the caller keeps
        dict(name="prompt-0.5B-fp16-300", kind="prefill", model="0.5B", quant="fp16", kv="fp16", layers=8, tokens=300,
             pos=0, keep=True),
    ]


MODELS = ("0.5B", "1.5B", "3B", "7B", "14B")


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["gemv", "layer", "attn", "attn", "head", "decode", "decode", "prefill", "prefill", "prefill",
                       "prefill", "prefill"])
    model = rng.choice(MODELS)
    quant = rng.choice(["fp16", "int8", "int4", "int4"])
    kv = rng.choice(["fp16", "fp16", "int8", "fp8"])
    if kind == "gemv":
        cols = 128 * _log_int(rng, 4, 148)
        return dict(kind=kind, quant=quant, rows=_log_int(rng, 64, 20000), cols=cols)
    if kind == "layer":
        return dict(kind=kind, model=model, quant=quant, ctx=_log_int(rng, 1, 32768))
    if kind == "attn":
        return dict(kind=kind, model=model, kv=kv, ctx=_log_int(rng, 1, 32768))
    if kind == "head":
        return dict(kind=kind, model=model, quant=quant, history=_log_int(rng, 1, 4000))
    if kind == "decode":
        return dict(kind=kind, model=model, quant=quant, kv=kv, layers=rng.randint(2, 6), pos=_log_int(rng, 1, 32767),
                    history=_log_int(rng, 1, 1000))
    c = cq.preset(model, quant)
    tokens = _log_int(rng, 2, 2048)
    keep = tokens <= 500 and rng.random() < 0.3
    layers = 2 if model == "14B" else rng.randint(2, 3) if tokens > 512 else rng.randint(2, 6)
    pos = 0 if keep or rng.random() < 0.3 else _log_int(rng, 1, 32768 - tokens)
    # no more attention than the longest listed prompt (half of it over a quantized cache)
    most = (3.5e11 if kv == "fp16" else 1.7e11) / (c.n_heads * c.head_dim * layers * tokens)
    return dict(kind=kind, model=model, quant=quant, kv=kv, layers=layers, tokens=tokens,
                pos=max(0, min(pos, int(most) - tokens // 2)), keep=keep)


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _randn(g, *shape, std=1.0, mean=0.0):
    return (torch.randn(*shape, generator=g, device=DEV) * std + mean).half()


def _quantize(w, quant):
    """Group-128 symmetric quantization of [rows][cols] fp16 into the
    exporter's bytes and fp16 scales."""
    if quant == "fp16":
        return w, None
    rows, cols = w.shape
    qmax = 7.0 if quant == "int4" else 127.0
    v = w.float().view(rows, cols // GROUP, GROUP)
    s = v.abs().amax(-1, keepdim=True) / qmax
    q = torch.round(v / torch.where(s > 0, s, torch.ones_like(s))).clamp(-qmax, qmax).to(torch.int8).view(rows, cols)
    if quant == "int4":
        n = q.view(torch.uint8) & 15
        q = n[:, 0::2] | (n[:, 1::2] << 4)
    return q.contiguous(), s.half().view(rows, cols // GROUP).contiguous()


def _dequant(w, s, quant):
    """The matrix the bytes and scales stand for, in 64 bits."""
    if quant == "fp16":
        return w.double()
    if quant == "int4":
        b = w.view(torch.uint8)
        n = torch.stack([b & 15, b >> 4], -1).view(b.shape[0], -1).to(torch.int8)
        q = (n ^ 8) - 8
    else:
        q = w.view(torch.int8)
    return (q.double().view(q.shape[0], -1, GROUP) * s.double().unsqueeze(-1)).view(q.shape[0], -1)


def _tile_k(k):   # [n_kv][T][hd], T a multiple of 32 -> the tiled order of cq_kv_k_offset
    n, t, hd = k.shape
    return k.view(n, t // 16, 16, hd // 32, 4, 8).permute(0, 1, 3, 4, 2, 5).contiguous()


def _tile_v(v):   # -> the order of cq_kv_v_offset
    n, t, hd = v.shape
    return v.view(n, t // 32, 2, 4, 4, hd // 16, 16).permute(0, 1, 5, 3, 6, 2, 4).contiguous()


def _pairs(x, hd):   # fp16 tiled order -> the byte caches' (operand pieces of instruction pairs side by side)
    n = x.shape[0]
    return x.reshape(n, -1, 2, 64, 8).permute(0, 1, 3, 2, 4).contiguous()


def _codes(x, kv):
    """Rows of [..., hd] fp16 as cache codes and their fp32 scales."""
    top = 127.0 if kv == "int8" else 448.0
    s = x.float().abs().amax(-1) / top
    v = x.float() / torch.where(s > 0, s, torch.ones_like(s)).unsqueeze(-1)
    q = torch.round(v).clamp(-top, top).to(torch.int8) if kv == "int8" else v.to(torch.float8_e4m3fn).view(torch.int8)
    return q, s


def _value(q, s, kv):
    return (q if kv == "int8" else q.view(torch.float8_e4m3fn)).double() * s.double().unsqueeze(-1)


class _Model:
    """A weight set and a state of it; given back with the object."""

    def __init__(self, case, seed):
        self.cfg = cq.preset(case["model"], case["quant"]).replace(n_layers=case["layers"])
        self.w = cq.synth_weights(self.cfg, int(seed))
        self.st = cq.State(self.cfg, self.w, kv_dtype=KV[case["kv"]])
        if case["pos"]:
            self.st.fill_kv(case["pos"], int(seed) + 1)

    def __del__(self):
        if getattr(self, "st", None) is not None:
            self.st.free()
        if getattr(self, "w", None) is not None:
            self.w.free()


def _prompt(case, seed):
    n = case["tokens"] if case["kind"] == "prefill" else case["history"] + 1
    return np.random.default_rng(int(seed) + 2).integers(0, cq.preset(case["model"], case["quant"]).vocab_size, n).tolist()


def _attn_inputs(case, seed):
    c, g = cq.preset(case["model"], "int4"), _gen(seed)
    t, n, hd = case["ctx"], c.n_kv_heads, c.head_dim
    ms = (t + 31) // 32 * 32
    d = {"q": _randn(g, c.n_heads, hd), "k": _randn(g, n, ms, hd), "v": _randn(g, n, ms, hd)}
    return c, ms, d


def _layer_inputs(case, seed):
    c, g = cq.preset(case["model"], case["quant"]), _gen(seed)
    qd, kvd = c.n_heads * c.head_dim, c.n_kv_heads * c.head_dim
    d = {"embed": _randn(g, 4096, c.dim, std=0.02), "token": 17 + seed % 4000,
         "norm1": _randn(g, c.dim, std=0.02, mean=1.0), "norm2": _randn(g, c.dim, std=0.02, mean=1.0)}
    for name, rows in (("bq", qd), ("bk", kvd), ("bv", kvd)):
        d[name] = _randn(g, rows, std=0.02)
    for name, rows, cols in (("q", qd, c.dim), ("k", kvd, c.dim), ("v", kvd, c.dim), ("o", c.dim, qd),
                             ("g", c.intermediate_size, c.dim), ("u", c.intermediate_size, c.dim),
                             ("d", c.dim, c.intermediate_size)):
        d["W" + name], d["S" + name] = _quantize(_randn(g, rows, cols, std=0.02), case["quant"])
    ms = (case["ctx"] + 31) // 32 * 32
    d["kc"], d["vc"] = _randn(g, c.n_kv_heads, ms, c.head_dim), _randn(g, c.n_kv_heads, ms, c.head_dim)
    return c, ms, d


def _head_inputs(case, seed):
    c, g = cq.preset(case["model"], case["quant"]), _gen(seed)
    w = _randn(g, c.vocab_size, c.dim, std=0.02)
    # a hidden state that points at one row, as a model's does at the token it is sure of
    x = w[int(seed) % c.vocab_size].float() * 40 + torch.randn(c.dim, generator=g, device=DEV) * 0.2
    q, s = _quantize(w, "int8") if c.lm_head_fmt else (w, None)
    hist = torch.randint(0, c.vocab_size, (case["history"],), generator=g, device=DEV, dtype=torch.int32)
    return c, {"w": q, "s": s, "x": x.half(), "hist": hist}


def _int(v):
    return torch.tensor([v], dtype=torch.int32, device=DEV)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "gemv":
        g = _gen(seed)
        w, s = _quantize(_randn(g, case["rows"], case["cols"], std=0.02), case["quant"])
        x = _randn(g, case["cols"])
        return {"case": case, "w": w, "s": s, "x": x, "y": torch.empty(case["rows"], dtype=torch.float16, device=DEV)}
    if kind == "layer":
        c, ms, d = _layer_inputs(case, seed)
        qd, kvd, n = c.n_heads * c.head_dim, c.n_kv_heads * c.head_dim, c.n_kv_heads * 16 * 64
        half = lambda k: torch.empty(k, dtype=torch.float16, device=DEV)   # noqa: E731
        d.update(x=half(c.dim), qo=half(qd), ko=half(kvd), vo=half(kvd), ao=half(qd), inter=half(c.intermediate_size),
                 tok=_int(d["token"]), pos=_int(case["ctx"] - 1), po=torch.empty(n * c.head_dim, device=DEV),
                 pm=torch.empty(n, device=DEV), pl=torch.empty(n, device=DEV))
        return {"case": case, "c": c, "ms": ms, "d": d, "p": {k: _p(v) for k, v in d.items() if k != "token"}}
    if kind == "attn":
        c, ms, d = _attn_inputs(case, seed)
        t = case["ctx"]
        s = {"case": case, "c": c, "ms": ms, "q": d["q"], "pos": _int(t - 1), "out": torch.empty_like(d["q"]),
             "ws": torch.empty(cq.lib.cq_attention_workspace_bytes(c.n_heads, c.n_kv_heads, c.head_dim),
                               dtype=torch.uint8, device=DEV)}
        if case["kv"] == "fp16":
            s["k"], s["v"] = _tile_k(d["k"]), _tile_v(d["v"])
        else:
            for n, tile in (("k", _tile_k), ("v", _tile_v)):
                q, sc = _codes(d[n], case["kv"])
                s[n], s[n + "s"], s[n + "n"] = _pairs(tile(q), c.head_dim), sc, d[n][:, t - 1].contiguous()
        return s
    if kind == "head":
        c, d = _head_inputs(case, seed)
        d.update(logits=torch.empty(c.vocab_size, dtype=torch.float16, device=DEV), n=_int(case["history"]), tok=_int(0),
                 pw=torch.zeros(cq.lib.cq_penalty_workspace_bytes(c.vocab_size), dtype=torch.uint8, device=DEV),
                 aw=torch.zeros(cq.lib.cq_argmax_workspace_bytes(c.vocab_size), dtype=torch.uint8, device=DEV))
        return {"case": case, "c": c, "d": d}
    return {"case": case, "m": _Model(case, seed), "tokens": _prompt(case, seed)}


# --------------------------------------------------------------------- run
def _p(t):
    return None if t is None else t.data_ptr()


def run(state):
    case = state["case"]
    kind, L, ck = case["kind"], cq.lib, cq.check
    if kind == "gemv":
        ck(L.cq_gemv(QUANT[case["quant"]], GROUP if state["s"] is not None else 0, _p(state["w"]), _p(state["s"]),
                     _p(state["x"]), _p(state["y"]), case["rows"], case["cols"], None))
        return state["y"]
    if kind == "layer":
        c, ms, qt, d = state["c"], state["ms"], QUANT[case["quant"]], state["p"]
        ck(L.cq_embedding_lookup(d["embed"], d["tok"], d["x"], c.dim, None))
        ck(L.cq_fused_attn_block(qt, d["x"], d["norm1"], d["Wq"], d["Wk"], d["Wv"], d["Sq"], d["Sk"], d["Sv"], d["bq"],
                                 d["bk"], d["bv"], d["qo"], d["ko"], d["vo"], c.dim, c.n_heads, c.n_kv_heads, c.head_dim,
                                 d["pos"], c.rope_theta, c.norm_eps, None))
        ck(L.cq_kv_cache_store_hm(d["ko"], d["vo"], d["kc"], d["vc"], d["pos"], c.n_kv_heads, ms, c.head_dim, None))
        ck(L.cq_gqa_attention_decode_hm(d["qo"], d["kc"], d["vc"], d["ao"], d["pos"], c.n_heads, c.n_kv_heads,
                                        c.head_dim, ms, d["po"], d["pm"], d["pl"], None))
        ck(L.cq_gemv_add(qt, d["Wo"], d["So"], d["ao"], d["x"], c.dim, c.n_heads * c.head_dim, None))
        ck(L.cq_fused_mlp_stage1(qt, d["x"], d["norm2"], d["Wg"], d["Wu"], d["Sg"], d["Su"], d["inter"], c.dim,
                                 c.intermediate_size, c.norm_eps, None))
        ck(L.cq_fused_mlp_stage2(qt, d["x"], d["Wd"], d["Sd"], d["inter"], c.dim, c.intermediate_size, None))
        s = state["d"]
        return {"x": s["x"], "k": s["ko"], "v": s["vo"], "attn": s["ao"], "inter": s["inter"]}
    if kind == "attn":
        c, s = state["c"], state
        if case["kv"] == "fp16":
            ck(L.cq_gqa_attention_decode(_p(s["q"]), _p(s["k"]), _p(s["v"]), _p(s["out"]), _p(s["pos"]), c.n_heads,
                                         c.n_kv_heads, c.head_dim, s["ms"], _p(s["ws"]), None))
        else:
            f = L.cq_gqa_attention_decode_kv8 if case["kv"] == "int8" else L.cq_gqa_attention_decode_fp8
            ck(f(_p(s["q"]), _p(s["kn"]), _p(s["vn"]), _p(s["k"]), _p(s["v"]), _p(s["ks"]), _p(s["vs"]), _p(s["out"]),
                 _p(s["pos"]), c.n_heads, c.n_kv_heads, c.head_dim, s["ms"], _p(s["ws"]), None))
        return s["out"]
    if kind == "head":
        c, d = state["c"], state["d"]
        ck(L.cq_compute_logits(c.lm_head_fmt, _p(d["x"]), _p(d["w"]), _p(d["s"]), _p(d["logits"]), c.vocab_size, c.dim,
                               None))
        ck(L.cq_apply_repetition_penalty(_p(d["logits"]), _p(d["hist"]), _p(d["n"]), c.vocab_size, c.repetition_penalty,
                                         _p(d["pw"]), None))
        ck(L.cq_argmax(_p(d["logits"]), _p(d["tok"]), c.vocab_size, _p(d["aw"]), None))
        return {"logits": d["logits"], "token": d["tok"]}
    # the sampled id of a random network hangs on near ties of its logits: the logits are what is returned
    m = state["m"]
    if kind == "decode":
        m.st.forward(state["tokens"][0], case["pos"], state["tokens"][1:])
        return {"logits": m.st.logits()}
    m.st.prefill(state["tokens"], case["pos"])
    out = {"logits": m.st.logits()}
    if case["keep"]:
        out["kv"] = [m.st.kv_read(case["layers"] - 1, h, kind, case["tokens"])
                     for h in range(m.cfg.n_kv_heads) for kind in (0, 1)]
    return out


# -------------------------------------------------------------------- work
def _wbytes(quant, rows, cols):
    return rows * cols * {"fp16": 2, "int8": 1, "int4": 0.5}[quant] + (0 if quant == "fp16" else 2 * rows * cols / GROUP)


def _layer_shapes(c):
    qd, kvd = c.n_heads * c.head_dim, c.n_kv_heads * c.head_dim
    return (qd + 2 * kvd, c.dim), [(c.dim, qd), (2 * c.intermediate_size, c.dim), (c.dim, c.intermediate_size)]


def _row_bytes(c, kv):   # K and V of one position of one layer
    return 2 * c.n_kv_heads * (2 * c.head_dim if kv == "fp16" else c.head_dim + 4)


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        r, k = case["rows"], case["cols"]
        return {"bytes": _wbytes(case["quant"], r, k) + 2 * (r + k), "flops": 2 * r * k}
    c = cq.preset(case["model"], case.get("quant", "int4"))
    qd, V = c.n_heads * c.head_dim, c.vocab_size
    if kind == "attn":
        return {"bytes": case["ctx"] * _row_bytes(c, case["kv"]) + 4 * qd, "flops": 4 * qd * case["ctx"]}
    head = _wbytes("int8" if c.lm_head_fmt else "fp16", V, c.dim) + 2 * (V + c.dim)
    if kind == "head":
        return {"bytes": head + 4 * case["history"], "flops": 2 * V * c.dim}
    qkv, rest = _layer_shapes(c)
    mats = [qkv] + rest
    wl = sum(_wbytes(case["quant"], r, k) for r, k in mats)
    if kind == "layer":
        return {"bytes": wl + case["ctx"] * _row_bytes(c, "fp16") + 8 * c.dim,
                "flops": sum(2 * r * k for r, k in mats) + 4 * qd * case["ctx"]}
    n, pos, layers = case.get("tokens", 1), case["pos"], case["layers"]
    keys = n * pos + n * (n + 1) // 2   # (token, key) pairs of a layer
    b = layers * (wl + (pos + n) * _row_bytes(c, case["kv"])) + head + 2 * n * c.dim
    # the last layer's O-projection and MLP, and the head, are for the last token only
    f = layers * (2 * n * qkv[0] * qkv[1] + 4 * qd * keys) + 2 * V * c.dim
    f += sum(2 * r * k for r, k in rest) * ((layers - 1) * n + 1)
    return {"bytes": b, "flops": f}


# --------------------------------------------------------------- tolerance
def tolerance(case):
    """fp16 inputs and results with 32-bit sums: about four times the distance
    from the 64-bit results, measured over the listed and drawn cases."""
    return {
        "gemv": {"rel": 1e-3, "max": 1e-2},        # one fp16 rounding of a 32-bit sum: 2.0e-4
        "attn": {"rel": 2e-3, "max": 2e-2},        # scores and P in fp16: 5.4e-4
        "head": {"rel": 1e-3, "max": 1e-2},        # 2.1e-4
        "layer": {"rel": 6e-3, "max": 6e-2},       # norm inputs, attention and SwiGLU rounded on the way: 1.6e-3
        "decode": {"rel": 2e-2, "max": 2e-1},      # the same through the whole network: 5.5e-3
        "prefill": {"rel": 1.2e-2, "max": 1.2e-1},  # through a few layers: 3.2e-3
    }[case["kind"]]


# ------------------------------------------------------------------- exact
def _rope(x, pos, theta):   # [n][heads][hd], positions [n]
    hd = x.shape[-1]
    f = theta ** (-torch.arange(hd // 2, dtype=torch.float64, device=DEV) * 2 / hd)
    a = pos.double()[:, None] * f
    s, c = a.sin()[:, None], a.cos()[:, None]
    x0, x1 = x[..., :hd // 2], x[..., hd // 2:]
    return torch.cat([x0 * c - x1 * s, x1 * c + x0 * s], -1)


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _attend(q, k, v, first):
    """Causal attention of q [n][H][hd], whose row i sees keys 0 .. first + i,
    over k, v [n_kv][T][hd]."""
    n, H, hd = q.shape
    out = torch.empty_like(q)
    g = H // k.shape[0]
    block = max(1, (1 << 28) // k.shape[1])
    t = torch.arange(k.shape[1], device=DEV)
    for h in range(H):
        kt = k[h // g].t().contiguous()
        for a in range(0, n, block):
            b = min(n, a + block)
            s = q[a:b, h] @ kt / math.sqrt(hd)
            s.masked_fill_(t[None] > (first + torch.arange(a, b, device=DEV))[:, None], -math.inf)
            out[a:b, h] = torch.softmax(s, -1) @ v[h // g]
    return out


def _silu(x):
    return x / (1 + torch.exp(-x))


_M64 = (1 << 64) - 1


def _s64(v):
    v &= _M64
    return v - (1 << 64) if v >> 63 else v


def _mix(z):   # splitmix64's finaliser on int64 tensors (wrapping multiplies, logical shifts)
    lsr = lambda x, k: (x >> k) & ((1 << (64 - k)) - 1)   # noqa: E731
    z = (z ^ lsr(z, 30)) * _s64(0xBF58476D1CE4E5B9)
    z = (z ^ lsr(z, 27)) * _s64(0x94D049BB133111EB)
    return z ^ lsr(z, 31)


def _filled(seed, stream, n):
    """The first n values cq_state_fill_kv gives a row stream (cq_synth_normal)."""
    gold = 0x9E3779B97F4A7C15
    key = _mix(torch.tensor([_s64(seed + gold * (stream + 1))], dtype=torch.int64, device=DEV))
    r = _mix(key + (torch.arange(n, dtype=torch.int64, device=DEV) + 1) * _s64(gold))
    u = sum((r >> k) & 0xFFFF for k in (0, 16, 32, 48)) - 131070
    return (u.float() * float(np.float32(1.0 / 37836.51))).half()


def _tensor(w, name, layer, dtype, shape):
    """A copy of one weight tensor of the model."""
    p, nbytes = w.tensor(name, layer)
    t = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    cq.check(cq.lib.cq_memcpy_d2d(t.data_ptr(), p, nbytes))
    cq.synchronize()
    return t.view(dtype).view(*shape)


def _matrix(w, name, scale, layer, quant, rows, cols):
    wt = {"fp16": torch.float16, "int8": torch.int8, "int4": torch.uint8}[quant]
    s = None if quant == "fp16" else _tensor(w, scale, layer, torch.float16, (-1,))
    if name == "wo":   # 128-column panels [cols / 128][rows][128], scales [cols / 128][rows]
        p = cols // GROUP
        b = _tensor(w, name, layer, wt, (p, rows, -1)).permute(1, 0, 2).reshape(rows, -1).contiguous()
        return _dequant(b, None if s is None else s.view(p, rows).t().contiguous(), quant)
    b = _tensor(w, name, layer, wt, (rows, -1))
    return _dequant(b, None if s is None else s.view(rows, -1), quant)


def _exact_model(case, seed):
    cfg = cq.preset(case["model"], case["quant"]).replace(n_layers=case["layers"])
    toks = _prompt(case, seed)
    ids = toks if case["kind"] == "prefill" else toks[:1]
    n, pos, qt, kv = len(ids), case["pos"], case["quant"], case["kv"]
    H, NKV, hd, I, V = cfg.n_heads, cfg.n_kv_heads, cfg.head_dim, cfg.intermediate_size, cfg.vocab_size
    at = torch.arange(pos, pos + n, device=DEV)
    w = cq.synth_weights(cfg, int(seed))
    kept = []
    try:
        embed = _tensor(w, "embed", -1, torch.float16, (V, cfg.dim))
        x = embed[torch.tensor(ids, device=DEV)].double()
        for l in range(cfg.n_layers):
            vec = lambda name: _tensor(w, name, l, torch.float16, (-1,))   # noqa: B023, E731
            proj = lambda y, name, sc, r, k: y @ _matrix(w, name, sc, l, qt, r, k).t()   # noqa: B023, E731
            h = _norm(x, vec("in_norm"))
            q = (proj(h, "wq", "sq", H * hd, cfg.dim) + vec("bq").double()).view(n, H, hd)
            k = (proj(h, "wk", "sk", NKV * hd, cfg.dim) + vec("bk").double()).view(n, NKV, hd)
            v = (proj(h, "wv", "sv", NKV * hd, cfg.dim) + vec("bv").double()).view(n, NKV, hd)
            q, k = _rope(q, at, cfg.rope_theta), _rope(k, at, cfg.rope_theta)
            new = {0: k, 1: v}
            cache = {}
            for kind in (0, 1):
                old = [_filled(int(seed) + 1, int(cq.lib.cq_kv_stream_id(l, hh, kind)), pos * hd).view(pos, hd)
                       for hh in range(NKV)]
                old, fresh = torch.stack(old), new[kind].permute(1, 0, 2)
                if kv == "fp16":
                    old = old.double()
                else:
                    old, fresh = (_value(*_codes(r, kv), kv) for r in (old, fresh.half()))
                cache[kind] = torch.cat([old, fresh], 1).contiguous()
            if case.get("keep") and l == cfg.n_layers - 1:
                kept = [cache[kind][hh].clone() for hh in range(NKV) for kind in (0, 1)]
            a = _attend(q, cache[0], cache[1], pos).view(n, H * hd)
            del cache
            if l == cfg.n_layers - 1:
                a, x = a[-1:], x[-1:]
            x = x + proj(a, "wo", "so", cfg.dim, H * hd)
            h = _norm(x, vec("post_norm"))
            m = _silu(proj(h, "wg", "sg", I, cfg.dim)) * proj(h, "wu", "su", I, cfg.dim)
            x = x + proj(m, "wd", "sd", cfg.dim, I)
        h = _norm(x, _tensor(w, "final_norm", -1, torch.float16, (-1,)))
        head = (_matrix(w, "lm_head", "lm_head_scale", -1, "int8", V, cfg.dim) if cfg.lm_head_fmt
                else _tensor(w, "lm_head", -1, torch.float16, (V, cfg.dim)).double())
        logits = (h @ head.t()).view(-1)
    finally:
        w.free()
    if case["kind"] == "decode":
        logits = _penalize(logits, torch.tensor(toks[1:], device=DEV))
    return {"logits": logits, "kv": kept} if case.get("keep") else {"logits": logits}


def _penalize(logits, ids):
    ids = torch.unique(ids.long())
    out = logits.clone()
    l = logits[ids]
    out[ids] = torch.where(l < 0, l * PENALTY, l / PENALTY)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemv":
        s = prepare(case, seed)
        return _dequant(s["w"], s["s"], case["quant"]) @ s["x"].double()
    if kind == "attn":
        c, _, d = _attn_inputs(case, seed)
        k, v = (d[n][:, :case["ctx"]] for n in ("k", "v"))
        k, v = (k.double(), v.double()) if case["kv"] == "fp16" else (_value(*_codes(r, case["kv"]), case["kv"]) for r in (k, v))
        return _attend(d["q"].double().unsqueeze(0), k.contiguous(), v.contiguous(), case["ctx"] - 1)[0]
    if kind == "head":
        c, d = _head_inputs(case, seed)
        w = d["w"].double() if d["s"] is None else _dequant(d["w"], d["s"], "int8")
        logits = _penalize(w @ d["x"].double(), d["hist"])
        return {"logits": logits, "token": None}
    if kind == "layer":
        c, ms, d = _layer_inputs(case, seed)
        t, qt, hd = case["ctx"], case["quant"], c.head_dim
        W = lambda n: _dequant(d["W" + n], d["S" + n], qt)   # noqa: E731
        x = d["embed"][d["token"]].double()
        h = _norm(x, d["norm1"])
        at = torch.tensor([t - 1], device=DEV)
        q = _rope((W("q") @ h + d["bq"].double()).view(1, c.n_heads, hd), at, c.rope_theta)
        k = _rope((W("k") @ h + d["bk"].double()).view(1, c.n_kv_heads, hd), at, c.rope_theta)[0]
        v = (W("v") @ h + d["bv"].double()).view(c.n_kv_heads, hd)
        kc, vc = d["kc"][:, :t].double(), d["vc"][:, :t].double()
        kc[:, t - 1], vc[:, t - 1] = k, v
        a = _attend(q, kc, vc, t - 1).view(-1)
        x = x + W("o") @ a
        h = _norm(x, d["norm2"])
        m = _silu(W("g") @ h) * (W("u") @ h)
        return {"x": x + W("d") @ m, "k": k.reshape(-1), "v": v.reshape(-1), "attn": a, "inter": m}
    return _exact_model(case, seed)
