"""Workloads of the quantized linear layer and its attention, as a Llama runtime calls them.

Each case is one piece of work that a program built on ``unillm_amd`` does: a single
projection, an MLP, the projections of a batched decode step, a whole decode step
captured as a HIP graph, or a prompt's attention.  Weights are GGUF blocks made here in
plain torch from a seed (so that ``exact`` knows their values without the library), and
everything runs through ``QuantLinear`` and ``KvCache``.

Model shapes are Llama-2-7B's (hidden 4096, MLP 11008, 32 heads of 128), Mistral-7B's
(MLP 14336, 8 KV heads) and TinyLlama-1.1B's (hidden 2048, MLP 5632, 32 heads of 64 over
4 KV heads); drawn cases take sizes between and around them.
"""
from __future__ import annotations

import math

import torch

from unillm_amd import (BF16, F16, F32, Q4_0, Q4_K, Q5_0, Q5_K, Q6_K, Q8_0, KvCache,
                        QuantLinear)

QTYPES = {"q4_0": Q4_0, "q5_0": Q5_0, "q8_0": Q8_0, "q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K,
          "f32": F32, "f16": F16, "bf16": BF16}
DENSE = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
# GGUF bytes and weights of a block
BLOCK = {"q4_0": (18, 32), "q5_0": (22, 32), "q8_0": (34, 32), "q4_k": (144, 256),
         "q5_k": (176, 256), "q6_k": (210, 256), "f32": (4, 1), "f16": (2, 1), "bf16": (2, 1)}
EPS = 1e-6
THETA = 10000.0
DECODE_ROOM = 64  # positions a decode case's cache holds past its prompt


# ---- the cases --------------------------------------------------------------------------
def _linear(name, qtype, m, n, k, epi):
    return {"name": name, "kind": "linear", "qtype": qtype, "m": m, "n": n, "k": k, "epi": epi}


def listed():
    return [
        # the smallest call of a decode loop: TinyLlama's MLP up projection, one token,
        # called eagerly (launch and host latency)
        _linear("q8_0_m1_tinyllama_up", "q8_0", 1, 5632, 2048, "store"),
        # one token through two Llama-2-7B layers, the final norm and the lm_head, over
        # 1024 cached positions: the generation loop's captured step
        {"name": "decode_step_llama7b_q4_0", "kind": "decode_step", "qtype": "q4_0",
         "head_qtype": "q8_0", "hidden": 4096, "inter": 11008, "heads": 32, "kv_heads": 32,
         "hd": 128, "vocab": 32000, "layers": 2, "past": 1024},
        # the same on Mistral-7B's shape from a Q4_K_M file (Q6_K head), grouped-query
        # attention over a long context
        {"name": "decode_step_mistral7b_q4_k", "kind": "decode_step", "qtype": "q4_k",
         "head_qtype": "q6_k", "hidden": 4096, "inter": 14336, "heads": 32, "kv_heads": 8,
         "hd": 128, "vocab": 32000, "layers": 2, "past": 4000},
        # the projections of one Llama-2-7B layer for a continuous batch of 16 sequences
        {"name": "batch16_layer_llama7b_q4_0", "kind": "batch_layer", "qtype": "q4_0", "m": 16,
         "hidden": 4096, "inter": 11008, "qkv": 12288},
        # Mistral's MLP for a batch of 64 (the widest continuous batch)
        {"name": "mlp_m64_mistral7b_q4_k", "kind": "mlp", "qtype": "q4_k", "m": 64,
         "hidden": 4096, "inter": 14336},
        # a short prompt's attention output projection with its residual add
        _linear("q8_0_m100_llama7b_o", "q8_0", 100, 4096, 4096, "add"),
        # a long prompt through Mistral's gate or up projection
        _linear("q4_0_m2048_mistral7b_up", "q4_0", 2048, 14336, 4096, "store"),
        # a 512-token prompt through Llama-2-7B's MLP
        {"name": "mlp_m512_llama7b_q8_0", "kind": "mlp", "qtype": "q8_0", "m": 512,
         "hidden": 4096, "inter": 11008},
        # a 2048-token prompt's attention into an empty cache, Llama-2-7B
        {"name": "prompt_attention_m2048_llama7b", "kind": "prompt_attention", "m": 2048,
         "past": 0, "heads": 32, "kv_heads": 32, "hd": 128},
        # the next turn of a chat: 500 new tokens behind 777 cached ones, TinyLlama
        {"name": "prompt_attention_m500_tinyllama", "kind": "prompt_attention", "m": 500,
         "past": 777, "heads": 32, "kv_heads": 4, "hd": 64},
        # projections of unquantized GGUF files: one token through an F16 file's gate
        # projection, and a 512-token prompt through a BF16 file's
        _linear("f16_m1_llama7b_gate", "f16", 1, 11008, 4096, "store"),
        _linear("bf16_m512_llama7b_gate", "bf16", 512, 11008, 4096, "store"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, qtype, k_hi, n_hi):
    unit = BLOCK[qtype][1] if qtype not in DENSE else 8
    k = max(unit, _log(rng, 1024, k_hi) // unit * unit)
    return k, _log(rng, 512, n_hi)


def draw(rng):
    kind = rng.choice(["linear"] * 4 + ["mlp", "batch_layer", "prompt_attention",
                                        "prompt_attention", "decode_step", "dense"])
    quant = rng.choice(["q4_0", "q4_0", "q8_0", "q4_k", "q4_k", "q5_0", "q5_k", "q6_k"])
    if kind == "linear":
        k, n = _shape(rng, quant, 14336, 32000)
        m = min(_log(rng, 1, 2048), 2048 * 4096 * 14336 // (n * k))
        epi = rng.choice(["store", "store", "add", "norm"])
        return {"kind": "linear", "qtype": quant, "m": m, "n": n, "k": k, "epi": epi}
    if kind == "dense":
        qtype = rng.choice(["f16", "bf16", "f32"])
        k, n = _shape(rng, qtype, 11008, 16384)
        m = min(_log(rng, 1, 512), 512 * 4096 * 11008 // (n * k))
        return {"kind": "linear", "qtype": qtype, "m": m, "n": n, "k": k,
                "epi": rng.choice(["store", "store", "add"])}
    unit = max(BLOCK[quant][1], 128)
    hidden = rng.choice([2048, 2560, 3072, 4096])
    inter = _log(rng, 4096, 14336) // unit * unit
    if kind == "mlp":
        m = min(_log(rng, 2, 512), 512 * 4096 * 11008 // (hidden * inter))
        return {"kind": "mlp", "qtype": quant, "m": m, "hidden": hidden, "inter": inter}
    if kind == "batch_layer":
        return {"kind": "batch_layer", "qtype": quant, "m": _log(rng, 2, 64), "hidden": hidden,
                "inter": inter, "qkv": hidden + 2 * rng.choice([256, 512, 1024, 2048])}
    hd = rng.choice([64, 128, 128])
    if kind == "decode_step":
        heads = hidden // hd
        kv_heads = rng.choice([h for h in (4, 8, heads) if heads % h == 0 and heads // h <= 16])
        return {"kind": "decode_step", "qtype": quant,
                "head_qtype": rng.choice(["q8_0", "q6_k"]), "hidden": hidden, "inter": inter,
                "heads": heads, "kv_heads": kv_heads, "hd": hd,
                "vocab": rng.randrange(16000, 32001), "layers": rng.choice([1, 2]),
                "past": _log(rng, 16, 4096)}
    heads = rng.choice([16, 24, 32])
    kv_heads = rng.choice([4, 8, heads])
    past = rng.choice([0, 0, _log(rng, 16, 2048)])
    m = _log(rng, 32, 2048)
    while heads * hd * m * (past + m / 2) > 32 * 128 * 2048 * 1024:
        m = m * 3 // 4
    return {"kind": "prompt_attention", "m": m, "past": past, "heads": heads,
            "kv_heads": kv_heads, "hd": hd}


# ---- GGUF blocks from a seed, and the values they stand for -----------------------------
def _gen(seed, tag):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + tag * 7919 + 17) & 0x7FFFFFFFFFFF)
    return g


def _randn(g, *shape):
    return torch.empty(*shape, device="cuda").normal_(generator=g)


def _codes(g, shape, hi, spread):
    """Whole codes 0 .. hi, normal around the middle."""
    mid = (hi + 1) / 2
    return (_randn(g, *shape) * spread + mid).round_().clamp_(0, hi).to(torch.uint8)


def _bytes(t):
    return t.contiguous().view(torch.uint8)


def _nibbles(q):
    """[.., 32] codes -> 16 bytes: low nibbles elements 0 .. 15, high nibbles 16 .. 31."""
    return q[..., :16] | (q[..., 16:] << 4)


def _pack_scales(sc, mn):
    """Eight 6-bit scales and minima of a 256-block -> GGML's 12 bytes."""
    lo = sc[..., :4] | ((sc[..., 4:] >> 4) << 6)
    mid = mn[..., :4] | ((mn[..., 4:] >> 4) << 6)
    hi = (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)
    return torch.cat([lo, mid, hi], dim=-1)


def _weight(qtype, n, k, seed, tag, values=False):
    """The GGUF bytes of an [n, k] weight of about N(0, 0.02); with values, its f64 values."""
    g = _gen(seed, tag)
    if qtype in DENSE:
        w = (_randn(g, n, k) * 0.02).to(DENSE[qtype])
        return w.double() if values else w
    nb = k // BLOCK[qtype][1]
    if qtype in ("q4_0", "q5_0", "q8_0"):
        hi, spread = {"q4_0": (15, 3.4), "q5_0": (31, 7.0), "q8_0": (255, 55.0)}[qtype]
        q = _codes(g, (n, nb, 32), hi, spread)
        d = (0.02 / spread * (1.0 + 0.1 * _randn(g, n, nb, 1))).half()
        if values:
            return (d.double() * (q.double() - (hi + 1) // 2)).view(n, k)
        if qtype == "q4_0":
            parts = [_bytes(d), _nibbles(q)]
        elif qtype == "q5_0":
            top = (q >> 4).to(torch.int64) << torch.arange(32, device="cuda")
            top = top.sum(-1, keepdim=True)
            qh = torch.cat([((top >> s) & 255).to(torch.uint8) for s in (0, 8, 16, 24)], dim=-1)
            parts = [_bytes(d), qh, _nibbles(q & 15)]
        else:
            parts = [_bytes(d), (q.to(torch.int16) - 128).to(torch.int8).view(torch.uint8)]
        return torch.cat(parts, dim=-1).contiguous().view(-1)
    if qtype in ("q4_k", "q5_k"):
        hi, spread = {"q4_k": (15, 3.4), "q5_k": (31, 7.0)}[qtype]
        q = _codes(g, (n, nb, 8, 32), hi, spread)
        sc = (40 + 8 * _randn(g, n, nb, 8)).round_().clamp_(16, 63).to(torch.uint8)
        mn = (sc.float() + _randn(g, n, nb, 8)).round_().clamp_(0, 63).to(torch.uint8)
        d = (0.02 / spread / 40 * (1.0 + 0.1 * _randn(g, n, nb, 1))).half()
        dmin = (d.float() * ((hi + 1) / 2)).half()
        if values:
            w = (d.double().unsqueeze(-1) * sc.double().unsqueeze(-1) * q.double()
                 - dmin.double().unsqueeze(-1) * mn.double().unsqueeze(-1))
            return w.view(n, k)
        low = q & 15
        qs = (low[:, :, 0::2] | (low[:, :, 1::2] << 4)).reshape(n, nb, 128)
        parts = [_bytes(d), _bytes(dmin), _pack_scales(sc, mn)]
        if qtype == "q5_k":
            shift = torch.arange(8, device="cuda", dtype=torch.int32).view(8, 1)
            parts.append((((q >> 4).to(torch.int32) << shift).sum(2)).to(torch.uint8))
        return torch.cat(parts + [qs], dim=-1).contiguous().view(-1)
    q = _codes(g, (n, nb, 2, 4, 32), 63, 13.0)  # q6_k: halves of 128, four runs of 32
    sc = (60 + 10 * _randn(g, n, nb, 16)).round_().clamp_(20, 127).to(torch.int8)
    d = (0.02 / 13 / 60 * (1.0 + 0.1 * _randn(g, n, nb, 1))).half()
    if values:
        s16 = sc.double().repeat_interleave(16, dim=-1)
        return (d.double() * s16 * (q.double().view(n, nb, 256) - 32)).view(n, k)
    low = q & 15
    ql = torch.cat([low[..., 0, :] | (low[..., 2, :] << 4), low[..., 1, :] | (low[..., 3, :] << 4)],
                   dim=-1)
    top = q >> 4
    qh = (top[..., 0, :] | (top[..., 1, :] << 2) | (top[..., 2, :] << 4) | (top[..., 3, :] << 6))
    return torch.cat([ql.reshape(n, nb, 128), qh.reshape(n, nb, 64), sc.view(torch.uint8),
                      _bytes(d)], dim=-1).contiguous().view(-1)


def _load(qtype, n, k, seed, tag):
    w = _weight(qtype, n, k, seed, tag)
    if qtype in DENSE:
        return QuantLinear.from_dense(w)
    return QuantLinear.from_device_blocks(QTYPES[qtype], n, k, w)


# ---- prepare: weights on the device, inputs, caches and (decode) the captured graph -----
_STREAM = None


def _stream():
    """The one stream a program issues its decode steps on."""
    global _STREAM
    if _STREAM is None:
        _STREAM = torch.cuda.Stream()
    return _STREAM


def _layer_shapes(case):
    """(tag, n, k) of a layer's fused QKV, o, gate + up and down projections."""
    hidden, inter = case["hidden"], case["inter"]
    if case["kind"] == "decode_step":
        q, kv = case["heads"] * case["hd"], case["kv_heads"] * case["hd"]
        qkv = q + 2 * kv
    else:
        q, qkv = hidden, case["qkv"]
    return [(0, qkv, hidden), (1, hidden, q), (2, 2 * inter, hidden), (3, hidden, inter)]


def _gamma(seed, tag, k):
    return 1.0 + 0.1 * _randn(_gen(seed, tag), k)


def _capture(state, step):
    """`step` once eagerly (workspaces grow), then captured."""
    s = _stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s, capture_error_mode="thread_local"):
            step()
    torch.cuda.synchronize()
    state["graph"] = g
    state["stream"] = s


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind, "case": case}
    if kind == "linear":
        st["w"] = _load(case["qtype"], case["n"], case["k"], seed, 0)
        st["x"] = _randn(_gen(seed, 100), case["m"], case["k"])
        if case["epi"] == "add":
            st["y"] = _randn(_gen(seed, 101), case["m"], case["n"])
        if case["epi"] == "norm":
            st["gamma"] = _gamma(seed, 102, case["k"])
    elif kind == "mlp":
        hidden, inter = case["hidden"], case["inter"]
        st["gu"] = _load(case["qtype"], 2 * inter, hidden, seed, 2)
        st["down"] = _load(case["qtype"], hidden, inter, seed, 3)
        st["x"] = _randn(_gen(seed, 100), case["m"], hidden)
        st["y"] = torch.empty_like(st["x"])
        st["gamma"] = _gamma(seed, 102, hidden)
    elif kind == "prompt_attention":
        width = (case["heads"] + 2 * case["kv_heads"]) * case["hd"]
        st["kv"] = KvCache(case["kv_heads"], case["hd"], case["past"] + case["m"], THETA)
        if case["past"]:
            st["kv"].attention(_randn(_gen(seed, 103), case["past"], width), case["heads"])
        st["x"] = _randn(_gen(seed, 100), case["m"], width)
    elif kind == "batch_layer":
        shapes = _layer_shapes(case)
        st["w"] = [_load(case["qtype"], n, k, seed, t) for t, n, k in shapes]
        m, hidden = case["m"], case["hidden"]
        st["x"] = _randn(_gen(seed, 100), m, hidden)
        st["att"] = _randn(_gen(seed, 101), m, hidden)  # the sequences' attention outputs
        st["g1"], st["g2"] = _gamma(seed, 102, hidden), _gamma(seed, 103, hidden)
        st["h"] = torch.empty_like(st["x"])
        st["qkv"] = torch.empty(m, case["qkv"], device="cuda")
        st["act"] = torch.empty(m, case["inter"], device="cuda")
        s = _stream()

        def layer():
            qkv, o, gu, down = st["w"]
            st["h"].copy_(st["x"])
            qkv.forward_norm(st["h"], st["g1"], eps=EPS, out=st["qkv"], stream=s)
            o.forward_add(st["att"], st["h"], stream=s)
            gu.forward_swiglu(st["h"], out=st["act"], stream=s, norm=(st["g2"], None, EPS))
            down.forward_add(st["act"], st["h"], stream=s)

        _capture(st, layer)
    else:
        _prepare_decode(st, case, seed)
    return st


def _prepare_decode(st, case, seed):
    hidden, hd, heads, kv_heads = (case[x] for x in ("hidden", "hd", "heads", "kv_heads"))
    shapes = _layer_shapes(case)
    width = (heads + 2 * kv_heads) * hd
    st["layers"] = [[_load(case["qtype"], n, k, seed, 10 * i + t) for t, n, k in shapes]
                    for i in range(case["layers"])]
    st["head"] = _load(case["head_qtype"], case["vocab"], hidden, seed, 90)
    st["gamma"] = [_gamma(seed, 200 + i, hidden) for i in range(2 * case["layers"] + 1)]
    st["x"] = _randn(_gen(seed, 100), 1, hidden)
    st["h"] = torch.empty_like(st["x"])
    st["qkv"] = torch.empty(1, width, device="cuda")
    st["att"] = torch.empty(1, heads * hd, device="cuda")
    st["act"] = torch.empty(1, case["inter"], device="cuda")
    st["logits"] = torch.empty(1, case["vocab"], device="cuda")
    st["kv"] = [KvCache(kv_heads, hd, case["past"] + DECODE_ROOM, THETA)
                for _ in range(case["layers"])]
    for i, kv in enumerate(st["kv"]):  # the prompt
        kv.attention(_randn(_gen(seed, 300 + i), case["past"], width), heads)
    torch.cuda.synchronize()
    s = _stream()
    for kv in st["kv"]:  # a captured step cannot allocate: the longest context's workspace
        kv.reserve(1, heads, stream=s)

    def step():
        gam = st["gamma"]
        st["h"].copy_(st["x"])  # the token's embedding row
        for i, ((qkv, o, gu, down), kv) in enumerate(zip(st["layers"], st["kv"])):
            qkv.forward_norm(st["h"], gam[2 * i], eps=EPS, out=st["qkv"], stream=s)
            kv.attention(st["qkv"], heads, out=st["att"], stream=s)
            o.forward_add(st["att"], st["h"], stream=s)
            gu.forward_swiglu(st["h"], out=st["act"], stream=s, norm=(gam[2 * i + 1], None, EPS))
            down.forward_add(st["act"], st["h"], stream=s)
        st["head"].forward_norm(st["h"], gam[-1], eps=EPS, out=st["logits"], stream=s)

    _capture(st, step)
    for kv in st["kv"]:
        kv.truncate(case["past"])
    st["left"] = DECODE_ROOM


# ---- run: one pass ----------------------------------------------------------------------
def run(state):
    case, kind = state["case"], state["kind"]
    if kind == "linear":
        w, x = state["w"], state["x"]
        if case["epi"] == "add":
            return w.forward_add(x, state["y"])
        if case["epi"] == "norm":
            return w.forward_norm(x, state["gamma"], eps=EPS)
        return w.forward(x)
    if kind == "mlp":
        y = state["y"].copy_(state["x"])  # the layer's residual
        act = state["gu"].forward_swiglu(y, norm=(state["gamma"], None, EPS))
        return {"act": act, "out": state["down"].forward_add(act, y)}
    if kind == "prompt_attention":
        state["kv"].truncate(case["past"])  # a new prompt behind the kept prefix
        return state["kv"].attention(state["x"], case["heads"])
    if kind == "batch_layer":
        with torch.cuda.stream(state["stream"]):
            state["graph"].replay()
        return {"qkv": state["qkv"], "act": state["act"], "h": state["h"]}
    if state["left"] == 0:  # the cache is full: back to the prompt
        for kv in state["kv"]:
            kv.truncate(case["past"])
        state["left"] = DECODE_ROOM
    state["left"] -= 1
    with torch.cuda.stream(state["stream"]):
        state["graph"].replay()
    return {"logits": state["logits"], "h": state["h"]}


# ---- what a pass cannot do without ------------------------------------------------------
def _wbytes(qtype, n, k):
    size, elems = BLOCK[qtype]
    return n * k // elems * size


def _proj(qtype, m, n, k):
    return _wbytes(qtype, n, k) + 4 * m * (k + n), 2 * m * n * k


def work(case):
    kind = case["kind"]
    if kind == "linear":
        b, f = _proj(case["qtype"], case["m"], case["n"], case["k"])
        return {"bytes": b + (4 * case["m"] * case["n"] if case["epi"] == "add" else 0), "flops": f}
    if kind == "prompt_attention":
        m, past, hd = case["m"], case["past"], case["hd"]
        qkv = m * (case["heads"] + 2 * case["kv_heads"]) * hd
        cache = 2 * case["kv_heads"] * hd * (past + m)
        return {"bytes": 4 * (qkv + cache + m * case["heads"] * hd),
                "flops": 4 * case["heads"] * hd * m * (past + (m + 1) / 2)}
    hidden, inter = case["hidden"], case["inter"]
    if kind == "mlp":
        shapes, m = [(0, 2 * inter, hidden), (0, hidden, inter)], case["m"]
    else:
        shapes, m = _layer_shapes(case), case.get("m", 1)
    b = sum(_wbytes(case["qtype"], n, k) for _, n, k in shapes)
    f = sum(2 * m * n * k for _, n, k in shapes)
    if kind == "mlp":
        return {"bytes": b + 4 * m * (2 * hidden + 2 * inter), "flops": f}
    if kind == "batch_layer":
        return {"bytes": b + 4 * m * (3 * hidden + case["qkv"] + 2 * inter), "flops": f}
    length = case["past"] + 1
    b += 8 * case["kv_heads"] * case["hd"] * length
    f += 4 * case["heads"] * case["hd"] * length
    hb, hf = _proj(case["head_qtype"], 1, case["vocab"], hidden)
    return {"bytes": case["layers"] * b + hb, "flops": case["layers"] * f + hf}


def tolerance(case):
    # about four times the error against 64 bits that each path shows
    if case["kind"] == "linear" and case["qtype"] in DENSE:
        return {"rel": 4e-6}  # f32 products and sums over k (1.1e-6)
    if case["kind"] == "prompt_attention":
        return {"rel": 2e-6}  # f32 scores, exponentials and sums (4e-7)
    if case["kind"] == "decode_step":
        return {"rel": 1e-3}  # 16-bit fixed-point x, or f16 operands where k is large (1e-4, 3e-4)
    if case["kind"] == "linear":
        return {"rel": 1.5e-3}  # f16 operands: one rounding of x and of each weight (3e-4)
    return {"rel": 4e-3}  # two such projections and SwiGLU behind one another (1e-3)


# ---- the same in 64 bits ----------------------------------------------------------------
def _norm64(x, gamma):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + EPS) * gamma.double()


def _swiglu64(x, w):
    g, u = (x @ w.t()).chunk(2, dim=-1)
    return g * torch.sigmoid(g) * u


def _rope64(t, pos, hd):
    """Rotates [m, heads, hd] at f32 angles pos * inv_freq, halves i and i + hd / 2."""
    e = torch.arange(0, hd, 2, device="cuda", dtype=torch.float32) / hd
    inv = 1.0 / torch.pow(torch.tensor(THETA, dtype=torch.float64, device="cuda"),
                          e.double()).float()
    ang = (pos.float()[:, None] * inv[None, :]).double()
    c, s = ang.cos()[:, None, :], ang.sin()[:, None, :]
    a, b = t[..., : hd // 2], t[..., hd // 2:]
    return torch.cat([a * c - b * s, a * s + b * c], dim=-1)


def _split64(qkv, heads, kv_heads, hd, first):
    m = qkv.shape[0]
    pos = torch.arange(first, first + m, device="cuda")
    q, k, v = qkv.double().split([heads * hd, kv_heads * hd, kv_heads * hd], dim=-1)
    q = _rope64(q.view(m, heads, hd), pos, hd)
    return q, _rope64(k.view(m, kv_heads, hd), pos, hd), v.view(m, kv_heads, hd)


def _attention64(q, k, v, first):
    m, heads, hd = q.shape
    group = heads // k.shape[1]
    out = torch.empty(m, heads, hd, dtype=torch.float64, device="cuda")
    ahead = (torch.arange(k.shape[0], device="cuda")[None, :]
             > torch.arange(first, first + m, device="cuda")[:, None])
    for h in range(heads):
        s = (q[:, h] @ k[:, h // group].t()) / math.sqrt(hd)
        out[:, h] = torch.softmax(s.masked_fill(ahead, -math.inf), dim=-1) @ v[:, h // group]
    return out.view(m, heads * hd)


def _past64(case, seed, tag):
    width = (case["heads"] + 2 * case["kv_heads"]) * case["hd"]
    x = _randn(_gen(seed, tag), case["past"], width)
    return _split64(x, case["heads"], case["kv_heads"], case["hd"], 0)[1:]


def _attend64(case, qkv, past, first):
    q, k, v = _split64(qkv, case["heads"], case["kv_heads"], case["hd"], first)
    if past is not None:
        k, v = torch.cat([past[0], k]), torch.cat([past[1], v])
    return _attention64(q, k, v, first)


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        w = _weight(case["qtype"], case["n"], case["k"], seed, 0, values=True)
        x = _randn(_gen(seed, 100), case["m"], case["k"]).double()
        if case["epi"] == "norm":
            x = _norm64(x, _gamma(seed, 102, case["k"]))
        y = x @ w.t()
        if case["epi"] == "add":
            y += _randn(_gen(seed, 101), case["m"], case["n"]).double()
        return y
    if kind == "prompt_attention":
        width = (case["heads"] + 2 * case["kv_heads"]) * case["hd"]
        x = _randn(_gen(seed, 100), case["m"], width)
        past = _past64(case, seed, 103) if case["past"] else None
        return _attend64(case, x, past, case["past"])
    hidden, inter = case["hidden"], case["inter"]

    def weight(tag, n, k, qtype=case["qtype"]):
        return _weight(qtype, n, k, seed, tag, values=True)

    if kind == "mlp":
        x = _randn(_gen(seed, 100), case["m"], hidden).double()
        act = _swiglu64(_norm64(x, _gamma(seed, 102, hidden)), weight(2, 2 * inter, hidden))
        return {"act": act, "out": x + act @ weight(3, hidden, inter).t()}
    shapes = _layer_shapes(case)
    if kind == "batch_layer":
        x = _randn(_gen(seed, 100), case["m"], hidden).double()
        att = _randn(_gen(seed, 101), case["m"], hidden).double()
        qkv = _norm64(x, _gamma(seed, 102, hidden)) @ weight(*shapes[0]).t()
        h = x + att @ weight(*shapes[1]).t()
        act = _swiglu64(_norm64(h, _gamma(seed, 103, hidden)), weight(*shapes[2]))
        return {"qkv": qkv, "act": act, "h": h + act @ weight(*shapes[3]).t()}
    h = _randn(_gen(seed, 100), 1, hidden).double()
    for i in range(case["layers"]):
        w = [(10 * i + t, n, k) for t, n, k in shapes]
        qkv = _norm64(h, _gamma(seed, 200 + 2 * i, hidden)) @ weight(*w[0]).t()
        att = _attend64(case, qkv, _past64(case, seed, 300 + i), case["past"])
        h = h + att @ weight(*w[1]).t()
        act = _swiglu64(_norm64(h, _gamma(seed, 201 + 2 * i, hidden)), weight(*w[2]))
        h = h + act @ weight(*w[3]).t()
    head = weight(90, case["vocab"], hidden, case["head_qtype"])
    return {"logits": _norm64(h, _gamma(seed, 200 + 2 * case["layers"], hidden)) @ head.t(), "h": h}
