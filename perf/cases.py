"""Performance cases of the quantized decode-linear library.

A case is one call, or one short fixed sequence of calls, that a program using
the library makes over and over: a projection, the linears of decoder layers
at a batch or prefill size, a large prefill linear, the LM head with its
greedy argmax, decode attention over a long cache, and a whole decode step.
`draw` spreads further cases over the same ranges.

Kinds
  linear     one `Context.linear` call, launched eagerly
  layers     the linears of `layers` decoder layers of the 0.8B-shaped model
             (q/k/v grouped with RMSNorm-in; o_proj + residual; gate/up with
             RMSNorm-in and SwiGLU-out; down_proj + residual) on M rows,
             captured once into a HIP graph and replayed, as
             `DecodeSession.capture` does with a step
  lmhead     the LM head with the final RMSNorm fused, fp32 logits and argmax
  attention  RoPE, K/V append and decode attention over `length` positions
  decode     one fused decode step and its LM head, with the logits

Weights, activations, scales and norms have the distributions of the
benchmark's synthetic model (aiimage_amd/synth.py).
"""
import math

import numpy as np
import torch

from aiimage_amd import aexq, decoder

P4 = aexq.LAYOUT_PACK4_LINEAR
VOCAB = 151936
HIDDEN, QW, KVW, INTER = 1024, 2048, 512, 3584
HEAD_DIM, ROPE_BASE, EPS = 128, 1e6, 1e-6

# name: (bits, scale group (0: one per row), fp32 scales, nibble code)
FORMATS = {
    "q4g32": (4, 32, False, aexq.NIBBLE_OFFSET8),  # the benchmark's Q4
    "q4g16": (4, 16, True, aexq.NIBBLE_TWOS),      # the reference archives' shipping Q4
    "q8": (8, 0, False, aexq.NIBBLE_TWOS),         # the benchmark's Q8 and the tied LM head
    "q8f32": (8, 0, True, aexq.NIBBLE_TWOS),       # the reference archives' Q8
}

# M * N * K (SwiGLU counts both weights) a drawn linear stays below, and one
# whose K is no multiple of 64
MOST_MACS = 2 * 2048 * 8192 * 2048
MOST_MACS_ODD_K = 1 << 27


def listed():
    return [
        # the smallest call: one projection of one token
        {"name": "proj_m1", "kind": "linear", "fmt": "q4g32", "m": 1, "n": 512, "k": 1024,
         "epi": "plain", "f32": False},
        # a handful of sequences decoded together
        {"name": "layers_q4_m5", "kind": "layers", "fmt": "q4g32", "m": 5, "layers": 8},
        # batched decode in the format the reference ships
        {"name": "layers_q4g16_m16", "kind": "layers", "fmt": "q4g16", "m": 16, "layers": 8},
        # a short prompt
        {"name": "layers_q8_m64", "kind": "layers", "fmt": "q8f32", "m": 64, "layers": 4},
        # an ordinary prompt
        {"name": "layers_q4_m512", "kind": "layers", "fmt": "q4g32", "m": 512, "layers": 2},
        # a long prompt through the gate/up pair of a larger model
        {"name": "swiglu_q8_m2048", "kind": "linear", "fmt": "q8", "m": 2048, "n": 8192,
         "k": 2048, "epi": "swiglu", "f32": False},
        # a prompt of odd length through a square projection of a larger model
        {"name": "proj_q4g16_m1000", "kind": "linear", "fmt": "q4g16", "m": 1000, "n": 4096,
         "k": 4096, "epi": "residual", "f32": False},
        # odd and ragged in every dimension, with a bias and fp32 outputs
        {"name": "ragged_q8_m77", "kind": "linear", "fmt": "q8f32", "m": 77, "n": 1001, "k": 1008,
         "epi": "bias", "f32": True},
        # the next token of one sequence, and of eight
        {"name": "lmhead_m1", "kind": "lmhead", "m": 1, "n": VOCAB, "k": HIDDEN},
        {"name": "lmhead_m8", "kind": "lmhead", "m": 8, "n": VOCAB, "k": HIDDEN},
        # one layer's attention late in a long document
        {"name": "attention_16k", "kind": "attention", "heads_q": 16, "heads_kv": 4,
         "length": 16384},
        # one generated token of the whole model
        {"name": "decode_24l", "kind": "decode", "fmt": "q4g32", "layers": 24, "position": 2000,
         "capacity": 2048},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear"] * 5 + ["layers"] * 3 + ["lmhead", "attention", "decode"])
    if kind == "layers":
        m = _log_int(rng, 1, 1024)
        return {"kind": kind, "fmt": rng.choice(sorted(FORMATS)), "m": m,
                "layers": max(1, min(8, 1024 // m))}
    if kind == "lmhead":
        k = 128 * rng.randint(4, 16)
        n = min(_log_int(rng, 16000, VOCAB), VOCAB * HIDDEN // k)
        return {"kind": kind, "m": rng.randint(1, 16), "n": n, "k": k}
    if kind == "attention":
        hkv = rng.choice([1, 2, 4, 8])
        return {"kind": kind, "heads_q": hkv * rng.choice([1, 2, 4, 8]), "heads_kv": hkv,
                "length": _log_int(rng, 16, 32768)}
    if kind == "decode":
        cap = rng.choice([512, 1024, 2048])
        return {"kind": kind, "fmt": rng.choice(["q4g32", "q4g16", "q8f32"]),
                "layers": rng.randint(4, 24), "position": rng.randint(0, cap - 1), "capacity": cap}
    fmt = rng.choice(sorted(FORMATS))
    epi = rng.choice(["plain", "rms", "residual", "bias", "swiglu"])
    m, n = _log_int(rng, 1, 2048), _log_int(rng, 64, 8192)
    if epi != "swiglu" and rng.random() < 0.25:  # K only as aligned as the format needs
        step, most = (32 if fmt == "q4g32" else 16), MOST_MACS_ODD_K
    else:
        step, most = 64, MOST_MACS // 2 if epi == "swiglu" else MOST_MACS
    k = step * max(1, round(_log_int(rng, 256, 4096) / step))
    m = max(1, min(m, most // (n * k)))
    return {"kind": kind, "fmt": fmt, "m": m, "n": n, "k": k, "epi": epi,
            "f32": rng.random() < 0.25}


# ---------------------------------------------------------------- inputs

_ctx = None


def _context():
    """The program's one context (and so its one scratch)."""
    global _ctx
    if _ctx is None:
        _ctx = aexq.Context(0)
    return _ctx


class _Inputs:
    """Seeded inputs on the GPU, drawn in a fixed order."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.g, device="cuda")

    def acts(self, *shape):
        return self.normal(*shape).to(torch.float16)

    def gamma(self, k):
        return 1.0 + 0.02 * self.normal(k)

    def weight(self, fmt, n, k):
        """(int8 codes [n][k], scales, fmt)"""
        bits, group, f32, _ = FORMATS[fmt]
        top = 127 if bits == 8 else 7
        codes = torch.randint(-top, top + 1, (n, k), generator=self.g, device="cuda",
                              dtype=torch.int8)
        scales = self.normal(n if bits == 8 else n * k // group).abs() * (0.02 / top)
        return codes, scales if f32 else scales.to(torch.float16), fmt

    def layer(self, fmt):
        w = {name: self.weight(fmt, n, k) for name, n, k in
             (("q", QW, HIDDEN), ("k", KVW, HIDDEN), ("v", KVW, HIDDEN), ("o", HIDDEN, QW),
              ("gate", INTER, HIDDEN), ("up", INTER, HIDDEN), ("down", HIDDEN, INTER))}
        return w, self.gamma(HIDDEN), self.gamma(HIDDEN)


def _upload(weight):
    codes, scales, fmt = weight
    bits, group, _, nibble = FORMATS[fmt]
    n, k = codes.shape
    flat = codes.reshape(-1)
    if bits == 4:
        nib = (flat + 8 if nibble == aexq.NIBBLE_OFFSET8 else flat & 15).to(torch.uint8)
        flat = nib[0::2] | (nib[1::2] << 4)
    words = flat.cpu().numpy().view(np.uint32)
    return _context().weight(aexq.QuantizedTensor(n * k, group or k, words, scales.cpu().numpy(),
                                                  bits=bits, nibble_code=nibble), n, k)


def _exact_weight(weight):
    codes, scales, fmt = weight
    n, k = codes.shape
    group = FORMATS[fmt][1] or k
    s = scales.to(torch.float64).reshape(n, k // group, 1)
    return (codes.to(torch.float64).reshape(n, k // group, group) * s).reshape(n, k)


def _norm(x, gamma):
    x = x.to(torch.float64)
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gamma.to(torch.float64)


def _silu(v):
    return v / (1.0 + torch.exp(-v))


def _rope_tables(capacity):
    return decoder.rope_tables(capacity, HEAD_DIM, ROPE_BASE)


def _rope_row(position):
    """cos and sin of one position's angles (float32 angles, as the tables hold)."""
    j = np.arange(HEAD_DIM // 2, dtype=np.float32)
    inv = np.float32(1) / np.power(np.float64(np.float32(ROPE_BASE)),
                                   (j * np.float32(2.0 / HEAD_DIM)).astype(np.float64)
                                   ).astype(np.float32)
    angle = (np.float32(position) * inv).astype(np.float64)
    return (torch.as_tensor(np.cos(angle), device="cuda"),
            torch.as_tensor(np.sin(angle), device="cuda"))


def _rotate(x, cos, sin):
    h = HEAD_DIM // 2
    a, b = x[..., :h].to(torch.float64), x[..., h:].to(torch.float64)
    return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)


def _attend(q, k, v):
    """q [hq][d] over k, v [hkv][length][d], 64 bits."""
    hkv = k.shape[0]
    out = []
    for g, qg in enumerate(q.reshape(hkv, -1, HEAD_DIM)):
        p = torch.softmax(qg @ k[g].T.contiguous() / math.sqrt(HEAD_DIM), -1)
        out.append(p @ v[g])
    return torch.cat(out)


def _linear_inputs(case, seed):
    r = _Inputs(seed)
    m, n, k, epi = case["m"], case["n"], case["k"], case["epi"]
    d = {"w": r.weight(case["fmt"], n, k), "x": r.acts(m, k)}
    if epi == "swiglu":
        d["up"] = r.weight(case["fmt"], n, k)
    if epi in ("rms", "swiglu"):
        d["gamma"] = r.gamma(k)
    if epi == "residual":
        d["res"] = r.acts(m, n)
    if epi == "bias":
        d["c"] = r.normal(n)
    return d


def _layers_inputs(case, seed):
    r = _Inputs(seed)
    return [(r.layer(case["fmt"]), r.acts(case["m"], HIDDEN), r.acts(case["m"], QW))
            for _ in range(case["layers"])]


def _lmhead_inputs(case, seed):
    r = _Inputs(seed)
    return (r.weight("q8", case["n"], case["k"]), r.acts(case["m"], case["k"]),
            r.gamma(case["k"]))


def _attention_inputs(case, seed):
    r = _Inputs(seed)
    hq, hkv, cap = case["heads_q"], case["heads_kv"], case["length"]
    return (r.acts(hq, HEAD_DIM), r.acts(hkv, HEAD_DIM), r.acts(hkv, HEAD_DIM),
            r.acts(hkv, cap, HEAD_DIM), r.acts(hkv, cap, HEAD_DIM))


def _decode_inputs(case, seed):
    r = _Inputs(seed)
    cap = case["capacity"]
    lm, g_final = r.weight("q8", VOCAB, HIDDEN), r.gamma(HIDDEN)
    token = int(torch.randint(0, VOCAB, (1,), generator=r.g, device="cuda"))
    layers = [(r.layer(case["fmt"]), r.acts(4, cap, HEAD_DIM), r.acts(4, cap, HEAD_DIM))
              for _ in range(case["layers"])]
    return lm, g_final, token, layers


# ---------------------------------------------------------------- prepare and run

def _padded(t, n):
    """Rows of t [m][n] in Pack4 linear storage (the tail lanes zero)."""
    return torch.nn.functional.pad(t, (0, -n % 4)).contiguous()


def _rows(buf, m, n):
    """The logical [m][n] rows of a Pack4 linear buffer."""
    return buf.reshape(m, -1)[:, :n]


def _prepare_linear(case, seed):
    ctx, d = _context(), _linear_inputs(case, seed)
    m, n, k = case["m"], case["n"], case["k"]
    dt = torch.float32 if case["f32"] else torch.float16
    y = aexq.new_activation(m, n, dt, P4)
    kw = {}
    if "up" in d:
        kw["up"] = _upload(d["up"])
    if "gamma" in d:
        kw.update(rmsnorm=True, rms_gamma=d["gamma"], rms_eps=EPS)
    if "res" in d:
        kw["residual"] = aexq.describe(_padded(d["res"].to(dt), n), m, n, P4)
    if "c" in d:
        kw.update(c=d["c"], broadcast_c=4, alpha=1.0, beta=1.0)
    return {"ctx": ctx, "w": _upload(d["w"]), "x": aexq.describe(d["x"], m, k),
            "y": aexq.describe(y, m, n, P4), "kw": kw, "out": _rows(y, m, n)}


def _prepare_layers(case, seed):
    ctx, m = _context(), case["m"]
    d = aexq.describe
    work, outs = [], []
    for (w, g_attn, g_mlp), x, attn in _layers_inputs(case, seed):
        q = {name: _upload(v) for name, v in w.items()}
        y = {name: aexq.new_activation(m, n, torch.float16, P4) for name, n in
             (("q", QW), ("k", KVW), ("v", KVW), ("xb", HIDDEN), ("h", INTER), ("xa", HIDDEN))}
        t = {name: d(v, m, v.numel() // m, P4) for name, v in y.items()}
        t["x"], t["attn"] = d(x, m, HIDDEN, P4), d(attn, m, QW, P4)
        work.append((q, g_attn, g_mlp, t))
        outs.append({name: _rows(v, m, v.numel() // m) for name, v in y.items()})

    def linears():
        for q, g_attn, g_mlp, t in work:
            ctx.linear_group([q["q"], q["k"], q["v"]], t["x"], [t["q"], t["k"], t["v"]],
                             rmsnorm=True, rms_gamma=g_attn, rms_eps=EPS)
            ctx.linear(q["o"], t["attn"], t["xb"], residual=t["x"])
            ctx.linear(q["gate"], t["xb"], t["h"], rmsnorm=True, rms_gamma=g_mlp, rms_eps=EPS,
                       up=q["up"])
            ctx.linear(q["down"], t["h"], t["xa"], residual=t["xb"])

    stream, old = torch.cuda.Stream(), ctx.stream
    ctx.set_stream(stream)
    try:
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            linears()  # sizes the context's scratch before the capture
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
            linears()
    finally:
        ctx.set_stream(old)
    return {"graph": graph, "out": outs, "keep": work}


def _prepare_lmhead(case, seed):
    w, x, gamma = _lmhead_inputs(case, seed)
    m, n, k = case["m"], case["n"], case["k"]
    logits = aexq.new_activation(m, n, torch.float32, P4)
    return {"ctx": _context(), "w": _upload(w), "x": aexq.describe(x, m, k), "gamma": gamma,
            "logits": aexq.describe(logits, m, n, P4), "out": _rows(logits, m, n),
            "argmax": torch.zeros(m, dtype=torch.int32, device="cuda")}


def _prepare_attention(case, seed):
    q, k, v, kc, vc = _attention_inputs(case, seed)
    cos, sin = (torch.as_tensor(t[case["length"] - 1]).cuda()
                for t in _rope_tables(case["length"]))
    return {"ctx": _context(), "q": q, "k": k, "v": v, "kc": kc, "vc": vc, "cos": cos, "sin": sin,
            "out": torch.zeros_like(q), "case": case}


def _prepare_decode(case, seed):
    ctx = _context()
    lm, g_final, token, layers = _decode_inputs(case, seed)
    bits, group, f32, nibble = FORMATS[case["fmt"]]
    cfg = decoder.ModelConfig(layers=case["layers"], capacity=case["capacity"], group=group or 32,
                              scales_f32=f32, layer_bits=bits, nibble_code=nibble)
    long = {"q": "q_proj", "k": "k_proj", "v": "v_proj", "o": "o_proj", "gate": "gate_proj",
            "up": "up_proj", "down": "down_proj"}
    weights = decoder.ModelWeights(
        [{"w": {long[name]: _upload(v) for name, v in w.items()}, "g_attn": g_attn.cpu().numpy(),
          "g_mlp": g_mlp.cpu().numpy()} for (w, g_attn, g_mlp), _, _ in layers],
        _upload(lm), g_final.cpu().numpy())
    s = decoder.DecodeSession(ctx, cfg, fused=True, weights=weights)
    for mine, (_, kc, vc) in zip(s.layers, layers):
        mine["k_cache"].copy_(kc.reshape(-1))
        mine["v_cache"].copy_(vc.reshape(-1))
    s.token.fill_(token)
    s.set_position(case["position"])
    logits = aexq.new_activation(1, VOCAB, torch.float32, P4)
    return {"session": s, "logits": aexq.describe(logits, 1, VOCAB, P4), "out": logits}


def prepare(case, seed):
    return {"kind": case["kind"], **globals()["_prepare_" + case["kind"]](case, seed)}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        state["ctx"].linear(state["w"], state["x"], state["y"], **state["kw"])
        return state["out"]
    if kind == "layers":
        state["graph"].replay()
        return state["out"]
    if kind == "lmhead":
        state["ctx"].lmhead_argmax(state["w"], state["x"], state["logits"], state["argmax"],
                                   rmsnorm=True, rms_gamma=state["gamma"], rms_eps=EPS)
        return {"logits": state["out"], "argmax": state["argmax"]}
    if kind == "attention":
        s, c = state, state["case"]
        s["ctx"].attention_decode_rope(s["q"], s["k"], s["v"], s["kc"], s["vc"], c["heads_q"],
                                       c["heads_kv"], HEAD_DIM, c["length"], c["length"], s["cos"],
                                       s["sin"], 1.0 / math.sqrt(HEAD_DIM), s["out"])
        return {"out": s["out"], "k_new": s["kc"][:, -1], "v_new": s["vc"][:, -1],
                "k_cache": s["kc"], "v_cache": s["vc"]}
    s = state["session"]
    s.fused.run(s.token, s.pos, s.xa)
    s.ctx.lmhead_argmax(s.lm, s.d["xa"], state["logits"], s.next_token, rmsnorm=True,
                        rms_gamma=s.g_final, rms_eps=s.cfg.eps)
    p = s.position
    cache = lambda name: torch.stack([c[name].view(4, -1, HEAD_DIM)[:, p] for c in s.layers])  # noqa: E731
    return {"hidden": s.xa, "logits": state["out"], "k_new": cache("k_cache"),
            "v_new": cache("v_cache")}


# ---------------------------------------------------------------- what it takes, and how exact

def _weight_bytes(fmt, n, k):
    bits, group, f32, _ = FORMATS[fmt]
    return n * k * bits // 8 + (n if bits == 8 else n * k // group) * (4 if f32 else 2)


def _layer_shapes():
    return ((QW, HIDDEN), (KVW, HIDDEN), (KVW, HIDDEN), (HIDDEN, QW), (INTER, HIDDEN),
            (INTER, HIDDEN), (HIDDEN, INTER))


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        nw = 2 if case["epi"] == "swiglu" else 1
        e = 4 if case["f32"] else 2
        out = m * n * e * (2 if case["epi"] == "residual" else 1)
        return {"bytes": nw * _weight_bytes(case["fmt"], n, k) + 2 * m * k + out
                + (4 * n if case["epi"] == "bias" else 0), "flops": 2 * nw * m * n * k}
    if kind == "layers":
        m, count = case["m"], case["layers"]
        weights = sum(_weight_bytes(case["fmt"], n, k) for n, k in _layer_shapes())
        acts = 2 * m * (HIDDEN + QW + QW + 2 * KVW + HIDDEN + INTER + HIDDEN)
        return {"bytes": count * (weights + acts),
                "flops": count * 2 * m * sum(n * k for n, k in _layer_shapes())}
    if kind == "lmhead":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _weight_bytes("q8", n, k) + 2 * m * k + 4 * m * n + 4 * m,
                "flops": 2 * m * n * k}
    if kind == "attention":
        hq, hkv, length = case["heads_q"], case["heads_kv"], case["length"]
        return {"bytes": 2 * HEAD_DIM * (2 * hkv * length + 2 * hq + 2 * hkv),
                "flops": 4 * hq * length * HEAD_DIM}
    length, count = case["position"] + 1, case["layers"]
    weights = sum(_weight_bytes(case["fmt"], n, k) for n, k in _layer_shapes())
    kv = 2 * 4 * length * HEAD_DIM * 2
    macs = sum(n * k for n, k in _layer_shapes())
    return {"bytes": count * (weights + kv) + _weight_bytes("q8", VOCAB, HIDDEN) + 4 * VOCAB,
            "flops": 2 * (count * (macs + 2 * 16 * length * HEAD_DIM) + VOCAB * HIDDEN)}


def tolerance(case):
    """About four times the error measured against `exact` at the start."""
    kind = case["kind"]
    if kind == "linear":
        # fp32 outputs without a norm differ by the order of the sums only, unless
        # Q4 weight tiles are rounded to fp16 (more than 8 rows)
        if (case["f32"] and case["epi"] in ("plain", "residual", "bias")
                and (case["fmt"].startswith("q8") or case["m"] <= 8)):
            return {"rel": 1e-5}
        return {"rel": 2e-3}  # 5.5e-4: fp16 activations, weight tiles and outputs
    if kind == "layers":
        return {"rel": 2.5e-3}  # 6.6e-4 after the SwiGLU
    if kind == "lmhead":
        return {"rel": 8e-4}  # 2.1e-4: the normalised row is rounded to fp16
    if kind == "attention":
        return {"rel": 1.2e-3}  # 3.1e-4: q, the new k row and the output in fp16
    return {"rel": 1.2e-2}  # 3.1e-3 after 24 layers in fp16


# ---------------------------------------------------------------- 64-bit results

def _exact_linear(case, seed):
    d = _linear_inputs(case, seed)
    x = _norm(d["x"], d["gamma"]) if "gamma" in d else d["x"].to(torch.float64)
    y = x @ _exact_weight(d["w"]).T
    if "up" in d:
        y = _silu(y) * (x @ _exact_weight(d["up"]).T)
    if "res" in d:
        y = y + d["res"].to(torch.float64)
    if "c" in d:
        y = y + d["c"].to(torch.float64)
    return y


def _exact_layers(case, seed):
    outs = []
    for (w, g_attn, g_mlp), x, attn in _layers_inputs(case, seed):
        e = {name: _exact_weight(v).T for name, v in w.items()}
        xn = _norm(x, g_attn)
        xb = attn.to(torch.float64) @ e["o"] + x.to(torch.float64)
        hn = _norm(xb, g_mlp)
        h = _silu(hn @ e["gate"]) * (hn @ e["up"])
        outs.append({"q": xn @ e["q"], "k": xn @ e["k"], "v": xn @ e["v"], "xb": xb, "h": h,
                     "xa": h @ e["down"] + xb})
    return outs


def _exact_lmhead(case, seed):
    w, x, gamma = _lmhead_inputs(case, seed)
    return {"logits": _norm(x, gamma) @ _exact_weight(w).T, "argmax": None}


def _exact_attention(case, seed):
    q, k, v, kc, vc = _attention_inputs(case, seed)
    cos, sin = _rope_row(case["length"] - 1)
    kc, vc = kc.to(torch.float64), vc.to(torch.float64)
    kc[:, -1], vc[:, -1] = _rotate(k, cos, sin), v.to(torch.float64)
    return {"out": _attend(_rotate(q, cos, sin), kc, vc), "k_new": kc[:, -1], "v_new": vc[:, -1],
            "k_cache": kc, "v_cache": vc}


def _exact_decode(case, seed):
    lm, g_final, token, layers = _decode_inputs(case, seed)
    p = case["position"]
    cos, sin = _rope_row(p)
    x = (lm[0][token].to(torch.float64) * lm[1][token].to(torch.float64)).reshape(1, -1)
    k_new, v_new = [], []
    for (w, g_attn, g_mlp), kc, vc in layers:
        e = {name: _exact_weight(v).T for name, v in w.items()}
        xn = _norm(x, g_attn)
        k = _rotate((xn @ e["k"]).reshape(4, HEAD_DIM), cos, sin)
        v = (xn @ e["v"]).reshape(4, HEAD_DIM)
        k_new.append(k)
        v_new.append(v)
        ks = torch.cat([kc[:, :p].to(torch.float64), k[:, None]], 1)
        vs = torch.cat([vc[:, :p].to(torch.float64), v[:, None]], 1)
        a = _attend(_rotate((xn @ e["q"]).reshape(16, HEAD_DIM), cos, sin), ks, vs)
        x = a.reshape(1, -1) @ e["o"] + x
        hn = _norm(x, g_mlp)
        x = (_silu(hn @ e["gate"]) * (hn @ e["up"])) @ e["down"] + x
    return {"hidden": x.reshape(-1), "logits": (_norm(x, g_final) @ _exact_weight(lm).T).reshape(-1),
            "k_new": torch.stack(k_new), "v_new": torch.stack(v_new)}


def exact(case, seed):
    return globals()["_exact_" + case["kind"]](case, seed)
