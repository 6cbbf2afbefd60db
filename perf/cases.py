"""The work a user of this package has it do, as measurable cases.

Each case is one pass through public entry points of ``pageserve_amd`` at the
sizes of the models this repository serves: the 2048-hidden, 11008-wide,
36-layer model ("3b") and the 896-hidden, 4864-wide one ("0.5b"), both with a
151936-entry vocabulary.  Kinds:

``linear``     one projection of one weight through the drop-in
               ``F.linear(x, w.get(), bias)``: the smallest call.
``decode``     a decode step's linears for a batch of ``tokens`` sequences: per
               layer ``decode_span`` (o + residual, norm, gate|up, down +
               residual, the next layer's norm, q|k|v and RoPE), captured in a
               HIP graph as a serving loop does.
``prefill``    the same layers for a prompt (chunk) of ``tokens`` tokens through
               the explicit fused calls, launched eagerly.
``logits``     the fp32 lm_head logits of ``tokens`` rows.
``greedy``     the greedy next token of ``tokens`` rows (argmax inside the
               lm_head).
``quantize``   a layer's weights quantized at load (``QuantizedWeight(w)``) from
               an fp32 or bf16 checkpoint.
``rows``       ``quantize_per_channel`` and ``dequantize`` of one weight in
               row-major form, any shape.
``dense``      the dense weights of a layer (``QuantizedWeight.dense``), what
               every operation other than the fused linear computes on.

Attention itself is not part of the package: its outputs are inputs here.
"""

from __future__ import annotations

import torch
import torch.nn.functional as F

from pageserve_amd import quantization as Q
from pageserve_amd import span as S

EPS = 1e-6
VOCAB = 151936
#        hidden, intermediate, kv width, head_dim
MODELS = {"3b": (2048, 11008, 256, 128), "0.5b": (896, 4864, 128, 64)}


def listed():
    return [
        # one small projection of one token through the unchanged F.linear call site
        {"name": "linear-0.5b-1", "kind": "linear", "model": "0.5b", "tokens": 1},
        # one user's decode step (4 of the layers)
        {"name": "decode-3b-1", "kind": "decode", "model": "3b", "tokens": 1, "layers": 4},
        # a small decode batch, and one above 16 sequences
        {"name": "decode-3b-6", "kind": "decode", "model": "3b", "tokens": 6, "layers": 4},
        {"name": "decode-3b-24", "kind": "decode", "model": "3b", "tokens": 24, "layers": 4},
        # a short prompt
        {"name": "prefill-3b-100", "kind": "prefill", "model": "3b", "tokens": 100, "layers": 3},
        # a chunk of the usual prefill token budget
        {"name": "prefill-3b-512", "kind": "prefill", "model": "3b", "tokens": 512, "layers": 2},
        # a long ragged prompt on the small model
        {"name": "prefill-0.5b-1501", "kind": "prefill", "model": "0.5b", "tokens": 1501, "layers": 8},
        # the largest prefill chunk
        {"name": "prefill-3b-2048", "kind": "prefill", "model": "3b", "tokens": 2048, "layers": 2},
        # sampling from the logits of a small batch
        {"name": "logits-3b-8", "kind": "logits", "model": "3b", "tokens": 8},
        # greedy decoding, one sequence
        {"name": "greedy-3b-1", "kind": "greedy", "model": "3b", "tokens": 1},
        # loading one layer of an fp32 checkpoint
        {"name": "quantize-3b-f32", "kind": "quantize", "model": "3b", "dtype": "f32"},
        # one layer's dense weights
        {"name": "dense-3b-bf16", "kind": "dense", "model": "3b", "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(["linear", "decode", "decode", "prefill", "prefill", "prefill", "logits", "greedy", "quantize",
                       "rows", "dense"])
    model = rng.choice(["3b", "3b", "0.5b"])
    if kind == "linear":
        return {"kind": kind, "model": model, "tokens": _log_int(rng, 1, 2048)}
    if kind == "decode":
        return {"kind": kind, "model": model, "tokens": _log_int(rng, 1, 32), "layers": rng.randint(2, 6)}
    if kind == "prefill":
        return {"kind": kind, "model": model, "tokens": _log_int(rng, 33, 2048), "layers": rng.randint(1, 2)}
    if kind == "logits":
        return {"kind": kind, "model": model, "tokens": _log_int(rng, 1, 256)}
    if kind == "greedy":
        return {"kind": kind, "model": model, "tokens": _log_int(rng, 1, 32)}
    if kind == "rows":
        k = _log_int(rng, 64, 8192)
        if rng.random() < 0.5:
            k = (k + 63) // 64 * 64
        return {"kind": kind, "rows": _log_int(rng, 64, 16384), "cols": k, "dtype": rng.choice(["f32", "bf16"])}
    return {"kind": kind, "model": model, "dtype": rng.choice(["f32", "bf16"])}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def _shapes(model):
    h, inter, kv, _ = MODELS[model]
    return {"q": (h, h), "k": (kv, h), "v": (kv, h), "o": (h, h), "gate": (inter, h), "up": (inter, h),
            "down": (h, inter)}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(gen, *shape, std=1.0, dtype=torch.bfloat16):
    return (torch.randn(shape, generator=gen, device="cuda") * std).to(dtype)


def _inputs(case, seed):
    """The tensors a checkpoint and the caller supply, from the seed alone."""
    gen = _gen(seed)
    kind = case["kind"]
    if kind == "rows":
        return {"w": _randn(gen, case["rows"], case["cols"], std=0.02, dtype=_DTYPES[case["dtype"]])}
    h, inter, kv, hd = MODELS[case["model"]]
    if kind == "linear":
        return {"w": _randn(gen, inter, h, std=0.02), "b": _randn(gen, inter, std=0.1),
                "x": _randn(gen, case["tokens"], h)}
    if kind in ("logits", "greedy"):
        return {"w": _randn(gen, VOCAB, h, std=0.02), "x": _randn(gen, case["tokens"], h)}
    if kind in ("quantize", "dense"):
        return {n: _randn(gen, *s, std=0.02, dtype=_DTYPES[case["dtype"]])
                for n, s in _shapes(case["model"]).items()}
    m = case["tokens"]
    pos = torch.arange(m, device="cuda") if kind == "prefill" else torch.randint(0, 2048, (m,), generator=gen,
                                                                                   device="cuda")
    inv = 1e6 ** (-torch.arange(0, hd, 2, device="cuda").float() / hd)
    ang = (pos.float()[:, None] * inv).repeat(1, 2)
    layers = []
    for _ in range(case["layers"] + (kind == "decode")):
        L = {n: _randn(gen, *s, std=0.02) for n, s in _shapes(case["model"]).items()}
        L["bias"] = [_randn(gen, n, std=0.1) for n in (h, kv, kv)]
        L["ln_in"], L["ln_post"] = ((1 + 0.1 * _randn(gen, h, dtype=torch.float32)).to(torch.bfloat16) for _ in "ab")
        L["attn"] = _randn(gen, m, h)
        layers.append(L)
    return {"layers": layers, "x": _randn(gen, m, h), "cos": ang.cos().to(torch.bfloat16),
            "sin": ang.sin().to(torch.bfloat16)}


def prepare(case, seed):
    kind = case["kind"]
    st = _inputs(case, seed)
    st["case"] = case
    if kind in ("linear", "logits", "greedy"):
        st["w"] = Q.QuantizedWeight(st["w"])
    elif kind == "dense":
        for n in _shapes(case["model"]):
            st[n] = Q.QuantizedWeight(st[n])
    elif kind in ("decode", "prefill"):
        for L in st["layers"]:
            for n in _shapes(case["model"]):
                L[n] = Q.QuantizedWeight(L[n])
        if kind == "decode":
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                _decode(st)  # the warm-up a capture needs
            torch.cuda.current_stream().wait_stream(side)
            st["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(st["graph"]):
                st["out"] = _decode(st)
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def _decode(st):
    """From one layer's attention output to the next layer's q, k, v."""
    x, outs = st["x"], []
    hd = MODELS[st["case"]["model"]][3]
    layers = st["layers"]
    for L, nxt in zip(layers, layers[1:]):
        x, qkv = S.decode_span(L["attn"], x, L["o"], L["ln_post"], L["gate"], L["up"], L["down"], EPS,
                               next_ln=nxt["ln_in"], next_qkv=(nxt["q"], nxt["k"], nxt["v"]),
                               next_bias=tuple(nxt["bias"]), cos=st["cos"], sin=st["sin"], head_dim=hd)
        outs.append([x, *qkv])
    return outs


def _prefill(st):
    x, outs = st["x"], []
    hd = MODELS[st["case"]["model"]][3]
    m = x.shape[0]
    for L in st["layers"]:
        q, k, v = Q.rmsnorm_linear_group(x, L["ln_in"], EPS, [L["q"], L["k"], L["v"]], L["bias"])
        q, k = Q.rope_qk(q.view(m, -1, hd), k.view(m, -1, hd), st["cos"], st["sin"])
        x = L["o"].linear(L["attn"], residual=x)
        x = Q.rmsnorm_mlp(x, L["ln_post"], EPS, L["gate"], L["up"], L["down"], residual=x)
        outs.append([q, k, v, x])
    return outs


def run(st):
    kind = st["case"]["kind"]
    if kind == "linear":
        return F.linear(st["x"], st["w"].get(), st["b"])
    if kind == "decode":
        st["graph"].replay()
        return st["out"]
    if kind == "prefill":
        return _prefill(st)
    if kind == "logits":
        return Q.linear(st["x"], st["w"], out_dtype=torch.float32)
    if kind == "greedy":
        return Q.linear_argmax(st["x"], st["w"], return_values=True)
    if kind == "quantize":
        out = {}
        for n in _shapes(st["case"]["model"]):
            w = Q.QuantizedWeight(st[n])
            out[n] = [w.qp, w.scale]
        return out
    if kind == "rows":
        q, scale = Q.quantize_per_channel(st["w"])
        return [q, scale, Q.dequantize(q, scale, st["w"].dtype)]
    return {n: st[n].dense() for n in _shapes(st["case"]["model"])}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _linear_work(m, n, k, out_bytes=2):
    return {"bytes": n * k + 4 * n + 2 * m * k + out_bytes * m * n, "flops": 2 * m * n * k}


def work(case):
    kind = case["kind"]
    if kind == "rows":
        n, k = case["rows"], case["cols"]
        e = 4 if case["dtype"] == "f32" else 2
        return {"bytes": n * k * (e + 1 + e) + 4 * n, "flops": 0}
    h, inter, kv, hd = MODELS[case["model"]]
    if kind == "linear":
        w = _linear_work(case["tokens"], inter, h)
        return {"bytes": w["bytes"] + 2 * inter, "flops": w["flops"]}
    if kind == "logits":
        return _linear_work(case["tokens"], VOCAB, h, 4)
    if kind == "greedy":
        m = case["tokens"]
        return {"bytes": VOCAB * (h + 4) + 2 * m * h + 12 * m, "flops": 2 * m * VOCAB * h}
    rows = sum(n for n, _ in _shapes(case["model"]).values())
    weights = sum(n * k for n, k in _shapes(case["model"]).values())
    if kind in ("quantize", "dense"):
        e = 4 if case["dtype"] == "f32" else 2
        return {"bytes": weights * (e + 1) + 4 * rows, "flops": 0}
    m, layers = case["tokens"], case["layers"]
    # per layer: the weights and scales, biases and norm weights, the
    # attention output in, q, k, v and x out; x in and the RoPE rows once
    per = weights + 4 * rows + 2 * (h + 2 * kv) + 4 * h + 2 * m * h + 2 * m * (2 * h + 2 * kv)
    return {"bytes": layers * per + 2 * m * h + 4 * m * hd, "flops": layers * 2 * m * weights}


def tolerance(case):
    kind = case["kind"]
    if kind in ("quantize", "rows", "dense"):
        return "exact"
    if kind == "logits":
        return {"rel": 1e-5, "max": 1e-4}  # fp32 sums of exact products
    if kind == "greedy":
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.04}  # a tie among the 151936 logits of a row
    # bf16 results of fp32 sums; in the layers, bf16 at every boundary
    return {"rel": 1e-2, "max": 8e-2}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------

def _quant(w):
    """(q, scale) of the definition: per row absmax / 127 in fp32, the fp32
    quotient rounded half to even (both quotients correctly rounded: taken in
    64 bits, then rounded to fp32)."""
    amax = w.float().abs().amax(dim=1, keepdim=True).clamp(min=1e-8)
    scale = (amax.double() / 127.0).float()
    return (w.double() / scale.double()).float().round().clamp(-127, 127), scale


def _deq(w):
    q, scale = _quant(w)
    return q.double() * scale.double()


def _packed(q):
    """Row-major [n, k] in the stored order: 16-row x 64-column blocks, in
    each the four 16-column groups, in each the rows."""
    n, k = q.shape
    tn, tk = -(-n // 16), -(-k // 64)
    p = torch.zeros((tn * 16, tk * 64), dtype=q.dtype, device=q.device)
    p[:n, :k] = q
    return p.view(tn, 16, tk, 4, 16).permute(0, 2, 3, 1, 4).reshape(-1)


def _norm(x, w):
    return w.double() * (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS))


def _rope(x, cos, sin, hd):
    x = x.view(x.shape[0], -1, hd)
    x1, x2 = x.chunk(2, dim=-1)
    return x * cos.double()[:, None] + torch.cat((-x2, x1), -1) * sin.double()[:, None]


def _qkv(L, x, st, hd):
    h = _norm(x, L["ln_in"])
    q, k, v = (h @ _deq(L[n]).T + b.double() for n, b in zip("qkv", L["bias"]))
    return _rope(q, st["cos"], st["sin"], hd), _rope(k, st["cos"], st["sin"], hd), v


def _after_attention(L, x):
    x = x + L["attn"].double() @ _deq(L["o"]).T
    h = _norm(x, L["ln_post"])
    return x + (F.silu(h @ _deq(L["gate"]).T) * (h @ _deq(L["up"]).T)) @ _deq(L["down"]).T


def exact(case, seed):
    kind = case["kind"]
    st = _inputs(case, seed)
    if kind == "rows":
        q, scale = _quant(st["w"])
        return [q.to(torch.int8), scale.double(), q.double() * scale.double()]
    if kind == "linear":
        return st["x"].double() @ _deq(st["w"]).T + st["b"].double()
    if kind in ("logits", "greedy"):
        x = st["x"].double()
        y = torch.cat([x @ _deq(w).T for w in st["w"].split(16384)], dim=1)
        if kind == "logits":
            return y
        v, i = y.max(dim=1)
        return [i, v]
    if kind == "quantize":
        out = {}
        for n in _shapes(case["model"]):
            q, scale = _quant(st[n])
            out[n] = [_packed(q.to(torch.int8)), scale.double()]
        return out
    if kind == "dense":
        return {n: _deq(st[n]) for n in _shapes(case["model"])}
    hd = MODELS[case["model"]][3]
    x, m, outs = st["x"].double(), case["tokens"], []
    layers = st["layers"]
    if kind == "decode":
        for L, nxt in zip(layers, layers[1:]):
            x = _after_attention(L, x)
            q, k, v = _qkv(nxt, x, st, hd)
            outs.append([x, q.reshape(m, -1), k.reshape(m, -1), v])
        return outs
    for L in layers:
        q, k, v = _qkv(L, x, st, hd)
        x = _after_attention(L, x)
        outs.append([q, k, v, x])
    return outs
