"""The work whose speed is measured: calls that a program built on this library makes.

The ranges behind the listed cases, which draw() samples:
  gemv      one token through a linear layer: MXFP4, int8 or fp16 weights, 256..16384 rows by 512..8192
            values (fp16 up to a vocabulary of 151,936 rows)
  rows      2..8 tokens (a speculative verify) through a linear layer or the fp16 head
  gemm      9..8192 tokens (a chat turn, a prompt, a piece of a long prompt) through MXFP4 or int8 weights
  attend    one token's attention over 64..65,536 cached keys, fp16 or int8
  prompt_attend  1..4096 tokens' causal attention, behind 0..8192 keys that the cache holds already
  moe       1..8 tokens through a mixture-of-experts layer, router choice included
  decode    steps of the whole 28-layer decoder behind 16..4096 tokens
  prompt    a prompt of 16..1024 tokens through the whole decoder
"""
import math

import torch

from hwnpu_amd import ops, qwen3

FP4 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0]
MODEL = dict(layers=28, hidden=2048, heads=16, kv_heads=8, inter=6144, vocab=151936)
THETA, EPS = 1e6, 1e-6


def listed():
    return [
        # the smallest call: one token through a decoder linear, where latency counts
        {"name": "gemv mxfp4 8192x2048", "kind": "gemv", "weights": "mxfp4", "n": 8192, "k": 2048, "out": "f16"},
        # a verify of 4 drafts through gate and up
        {"name": "rows mxfp4 5x12288x2048", "kind": "rows", "weights": "mxfp4", "tokens": 5, "n": 12288, "k": 2048,
         "out": "f32"},
        # the same verify through the tied head: a logits row for each token
        {"name": "rows head 5x151936x2048", "kind": "rows", "weights": "f16", "tokens": 5, "n": 151936, "k": 2048,
         "out": "f32"},
        # a short chat turn through the down projection
        {"name": "gemm mxfp4 37x2048x6144", "kind": "gemm", "weights": "mxfp4", "m": 37, "n": 2048, "k": 6144,
         "out": "f32"},
        # a prompt through an int8 linear
        {"name": "gemm int8 512x6144x2048", "kind": "gemm", "weights": "int8", "m": 512, "n": 6144, "k": 2048,
         "out": "f16"},
        # a long document through gate and up, SwiGLU included
        {"name": "gemm mxfp4 6001x12288x2048", "kind": "gemm", "weights": "mxfp4", "m": 6001, "n": 12288, "k": 2048,
         "out": "swiglu"},
        # one token over a long conversation
        {"name": "attend fp16 8191", "kind": "attend", "kv": "fp16", "heads": 32, "kv_heads": 8, "len": 8191,
         "out": "f16"},
        # one token over a book-sized context in an int8 cache
        {"name": "attend int8 32768", "kind": "attend", "kv": "int8", "heads": 32, "kv_heads": 8, "len": 32768,
         "out": "f16"},
        # a chat turn's attention over the conversation before it
        {"name": "prompt_attend 33 behind 8000", "kind": "prompt_attend", "heads": 16, "kv_heads": 8, "tokens": 33,
         "start": 8000, "out": "f16"},
        # a verify of 4 drafts through an MoE layer
        {"name": "moe 5 tokens", "kind": "moe", "tokens": 5, "hidden": 2048, "inter": 768, "experts": 32, "top": 4,
         "act": "silu"},
        # the decoder's steps behind a prompt, the tokens given (a sampler's choice, or a constrained output)
        {"name": "decode 8 behind 1024", "kind": "decode", "behind": 1024, "steps": 8},
        # a prompt through the decoder: logits, and the rows that a prompt store keeps
        {"name": "prompt 1024", "kind": "prompt", "tokens": 1024},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _mult(rng, lo, hi, of):
    return max(1, _log(rng, lo, hi) // of) * of


def draw(rng):
    kind = rng.choice(["gemv", "rows", "gemm", "gemm", "attend", "prompt_attend", "moe", "decode", "prompt"])
    if kind == "gemv":
        weights = rng.choice(["mxfp4", "int8", "f16"])
        return {"kind": kind, "weights": weights, "n": _log(rng, 256, 151936 if weights == "f16" else 16384),
                "k": _mult(rng, 512, 8192, 32), "out": rng.choice(["f32", "f16"])}
    if kind == "rows":
        weights, tokens = rng.choice(["mxfp4", "f16"]), rng.randint(2, 8)
        return {"kind": kind, "weights": weights, "tokens": tokens, "n": _log(rng, 256, 16384 if weights == "mxfp4" else 151936),
                "k": _mult(rng, 512, min(8192, 32768 // tokens), 32), "out": rng.choice(["f32", "f16"])}
    if kind == "gemm":
        out = rng.choice(["f32", "f16", "swiglu"])
        n = _mult(rng, 512, 16384, 16) if out == "swiglu" or rng.random() < 0.7 else _log(rng, 512, 16384)
        return {"kind": kind, "weights": rng.choice(["mxfp4", "int8"]), "m": _log(rng, 9, 8192), "n": n,
                "k": _mult(rng, 512, 8192, 32 if rng.random() < 0.3 else 128), "out": out}
    if kind == "attend":
        heads, kvh = rng.choice([(32, 8), (16, 8), (8, 8)])
        return {"kind": kind, "kv": rng.choice(["fp16", "int8"]), "heads": heads, "kv_heads": kvh,
                "len": _log(rng, 64, 65536), "out": rng.choice(["f32", "f16"])}
    if kind == "prompt_attend":
        heads, kvh = rng.choice([(32, 8), (16, 8), (8, 8)])
        return {"kind": kind, "heads": heads, "kv_heads": kvh, "tokens": _log(rng, 1, 4096),
                "start": rng.choice([0, _log(rng, 16, 8192)]), "out": rng.choice(["f32", "f16"])}
    if kind == "moe":
        if rng.random() < 0.5:
            return {"kind": kind, "tokens": rng.randint(1, 8), "hidden": 2048, "inter": _mult(rng, 512, 2048, 32),
                    "experts": rng.choice([16, 32, 64]), "top": rng.choice([2, 4, 8]), "act": "silu"}
        return {"kind": kind, "tokens": rng.randint(1, 8), "hidden": 2880, "inter": 2880, "experts": 32, "top": 4,
                "act": "gptoss"}
    if kind == "decode":
        return {"kind": kind, "behind": _log(rng, 16, 4096), "steps": rng.randint(1, 12)}
    return {"kind": kind, "tokens": _log(rng, 16, 1023)}


# ---- inputs, from the seed alone ----

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, *shape, dtype=torch.float16):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def _bytes(g, lo, hi, *shape):
    return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.uint8)


def _mxfp4(g, *lead, k):
    """Codes over all 16 values and block scales 2^-9 .. 2^-7: values of about 0.02, as a model's weights."""
    return _bytes(g, 0, 256, *lead, k // 2), _bytes(g, 118, 121, *lead, k // 32)


def _weights(g, c, n, k):
    if c["weights"] == "mxfp4":
        return _mxfp4(g, n, k=k)
    if c["weights"] == "int8":
        q = torch.randint(-127, 128, (n, k), generator=g, device="cuda", dtype=torch.int8)
        s = (torch.rand(n, generator=g, device="cuda") * 3e-4 + 1e-4).half()
        return q, s
    return ((_normal(g, n, k, dtype=torch.float32) * 0.02).half(),)


def _kv(g, kvh, rows, int8):
    """A cache's rows: fp16, or int8 codes with the fp16 scale of each row's largest value over 127."""
    x = _normal(g, kvh, rows, 128, dtype=torch.float32)
    if not int8:
        return x.half(), None
    s = (x.abs().amax(-1) / 127).half()
    return (x / s.float()[..., None]).round().clamp(-127, 127).to(torch.int8), s


def _model_names(layers):
    for i in range(layers):
        for lin in ("qkv", "o", "gate_up", "down"):
            yield i, lin


def _model_shape(lin):
    h, a, kv, f = MODEL["hidden"], MODEL["heads"] * 128, MODEL["kv_heads"] * 128, MODEL["inter"]
    return {"qkv": (a + 2 * kv, h), "o": (h, a), "gate_up": (2 * f, h), "down": (h, f)}[lin]


def _model_weights(seed):
    """(name, tensor) of every weight of the decoder, one after another."""
    g = _gen(seed)
    for i, lin in _model_names(MODEL["layers"]):
        n, k = _model_shape(lin)
        w, e = _mxfp4(g, n, k=k)
        yield f"layers.{i}.{lin}.blocks", w
        yield f"layers.{i}.{lin}.scales", e
    for i in range(MODEL["layers"]):
        for name, n in (("input_norm", MODEL["hidden"]), ("post_norm", MODEL["hidden"]), ("q_norm", 128), ("k_norm", 128)):
            yield f"layers.{i}.{name}", 1 + 0.1 * _normal(g, n, dtype=torch.float32)
    yield "norm", 1 + 0.1 * _normal(g, MODEL["hidden"], dtype=torch.float32)
    yield "embed", (_normal(g, MODEL["vocab"], MODEL["hidden"], dtype=torch.float32) * 0.02).half()


def _tokens(c, seed):
    """The prompt's tokens and those of the steps after it."""
    n = c["tokens"] if c["kind"] == "prompt" else c["behind"] + c["steps"]
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, MODEL["vocab"], (n,), generator=g).tolist()


def prepare(c, seed):
    kind = c["kind"]
    if kind in ("decode", "prompt"):
        tokens = _tokens(c, seed)
        room = -(-(len(tokens) + 2) // 256) * 256
        m = qwen3.Qwen3(**MODEL, head_dim=128, max_ctx=room, max_prompt=min(1024, room), theta=THETA, eps=EPS)
        for name, t in _model_weights(seed):
            ptr, size = m.tensor(name)
            assert size == t.numel() * t.element_size(), name
            qwen3.d2d(ptr, t.data_ptr(), size)
        if kind == "decode":
            m.prefill(tokens[:c["behind"]])
            m.capture()
            tokens = tokens[c["behind"]:]
        return {"c": c, "model": m, "tokens": tokens}
    g = _gen(seed)
    s = {"c": c}
    if kind == "gemv":
        s["w"], s["x"] = _weights(g, c, c["n"], c["k"]), _normal(g, c["k"])
    elif kind == "rows":
        s["w"], s["x"] = _weights(g, c, c["n"], c["k"]), _normal(g, c["tokens"], c["k"])
    elif kind == "gemm":
        s["w"], s["x"] = _weights(g, c, c["n"], c["k"]), _normal(g, c["m"], c["k"])
    elif kind == "attend":
        room = -(-c["len"] // 256) * 256
        s["q"] = _normal(g, c["heads"], 128)
        s["k"], s["ks"] = _kv(g, c["kv_heads"], room, c["kv"] == "int8")
        s["v"], s["vs"] = _kv(g, c["kv_heads"], room, c["kv"] == "int8")
        p = ops.attn_params(c["heads"], c["kv_heads"], c["len"], room, c["kv"] == "int8")
        s["ws"] = ops.attn_workspace(p)
    elif kind == "prompt_attend":
        room = -(-(c["tokens"] + c["start"]) // 256) * 256
        s["q"] = _normal(g, c["tokens"], c["heads"], 128)
        s["k"], _ = _kv(g, c["kv_heads"], room, False)
        s["v"], _ = _kv(g, c["kv_heads"], room, False)
    else:
        E, H, I = c["experts"], c["hidden"], c["inter"]
        s["x"], s["logits"] = _normal(g, c["tokens"], H), _normal(g, c["tokens"], E, dtype=torch.float32)
        gu, gs = _mxfp4(g, E, 2 * I, k=H)
        dn, ds = _mxfp4(g, E, H, k=I)
        s["experts"] = (gu.view(E, 2 * I, H // 32, 16), gs, dn.view(E, H, I // 32, 16), ds)
        s["bias"] = (None, None)
        if c["act"] == "gptoss":
            s["bias"] = (_normal(g, E, 2 * I, dtype=torch.float32), _normal(g, E, H, dtype=torch.float32))
    return s


def run(s):
    c = s["c"]
    kind = c["kind"]
    if kind == "decode":
        # a program that chooses the tokens itself gives each step its token; the logits follow the last
        m, at = s["model"], c["behind"]
        for i, t in enumerate(s["tokens"]):
            m.rewind(at + i, t)
            m.decode(1)
        return {"logits": m.logits(), "rows": m.export_rows(at, at + c["steps"]).view(torch.float16)}
    if kind == "prompt":
        m = s["model"]
        m.prefill(s["tokens"])
        return {"logits": m.logits(), "rows": m.export_rows(0, c["tokens"]).view(torch.float16)}
    if kind == "gemv":
        call = {"mxfp4": ops.mxfp4_gemv, "int8": ops.i8_gemv, "f16": ops.f16_gemv}[c["weights"]]
        return call(*s["w"], s["x"], c["out"])
    if kind == "rows":
        call = {"mxfp4": ops.mxfp4_gemv_rows, "f16": ops.f16_gemv_rows}[c["weights"]]
        return call(*s["w"], s["x"], c["out"])
    if kind == "gemm":
        call = {"mxfp4": ops.mxfp4_gemm, "int8": ops.i8_gemm}[c["weights"]]
        return call(s["x"], *s["w"], c["out"])
    if kind == "attend":
        return ops.attn_decode(s["q"], s["k"], s["v"], c["len"], s["ks"], s["vs"], c["out"], workspace=s["ws"])
    if kind == "prompt_attend":
        return ops.attn_prefill(s["q"], s["k"], s["v"], c["start"], c["out"])
    out, idx, w = ops.moe_layer(s["x"], s["logits"], c["top"], *s["experts"], gu_b=s["bias"][0], dn_b=s["bias"][1],
                                act=c["act"])
    return {"out": out, "idx": idx, "w": w}


# ---- the work that a pass cannot do without ----

def _weight_bytes(weights, n, k):
    return {"mxfp4": n * k * 17 // 32, "int8": n * k + 2 * n, "f16": 2 * n * k}[weights]


def _model_bytes_flops(tokens, behind, heads_run):
    c = MODEL
    weights = sum(math.prod(_model_shape(lin)) for lin in ("qkv", "o", "gate_up", "down")) * c["layers"]
    keys = sum(behind + t + 1 for t in range(tokens))
    head = c["vocab"] * c["hidden"]
    row = 2 * 2 * c["layers"] * c["kv_heads"] * 128
    flops = 2 * weights * tokens + 2 * head * heads_run + 4 * keys * c["heads"] * 128 * c["layers"]
    return weights * 17 // 32, 2 * head, row, keys, flops


def work(c):
    kind = c["kind"]
    if kind == "decode":
        n = c["steps"]
        weights, head, row, keys, flops = _model_bytes_flops(n, c["behind"], n)
        return {"bytes": n * (weights + head) + row * keys + 3 * n * row + 4 * MODEL["vocab"], "flops": flops}
    if kind == "prompt":
        n = c["tokens"]
        weights, head, row, _, flops = _model_bytes_flops(n, 0, 1)
        return {"bytes": weights + head + 3 * n * row + 4 * MODEL["vocab"], "flops": flops}
    if kind in ("gemv", "rows", "gemm"):
        t, n, k = c.get("m", c.get("tokens", 1)), c["n"], c["k"]
        size = {"f32": 4, "f16": 2, "swiglu": 1}[c["out"]]
        return {"bytes": _weight_bytes(c["weights"], n, k) + 2 * t * k + size * t * n, "flops": 2 * t * n * k}
    size = 2 if c.get("out") == "f16" else 4
    if kind == "attend":
        row = 2 * 128 * 2 if c["kv"] == "fp16" else 2 * (128 + 2)
        return {"bytes": c["len"] * c["kv_heads"] * row + c["heads"] * 128 * (2 + size),
                "flops": 4 * c["len"] * c["heads"] * 128}
    if kind == "prompt_attend":
        t, keys = c["tokens"], c["start"] + c["tokens"]
        seen = sum(c["start"] + i + 1 for i in range(t))
        return {"bytes": keys * c["kv_heads"] * 512 + t * c["heads"] * 128 * (2 + size),
                "flops": 4 * seen * c["heads"] * 128}
    t, E, H, I = c["tokens"], c["experts"], c["hidden"], c["inter"]
    chosen = E * (1 - (1 - c["top"] / E) ** t)  # the experts that t tokens choose, on the average
    expert = 3 * H * I * 17 // 32 + (4 * (2 * I + H) if c["act"] == "gptoss" else 0)
    return {"bytes": chosen * expert + t * (6 * H + 4 * E + 8 * c["top"]), "flops": 6 * t * c["top"] * H * I}


def tolerance(c):
    """About four times what is seen against exact(): 1.4e-3 after 28 layers that store fp16, 2.1e-4 for fp16
    results (their rounding), up to 3.5e-7 for fp32 sums."""
    if c["kind"] in ("decode", "prompt"):
        return {"rel": 6e-3}
    return {"rel": 8e-4 if c.get("out") in ("f16", "swiglu") else 2e-6}


# ---- the same in 64 bits, in plain torch ----

def _dequant(w, e):
    lut = torch.tensor(FP4, dtype=torch.float64, device=w.device)
    v = torch.stack((lut[(w & 15).long()], lut[(w >> 4).long()]), -1)
    v = v.view(*e.shape, 32) * torch.exp2(e.double() - 127)[..., None]
    return v.flatten(-2)


def _dense(c, w):
    if c["weights"] == "mxfp4":
        return _dequant(*w)
    return w[0].double() * w[1].double()[:, None] if c["weights"] == "int8" else w[0].double()


def _silu(x):
    return x * torch.sigmoid(x)


def _attend(q, k, v, start):
    """q (T, heads, 128) at positions start on over k, v (kv_heads, rows, 128): (T, heads, 128)."""
    T, heads, _ = q.shape
    G, keys = heads // k.shape[0], start + T
    out = torch.empty_like(q)
    for t0 in range(0, T, 1024):
        at = torch.arange(t0, min(T, t0 + 1024), device=q.device)
        hide = torch.arange(keys, device=q.device)[None, :] > start + at[:, None]
        for h in range(heads):
            s = (q[at, h] @ k[h // G, :keys].T) / math.sqrt(128)
            out[at, h] = torch.softmax(s.masked_fill(hide, -math.inf), -1) @ v[h // G, :keys]
    return out


def _norm(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _rope(x, pos):
    f = pos.double()[:, None] / THETA ** (torch.arange(0, 128, 2, device=x.device).double() / 128)
    cos, sin = f.cos()[:, None], f.sin()[:, None]
    a, b = x[..., :64], x[..., 64:]
    return torch.cat((a * cos - b * sin, b * cos + a * sin), -1)


def _forward(c, seed):
    """The decoder over all of the case's tokens: the last row's logits, and each position's K and V rows."""
    W = dict(_model_weights(seed))
    tokens = torch.tensor(_tokens(c, seed), device="cuda")
    T, heads, kvh = len(tokens), MODEL["heads"], MODEL["kv_heads"]
    pos = torch.arange(T, device="cuda")
    h = W["embed"][tokens].double()
    rows = {}
    for i in range(MODEL["layers"]):
        lin = lambda x, name: x @ _dequant(W[f"layers.{i}.{name}.blocks"], W[f"layers.{i}.{name}.scales"]).T  # noqa: E731
        nw = lambda name: W[f"layers.{i}.{name}"].double()  # noqa: E731
        x = lin(_norm(h, nw("input_norm")), "qkv").view(T, heads + 2 * kvh, 128)
        q = _rope(_norm(x[:, :heads], nw("q_norm")), pos)
        k = _rope(_norm(x[:, heads:heads + kvh], nw("k_norm")), pos)
        v = x[:, heads + kvh:]
        rows[f"kv_k_{i}_new"], rows[f"kv_v_{i}_new"] = k, v
        a = _attend(q, k.transpose(0, 1).contiguous(), v.transpose(0, 1).contiguous(), 0)
        h = h + lin(a.reshape(T, -1), "o")
        gu = lin(_norm(h, nw("post_norm")), "gate_up")
        h = h + lin(_silu(gu[:, 0::2]) * gu[:, 1::2], "down")
    last = _norm(h[-1:], W["norm"].double())
    logits = torch.cat([(part.double() @ last.T)[:, 0] for part in W["embed"].split(16384)])
    keep = slice(0, T) if c["kind"] == "prompt" else slice(c["behind"], T)
    packed = torch.stack([rows[name][keep].reshape(-1, kvh * 128) for name in sorted(rows)], 1)
    return {"logits": logits, "rows": packed.reshape(-1)}


def exact(c, seed):
    kind = c["kind"]
    if kind in ("decode", "prompt"):
        return _forward(c, seed)
    s = prepare(c, seed)
    if kind in ("gemv", "rows", "gemm"):
        y = s["x"].double() @ _dense(c, s["w"]).T
        return _silu(y[:, 0::2]) * y[:, 1::2] if c["out"] == "swiglu" else y
    if kind in ("attend", "prompt_attend"):
        k, v = s["k"].double(), s["v"].double()
        if kind == "prompt_attend":
            return _attend(s["q"].double(), k, v, c["start"])
        if s["ks"] is not None:
            k, v = k * s["ks"].double()[..., None], v * s["vs"].double()[..., None]
        return _attend(s["q"].double()[None], k, v, c["len"] - 1)[0]
    p = torch.softmax(s["logits"].double(), -1)
    w, idx = torch.sort(p, dim=-1, descending=True, stable=True)
    w, idx = w[:, :c["top"]], idx[:, :c["top"]]
    w = w / (w.sum(-1, keepdim=True) + 1e-6)
    gu, gs, dn, ds = s["experts"]
    out = torch.zeros(c["tokens"], c["hidden"], dtype=torch.float64, device="cuda")
    for t in range(c["tokens"]):
        for j in range(c["top"]):
            e = int(idx[t, j])
            y = _dequant(gu[e].flatten(1), gs[e]) @ s["x"][t].double()
            if c["act"] == "gptoss":
                y = y + s["bias"][0][e].double()
                g, u = y[0::2].clamp(max=7.0), y[1::2].clamp(-7.0, 7.0)
                a = g * torch.sigmoid(1.702 * g) * (u + 1)
            else:
                a = _silu(y[0::2]) * y[1::2]
            y = _dequant(dn[e].flatten(1), ds[e]) @ a
            if c["act"] == "gptoss":
                y = y + s["bias"][1][e].double()
            out[t] += w[t, j] * y
    return {"out": out, "idx": idx, "w": w}
