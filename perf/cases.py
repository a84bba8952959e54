"""The calls of this framework that a user's program spends its time in, as measurable cases.

Every case goes through the package's public entry points (`rust_ascend_hip.nn`, `HipRuntime`,
`DecoderLayer`) in async mode, as a training or serving loop runs them: work is queued on torch's
current stream and nothing waits inside a pass. Shapes are the decoder layer's (hidden 4096, 32
query and 8 KV heads of 128, SwiGLU 14336, vocabulary 32000) and generic smaller, larger and ragged
ones around them. Training cases return every gradient.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rust-ascend_amd"))

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32, "f16": torch.float16}


def listed():
    return [
        # one token of a batched generation loop: a new query per sequence against its KV cache
        {"name": "decode_attention", "kind": "decode_attention", "batch": 8, "q_heads": 32, "kv_heads": 8, "dim": 128,
         "queries": 1, "keys": 4096},
        # training or prefill of BF16 causal grouped-query attention, a length off every tile edge
        {"name": "causal_attention", "kind": "causal_attention", "batch": 2, "q_heads": 32, "kv_heads": 8, "dim": 128,
         "seq": 1900, "dtype": "bf16"},
        # the FP32 surface with an additive mask (relative-position bias, padded keys), trained
        {"name": "masked_attention", "kind": "masked_attention", "batch": 2, "q_heads": 16, "kv_heads": 8, "dim": 64,
         "value_dim": 64, "queries": 1040, "keys": 1056, "mask_grad": False},
        # the down projection of the same generation loop: 16 tokens against the whole weight
        {"name": "decode_linear", "kind": "decode_linear", "tokens": 16, "inputs": 14336, "outputs": 4096},
        # a trained FP32 Linear computed in BF16, mid-size
        {"name": "linear_f32", "kind": "linear_f32", "tokens": 2000, "inputs": 4096, "outputs": 4096},
        # the same for shapes with no alignment at all (a classifier head, a ragged batch)
        {"name": "padded_linear_f32", "kind": "padded_linear_f32", "tokens": 1777, "inputs": 2001, "outputs": 3003},
        # a trained FP32 SwiGLU feed-forward block of a small model
        {"name": "swiglu_f32", "kind": "swiglu_f32", "tokens": 2000, "inputs": 2048, "hidden": 5632},
        # the generic float matmul: [batch, tokens, k] by one [k, n] weight, in the inputs' own dtype
        {"name": "float_matmul", "kind": "float_matmul", "batch": 4, "shared": True, "m": 1000, "k": 1024, "n": 1000,
         "dtype": "f32"},
        # a pre-norm of a trained layer, a width and row count away from the benchmark's
        {"name": "rms_norm", "kind": "rms_norm", "rows": 12001, "width": 5120, "dtype": "bf16"},
        # the language-model loss: FP32 logits over the vocabulary, with its gradient
        {"name": "cross_entropy", "kind": "cross_entropy", "rows": 4096, "classes": 32000},
        # one small decoder layer, forward and backward: few tokens, so launches and tile counts decide
        {"name": "decoder_layer_small", "kind": "decoder_layer", "hidden": 2048, "heads": 16, "kv_heads": 4,
         "ffn": 5632, "vocab": 32000, "batch": 1, "seq": 512},
        # the flagship layer: 2 x 2048 tokens, hidden 4096, forward and backward
        {"name": "decoder_layer", "kind": "decoder_layer", "hidden": 4096, "heads": 32, "kv_heads": 8, "ffn": 14336,
         "vocab": 32000, "batch": 2, "seq": 2048},
    ]


def _log(rng, lo, hi, step=1):
    """A whole number in [lo, hi], a multiple of step, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    kind = rng.choice(["decode_attention", "causal_attention", "masked_attention", "decode_linear", "linear_f32",
                       "padded_linear_f32", "swiglu_f32", "float_matmul", "rms_norm", "cross_entropy",
                       "decoder_layer"])
    c = {"kind": kind}
    if kind == "decode_attention":
        batch = _log(rng, 1, 32)
        kv = rng.choice([4, 8])
        c.update(batch=batch, q_heads=kv * rng.choice([1, 4, 8]), kv_heads=kv, dim=rng.choice([64, 128, 128]),
                 queries=rng.choice([1, 1, 1, 2, 4]), keys=_log(rng, 200, min(16384, 131072 // batch)))
    elif kind == "causal_attention":
        kv = rng.choice([2, 4, 8])
        batch = rng.choice([1, 2, 4])
        c.update(batch=batch, q_heads=kv * rng.choice([1, 4]), kv_heads=kv, dim=rng.choice([64, 128, 128]),
                 seq=_log(rng, 128, 4096 // batch), dtype=rng.choice(["bf16", "bf16", "f32"]))
    elif kind == "masked_attention":
        kv = rng.choice([2, 4, 8])
        c.update(batch=rng.choice([1, 2]), q_heads=kv * rng.choice([1, 2, 4]), kv_heads=kv,
                 dim=rng.choice([64, 80, 96, 128]), value_dim=rng.choice([64, 96, 128]),
                 queries=_log(rng, 128, 1536, 16), keys=_log(rng, 128, 1536, 32), mask_grad=rng.random() < 0.25)
    elif kind == "decode_linear":
        c.update(tokens=_log(rng, 16, 128, 16), inputs=_log(rng, 1024, 14336, 16), outputs=_log(rng, 1024, 14336, 16))
    elif kind == "linear_f32":
        c.update(tokens=_log(rng, 64, 4096, 16), inputs=_log(rng, 512, 4096, 16), outputs=_log(rng, 512, 4096, 16))
    elif kind == "padded_linear_f32":
        c.update(tokens=_log(rng, 100, 4100), inputs=_log(rng, 300, 4100), outputs=_log(rng, 300, 4100))
    elif kind == "swiglu_f32":
        c.update(tokens=_log(rng, 128, 4096, 16), inputs=_log(rng, 512, 2048, 16), hidden=_log(rng, 1024, 5632, 16))
    elif kind == "float_matmul":
        c.update(batch=_log(rng, 1, 16), shared=rng.random() < 0.5, m=_log(rng, 100, 1000), k=_log(rng, 64, 1100),
                 n=_log(rng, 64, 1100), dtype=rng.choice(["f32", "f32", "f16", "bf16"]))
    elif kind == "rms_norm":
        width = _log(rng, 500, 8192)
        width = width if rng.random() < 0.25 else width // 64 * 64  # most widths are whole multiples
        c.update(rows=_log(rng, 16, (64 << 20) // width), width=width, dtype=rng.choice(["bf16", "bf16", "f32"]))
    elif kind == "cross_entropy":
        classes = _log(rng, 1000, 50000)
        c.update(rows=_log(rng, 64, (128 << 20) // classes), classes=classes)
    else:
        hidden = rng.choice([1024, 2048, 4096])
        heads = hidden // 128
        c.update(hidden=hidden, heads=heads, kv_heads=heads // rng.choice([1, 4]),
                 ffn=_log(rng, 2 * hidden, 7 * hidden // 2, 128), vocab=32000, batch=rng.choice([1, 2]),
                 seq=_log(rng, 128, 2048, 16))
    return c


# ---------------------------------------------------------------- inputs

def _randn(g, shape, dtype, scale=1.0):
    return (torch.randn(shape, generator=g, device=DEV) * scale).to(dtype)


def _inputs(c, seed):
    """What the call takes, from the seed alone."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    bf, f32 = torch.bfloat16, torch.float32
    kind = c["kind"]
    s = {}
    if kind == "decode_attention":
        b, hq, hkv, d, m, n = (c[k] for k in ("batch", "q_heads", "kv_heads", "dim", "queries", "keys"))
        s["q"], s["k"], s["v"] = (_randn(g, (b, h, r, d), bf) for h, r in ((hq, m), (hkv, n), (hkv, n)))
    elif kind == "causal_attention":
        b, hq, hkv, d, n = (c[k] for k in ("batch", "q_heads", "kv_heads", "dim", "seq"))
        dt = DTYPES[c["dtype"]]
        s["q"], s["k"], s["v"], s["dy"] = (_randn(g, (b, h, n, d), dt) for h in (hq, hkv, hkv, hq))
    elif kind == "masked_attention":
        b, hq, hkv, d, dv, m, n = (c[k] for k in ("batch", "q_heads", "kv_heads", "dim", "value_dim", "queries",
                                                  "keys"))
        s["q"], s["k"] = _randn(g, (b, hq, m, d), f32), _randn(g, (b, hkv, n, d), f32)
        s["v"], s["dy"] = _randn(g, (b, hkv, n, dv), f32), _randn(g, (b, hq, m, dv), f32)
        slope = torch.rand((1, hq, 1, 1), generator=g, device=DEV) * 0.05
        far = (torch.arange(m, device=DEV)[:, None] - torch.arange(n, device=DEV)[None, :]).abs().float()
        mask = (-slope * far).expand(b, hq, m, n).clone()
        mask[b - 1, :, :, n - n // 8:] = float("-inf")  # the last sequence is shorter
        s["mask"] = mask
    elif kind == "decode_linear":
        s["x"] = _randn(g, (c["tokens"], c["inputs"]), bf)
        s["w"] = _randn(g, (c["outputs"], c["inputs"]), bf, 0.02)
    elif kind in ("linear_f32", "padded_linear_f32"):
        s["x"] = _randn(g, (c["tokens"], c["inputs"]), f32)
        s["w"] = _randn(g, (c["outputs"], c["inputs"]), f32, 0.02)
        s["dy"] = _randn(g, (c["tokens"], c["outputs"]), f32)
    elif kind == "swiglu_f32":
        t, k, h = c["tokens"], c["inputs"], c["hidden"]
        s["x"], s["dy"] = _randn(g, (t, k), f32), _randn(g, (t, k), f32)
        s["gate"], s["up"], s["down"] = (_randn(g, sh, f32, 0.03) for sh in ((h, k), (h, k), (k, h)))
    elif kind == "float_matmul":
        dt, b, m, k, n = DTYPES[c["dtype"]], c["batch"], c["m"], c["k"], c["n"]
        s["a"] = _randn(g, (b, m, k), dt)
        s["b"] = _randn(g, (k, n) if c["shared"] else (b, k, n), dt, k ** -0.5)
        s["dy"] = _randn(g, (b, m, n), dt)
    elif kind == "rms_norm":
        dt = DTYPES[c["dtype"]]
        s["x"], s["dy"] = _randn(g, (c["rows"], c["width"]), dt), _randn(g, (c["rows"], c["width"]), dt)
        s["w"] = 1 + _randn(g, (c["width"],), f32, 0.1)
    elif kind == "cross_entropy":
        s["x"] = _randn(g, (c["rows"], c["classes"]), f32, 2.0)
        s["target"] = torch.randint(0, c["classes"], (c["rows"],), generator=g, device=DEV)
    else:
        h, f = c["hidden"], c["ffn"]
        w = (c["heads"] + 2 * c["kv_heads"]) * (h // c["heads"])
        for name, shape in (("table", (c["vocab"], h)), ("wqkv", (w, h)), ("wo", (h, h)), ("wg", (f, h)),
                            ("wu", (f, h)), ("wd", (h, f))):
            s[name] = _randn(g, shape, bf, 1.0 if name == "table" else 0.02)
        s["w1"], s["w2"] = 1 + _randn(g, (h,), f32, 0.1), 1 + _randn(g, (h,), f32, 0.1)
        s["ids"] = torch.randint(0, c["vocab"], (c["batch"], c["seq"]), generator=g, device=DEV)
        s["dy"] = _randn(g, (c["batch"], c["seq"], h), bf)
    return s


_GRADS = {"causal_attention": ("q", "k", "v"), "masked_attention": ("q", "k", "v"), "linear_f32": ("x", "w"),
          "padded_linear_f32": ("x", "w"), "swiglu_f32": ("x", "gate", "up", "down"), "float_matmul": ("a", "b"),
          "rms_norm": ("x", "w"), "cross_entropy": ("x",)}


def _wanted(c):
    return _GRADS.get(c["kind"], ()) + (("mask",) if c.get("mask_grad") else ())


def prepare(case, seed):
    import rust_ascend_hip as hk
    from rust_ascend_hip import nn
    from rust_ascend_hip.decoder import DecoderConfig, DecoderLayer

    hk.HipRuntime.set_async(True)
    c, s = case, _inputs(case, seed)
    kind = c["kind"]
    if kind == "decoder_layer":
        layer = DecoderLayer(DecoderConfig(hidden=c["hidden"], heads=c["heads"], kv_heads=c["kv_heads"], ffn=c["ffn"],
                                           vocab=c["vocab"], batch=c["batch"], seq=c["seq"]), device=DEV)
        for name in ("table", "wqkv", "wo", "wd", "w1", "w2"):
            getattr(layer, name).copy_(s[name])
        f, h = c["ffn"], c["hidden"]
        layer.w_gu.copy_(torch.stack([s["wg"].view(f // 16, 16, h), s["wu"].view(f // 16, 16, h)], 1).view(2 * f, h))
        ids, dy = s["ids"], s["dy"]

        def call():
            y = layer.forward(ids)
            return y, layer.backward(dy)
        return call
    for name in _wanted(c):
        s[name].requires_grad_(True)
    wanted = [s[name] for name in _wanted(c)]
    scale = c["dim"] ** -0.5 if "dim" in c else 0.0
    if kind == "decode_attention":
        start = c["keys"] - c["queries"]  # the queries are the newest positions of the cache
        return lambda: nn.causal_grouped_query_attention_bf16(s["q"], s["k"], s["v"], scale, start)
    if kind == "decode_linear":
        return lambda: hk.HipRuntime.gemm(s["x"], s["w"], hk.Transpose.No, hk.Transpose.Yes, torch.bfloat16)
    if kind == "cross_entropy":
        def call():
            loss = nn.cross_entropy(s["x"], s["target"])
            return loss.detach(), torch.autograd.grad(loss, wanted)
        return call
    if kind == "causal_attention":
        fn = nn.causal_grouped_query_attention_bf16 if c["dtype"] == "bf16" else \
            nn.causal_grouped_query_attention_bf16_fp32
        forward = lambda: fn(s["q"], s["k"], s["v"], scale)  # noqa: E731
    elif kind == "masked_attention":
        forward = lambda: nn.grouped_query_attention_bf16_fp32(s["q"], s["k"], s["v"], scale, s["mask"])  # noqa: E731
    elif kind == "linear_f32":
        forward = lambda: nn.linear_bf16_fp32(s["x"], s["w"])  # noqa: E731
    elif kind == "padded_linear_f32":
        forward = lambda: nn.linear_padded_bf16_fp32(s["x"], s["w"])  # noqa: E731
    elif kind == "swiglu_f32":
        forward = lambda: nn.swiglu_bf16_fp32(s["x"], s["gate"], s["up"], s["down"])  # noqa: E731
    elif kind == "float_matmul":
        forward = lambda: nn.float_matmul(s["a"], s["b"])  # noqa: E731
    else:
        forward = lambda: nn.rms_norm(s["x"], s["w"], 1e-6)  # noqa: E731

    def train():
        y = forward()
        return y.detach(), torch.autograd.grad(y, wanted, s["dy"])
    return train


def run(state):
    return state()


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    c = case
    kind = c["kind"]
    if kind == "decode_attention":
        b, hq, hkv, d, m, n = (c[k] for k in ("batch", "q_heads", "kv_heads", "dim", "queries", "keys"))
        return {"bytes": 2 * (2 * b * hkv * n * d + 2 * b * hq * m * d), "flops": 4 * b * hq * m * n * d}
    if kind == "causal_attention":
        b, hq, hkv, d, n = (c[k] for k in ("batch", "q_heads", "kv_heads", "dim", "seq"))
        e = 2 if c["dtype"] == "bf16" else 4
        return {"bytes": e * b * n * d * (4 * hq + 4 * hkv), "flops": 7 * b * hq * n * n * d}  # 3.5 x 4/2 (causal)
    if kind == "masked_attention":
        b, hq, hkv, d, dv, m, n = (c[k] for k in ("batch", "q_heads", "kv_heads", "dim", "value_dim", "queries",
                                                  "keys"))
        scores = b * hq * m * n
        size = 4 * b * (hq * m * (2 * d + 2 * dv) + hkv * n * (2 * d + 2 * dv))
        return {"bytes": size + 4 * scores * (2 if c["mask_grad"] else 1), "flops": 2 * scores * (4 * d + 3 * dv)}
    if kind == "decode_linear":
        t, i, o = c["tokens"], c["inputs"], c["outputs"]
        return {"bytes": 2 * (t * i + o * i + t * o), "flops": 2 * t * i * o}
    if kind in ("linear_f32", "padded_linear_f32"):
        t, i, o = c["tokens"], c["inputs"], c["outputs"]
        return {"bytes": 8 * (t * i + o * i + t * o), "flops": 6 * t * i * o}
    if kind == "swiglu_f32":
        t, k, h = c["tokens"], c["inputs"], c["hidden"]
        return {"bytes": 4 * (4 * t * k + 6 * k * h), "flops": 18 * t * k * h}
    if kind == "float_matmul":
        b, m, k, n = c["batch"], c["m"], c["k"], c["n"]
        e = 4 if c["dtype"] == "f32" else 2
        return {"bytes": 2 * e * (b * m * k + (1 if c["shared"] else b) * k * n + b * m * n), "flops": 6 * b * m * n * k}
    if kind == "rms_norm":
        e = 2 if c["dtype"] == "bf16" else 4
        return {"bytes": 4 * e * c["rows"] * c["width"], "flops": 10 * c["rows"] * c["width"]}
    if kind == "cross_entropy":
        return {"bytes": 8 * c["rows"] * c["classes"], "flops": 6 * c["rows"] * c["classes"]}
    t, h, f, d = c["batch"] * c["seq"], c["hidden"], c["ffn"], c["hidden"] // c["heads"]
    params = h * (c["heads"] + 2 * c["kv_heads"]) * d + h * h + 3 * h * f
    attention = 7 * c["batch"] * c["heads"] * c["seq"] * c["seq"] * d
    # weights read in BF16 and their gradients written in F32; the table's gradient is dense BF16
    return {"bytes": 6 * params + 2 * c["vocab"] * h + 2 * 4 * t * h, "flops": 6 * t * params + attention}


def tolerance(case):
    """About four times the error against 64 bits that the calls show (given in brackets)."""
    c = case
    kind = c["kind"]
    if kind == "float_matmul":
        return {"rel": {"f32": 4e-6, "f16": 2e-3, "bf16": 1e-2}[c["dtype"]]}  # [5.7e-7 in F32]
    if kind == "rms_norm":
        return {"rel": {"f32": 1e-6, "bf16": 1e-2}[c["dtype"]]}  # [1.7e-3 in BF16, 2.3e-7 in F32]
    if kind in ("linear_f32", "padded_linear_f32"):
        return {"rel": 4e-6}  # BF16 operands by contract, 32-bit sums [4e-7, growing with the contraction]
    if kind == "swiglu_f32":
        return {"rel": 3e-4}  # a 32-bit sum's last bit decides a BF16 rounding of the next operand [5e-5]
    if kind == "cross_entropy":
        return {"rel": 1e-6}  # [4.6e-8; the exponential and the logarithm are good to a few ulp]
    if kind == "decoder_layer":
        return {"rel": 4e-2}  # a chain of BF16 operations, each rounding what the next one reads [9.3e-3]
    return {"rel": 1e-2}  # BF16 operands and results [2.5e-3]


# ---------------------------------------------------------------- the same in 64 bits

def _bf(t):
    """Rounded to BF16 as the entry point's contract rounds its GEMM operands, then 64-bit."""
    return t.to(torch.bfloat16).double()


def _mm(a, b):
    return torch.matmul(a, b.contiguous())


def _attention(q, k, v, dy, scale, mask, mask_grad=False):
    """(o, dq, dk, dv[, dmask]) in 64 bits, one (batch, KV head) at a time; mask(b, kv head) is additive."""
    b, hq, m, d = q.shape
    hkv, n = k.shape[1], k.shape[2]
    grp = hq // hkv
    outs = [[], [], [], [], []]
    for i in range(b):
        for h in range(hkv):
            qs = q[i, h * grp:(h + 1) * grp].reshape(grp * m, d)
            kk, vv = k[i, h], v[i, h]
            sc = _mm(qs, kk.t()) * scale + mask(i, h)
            p = torch.softmax(sc, -1)
            outs[0].append(_mm(p, vv).view(grp, m, -1))
            if dy is None:
                continue
            do = dy[i, h * grp:(h + 1) * grp].reshape(grp * m, -1)
            dp = _mm(do, vv.t())
            ds = p * (dp - (p * dp).sum(-1, keepdim=True))
            outs[1].append((_mm(ds, kk) * scale).view(grp, m, d))
            outs[2].append(_mm(ds.t().contiguous(), qs) * scale)
            outs[3].append(_mm(p.t().contiguous(), do))
            if mask_grad:
                outs[4].append(ds.view(grp, m, n))
    o = torch.cat(outs[0]).view(b, hq, m, -1)
    if dy is None:
        return o
    grads = [torch.cat(outs[1]).view(b, hq, m, d), torch.stack(outs[2]).view(b, hkv, n, d),
             torch.stack(outs[3]).view(b, hkv, n, -1)]
    if mask_grad:
        grads.append(torch.cat(outs[4]).view(b, hq, m, n))
    return o, tuple(grads)


def _causal(grp, m, n, start):
    ok = torch.arange(n, device=DEV)[None, :] <= start + torch.arange(m, device=DEV)[:, None]
    z = torch.zeros((m, n), device=DEV, dtype=torch.float64).masked_fill_(~ok, float("-inf"))
    return z.repeat(grp, 1)


def _rms(x, w, eps, dy=None):
    rstd = (x.square().mean(-1, keepdim=True) + eps).rsqrt()
    return x * rstd * w, rstd


def _exact_layer(c, s):
    d = c["hidden"] // c["heads"]
    half = d // 2
    p = {k: s[k].double().requires_grad_(True) for k in ("table", "wqkv", "wo", "wg", "wu", "wd", "w1", "w2")}
    inv = 5e5 ** (-torch.arange(0, d, 2, device=DEV, dtype=torch.float64) / d)
    ang = torch.arange(c["seq"], device=DEV, dtype=torch.float64)[:, None] * inv
    cos, sin = ang.cos(), ang.sin()

    def rope(x):
        a, b = x[..., :half], x[..., half:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

    B, S, hq, hkv = c["batch"], c["seq"], c["heads"], c["kv_heads"]
    x0 = p["table"][s["ids"]]
    n1 = _rms(x0, p["w1"], 1e-5)[0]
    qkv = (n1 @ p["wqkv"].t()).view(B, S, hq + 2 * hkv, d).transpose(1, 2)
    q, k, v = rope(qkv[:, :hq]), rope(qkv[:, hq:hq + hkv]), qkv[:, hq + hkv:]
    keep = torch.ones((S, S), device=DEV, dtype=torch.bool).tril()
    heads = []
    for b in range(B):
        for h in range(hq):
            kv = h // (hq // hkv)
            sc = (q[b, h] @ k[b, kv].t() * d ** -0.5).masked_fill(~keep, float("-inf"))
            heads.append(torch.softmax(sc, -1) @ v[b, kv])
    o = torch.stack(heads).view(B, hq, S, d).transpose(1, 2).reshape(B, S, hq * d)
    h1 = x0 + o @ p["wo"].t()
    n2 = _rms(h1, p["w2"], 1e-5)[0]
    y = h1 + (torch.nn.functional.silu(n2 @ p["wg"].t()) * (n2 @ p["wu"].t())) @ p["wd"].t()
    names = list(p)
    grads = torch.autograd.grad(y, [p[n] for n in names], s["dy"].double())
    return y.detach(), dict(zip(names, grads))


def exact(case, seed):
    c, s = case, _inputs(case, seed)
    kind = c["kind"]
    D = {k: (v.double() if v.is_floating_point() else v) for k, v in s.items()} if kind != "decoder_layer" else {}
    scale = c["dim"] ** -0.5 if "dim" in c else 0.0
    grp = c["q_heads"] // c["kv_heads"] if "q_heads" in c else 1
    if kind == "decode_attention":
        mask = _causal(grp, c["queries"], c["keys"], c["keys"] - c["queries"])
        return _attention(D["q"], D["k"], D["v"], None, scale, lambda b, h: mask)
    if kind == "causal_attention":
        mask = _causal(grp, c["seq"], c["seq"], 0)
        return _attention(*(_bf(s[k]) for k in ("q", "k", "v", "dy")), scale, lambda b, h: mask)
    if kind == "masked_attention":
        mask = D["mask"].view(c["batch"], c["kv_heads"], grp * c["queries"], c["keys"])
        return _attention(*(_bf(s[k]) for k in ("q", "k", "v", "dy")), scale, lambda b, h: mask[b, h], c["mask_grad"])
    if kind == "decode_linear":
        return _mm(D["x"], D["w"].t())
    if kind in ("linear_f32", "padded_linear_f32"):
        x, w, dy = _bf(s["x"]), _bf(s["w"]), _bf(s["dy"])
        return _mm(x, w.t()), (_mm(dy, w), _mm(dy.t().contiguous(), x))
    if kind == "swiglu_f32":
        x, wg, wu, wd, dy = (_bf(s[k]) for k in ("x", "gate", "up", "down", "dy"))
        g, u = _mm(x, wg.t()), _mm(x, wu.t())
        sg = torch.sigmoid(g)
        act = _bf((g * sg * u).float())
        dm = _mm(dy, wd)
        dg, du = _bf((dm * u * sg * (1 + g * (1 - sg))).float()), _bf((dm * g * sg).float())
        dx = _mm(dg, wg) + _mm(du, wu)
        return _mm(act, wd.t()), (dx, _mm(dg.t().contiguous(), x), _mm(du.t().contiguous(), x),
                                  _mm(dy.t().contiguous(), act))
    if kind == "float_matmul":
        a, b, dy = D["a"], D["b"], D["dy"]
        if c["shared"]:
            da = _mm(dy, b.t())
            db = _mm(a.reshape(-1, c["k"]).t().contiguous(), dy.reshape(-1, c["n"]))
        else:
            da = _mm(dy, b.transpose(1, 2))
            db = _mm(a.transpose(1, 2).contiguous(), dy)
        return _mm(a, b), (da, db)
    if kind == "rms_norm":
        x, w, dy = D["x"], D["w"], D["dy"]
        y, rstd = _rms(x, w, 1e-6)
        g = dy * w
        dx = rstd * (g - x * rstd.square() * (g * x).mean(-1, keepdim=True))
        return y, (dx, (dy * x * rstd).sum(0))
    if kind == "cross_entropy":
        rows = c["rows"]
        x, t = D["x"], s["target"]
        lse = torch.logsumexp(x, -1)
        loss = (lse - x.gather(1, t[:, None])[:, 0]).mean().view(1)
        dx = torch.exp(x - lse[:, None])
        dx[torch.arange(rows, device=DEV), t] -= 1
        return loss, (dx / rows,)
    return _exact_layer(c, s)
