"""Performance cases: the work a program has this library do, through the
public entry points of the Python package, over the ranges it is used in.

Every case is one call (or one forward + backward pair) of a layer:

  linear      Linear::forward, y = x W^T + b, from one decode row to a prefill
  train       one layer's training step: C = A B, then both matmul gradients
  bmm         Tensor::matmul over batches (attention scores, per-head products)
  swiglu_f32  the LLaMA / Mistral feed-forward block in fp32
  swiglu_i8   the same block on int8 weights (QuantizedSwiGLU)
  qlinear     one int8 linear on fp32 activations (DynamicQuantization)
  gemv_w8     weight-only int8 decode product, x [B, K] times W [K, N]
  sdpa        scaled dot product attention on [B, H, S, D]
  mha         MultiHeadAttention::forward_with_cache on a whole sequence, the
              attention weights and new keys / values returned as the
              reference's signature has them
  mha_step    one generation step over an in-place key / value cache
  flash       FlashAttention::forward, the blockwise recurrence layer

`listed()` names one or two members of each, `draw()` gives others from the
same ranges.  Inputs are made on the GPU from the seed alone.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "ghost-flow_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import ghostflow_hip as gh  # noqa: E402


def listed():
    return [
        # a single token through a small square layer: launch latency and the
        # host path, nothing else
        {"name": "linear_m1_768", "kind": "linear", "m": 1, "k": 768, "n": 768, "bias": True},
        # a 4096-token prefill through a 4096-wide projection
        {"name": "linear_m4096_4096", "kind": "linear", "m": 4096, "k": 4096, "n": 4096, "bias": True},
        # a training step of an MLP layer on flattened 28 x 28 images, batch
        # 1000: no dimension is a multiple of a tile
        {"name": "train_m1000_k784_n1500", "kind": "train", "m": 1000, "k": 784, "n": 1500},
        # attention scores of 8 x 12 heads, head dimension 64, ragged length
        {"name": "bmm_b96_m500_k64", "kind": "bmm", "b": 96, "m": 500, "k": 64, "n": 500},
        # feed-forward block: 16 sequences decoding together in fp32
        {"name": "swiglu_f32_m16", "kind": "swiglu_f32", "m": 16, "hidden": 4096, "inter": 11008},
        # the same block on int8 weights, a 512-token prefill
        {"name": "swiglu_i8_m512", "kind": "swiglu_i8", "m": 512, "hidden": 4096, "inter": 11008},
        # int8 linear on a 100-token prompt
        {"name": "qlinear_m100", "kind": "qlinear", "m": 100, "k": 4096, "n": 11008, "bias": True},
        # weight-only int8 decoding of 4 sequences
        {"name": "gemv_w8_b4", "kind": "gemv_w8", "b": 4, "k": 4096, "n": 14336},
        # causal attention over prompts of 1000 tokens
        {"name": "sdpa_s1000_d128", "kind": "sdpa", "b": 4, "h": 32, "s": 1000, "d": 128, "causal": True},
        # an attention layer on whole sequences, the reference's own call
        # with a lower-triangular mask tensor and the weights returned
        {"name": "mha_b4_s512_e1024", "kind": "mha", "b": 4, "s": 512, "e": 1024, "h": 16, "mask": True},
        # one decode step of 4 sequences over 2047 cached positions
        {"name": "mha_step_b4_e4096", "kind": "mha_step", "b": 4, "s": 1, "e": 4096, "h": 32, "past": 2047},
        # FlashAttention::forward with its default blocks, causal
        {"name": "flash_b64_s1024_d64", "kind": "flash", "b": 64, "s": 1024, "d": 64, "block": 64, "causal": True},
    ]


# ---- drawing more cases of the same ranges ------------------------------------


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: mostly multiples of 64, some of 4, some of nothing."""
    v = _log(rng, lo, hi)
    step = rng.choice((64, 64, 4, 1))
    return min(hi, max(lo, v // step * step))


def _seconds(c):
    """A rough time of one pass, to keep drawn cases below the largest listed."""
    w = work(c)
    rate = {"swiglu_i8": 1.2e15, "qlinear": 1.2e15, "gemv_w8": 2e14, "linear": 1.2e14, "swiglu_f32": 1.2e14,
            "train": 1e14, "bmm": 8e13}.get(c["kind"], 6e13)
    return max(w["flops"] / rate, w["bytes"] / 3e12)


def draw(rng):
    most = 2.0 * 4096 ** 3 / 1.5e14
    while True:
        c = _draw(rng)
        if _seconds(c) <= 0.8 * most:
            return c


def _draw(rng):
    kind = rng.choice(("linear", "train", "bmm", "swiglu_f32", "swiglu_i8", "qlinear", "gemv_w8", "sdpa", "mha",
                       "mha_step", "flash"))
    c = {"kind": kind}
    if kind == "linear":
        c.update(m=_log(rng, 1, 4096), k=_width(rng, 256, 8192), n=_width(rng, 256, 14336), bias=rng.random() < 0.8)
    elif kind == "train":
        c.update(m=_log(rng, 64, 4096), k=_width(rng, 64, 4096), n=_width(rng, 64, 4096))
    elif kind == "bmm":
        c.update(b=_log(rng, 8, 128), m=_log(rng, 32, 1024), k=_width(rng, 32, 512), n=_width(rng, 32, 1024))
    elif kind in ("swiglu_f32", "swiglu_i8"):
        c.update(m=_log(rng, 1, 1024 if kind == "swiglu_f32" else 2048), hidden=_log(rng, 32, 256) * 16,
                 inter=_log(rng, 64, 896) * 16)
    elif kind == "qlinear":
        c.update(m=_log(rng, 1, 2048), k=_log(rng, 16, 512) * 16, n=_width(rng, 256, 14336), bias=rng.random() < 0.5)
    elif kind == "gemv_w8":
        c.update(b=_log(rng, 1, 16), k=_width(rng, 512, 8192), n=_log(rng, 8, 256) * 64)
    elif kind == "sdpa":
        c.update(b=_log(rng, 1, 8), h=_log(rng, 4, 32), s=_log(rng, 32, 2048), d=rng.choice((32, 64, 80, 96, 128)),
                 causal=rng.random() < 0.7)
    elif kind == "mha":
        d = rng.choice((64, 64, 80, 128))
        h = _log(rng, 4, 16)
        c.update(b=_log(rng, 1, 8), s=_log(rng, 32, 1024), e=h * d, h=h, mask=rng.random() < 0.6)
    elif kind == "mha_step":
        d = rng.choice((64, 64, 128))
        h = _log(rng, 4, 32)
        s = 1 if rng.random() < 0.6 else _log(rng, 2, 64)
        c.update(b=_log(rng, 1, 16), s=s, e=h * d, h=h, past=_log(rng, 16, 4096))
    else:
        c.update(b=_log(rng, 4, 128), s=_log(rng, 64, 2048), d=rng.choice((32, 64, 64, 128)),
                 block=rng.choice((64, 64, 128)), causal=rng.random() < 0.6)
    return c


# ---- what a program has in hand -------------------------------------------------


class _Make:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, device="cuda", generator=self.g) * std

    def uniform(self, *shape, bound):
        return (torch.rand(shape, device="cuda", generator=self.g) * 2 - 1) * bound

    def layer(self, n_in, n_out):
        """Weight [out, in] and bias with Linear::new's distributions."""
        return self.uniform(n_out, n_in, bound=math.sqrt(6.0 / n_in)), self.uniform(n_out, bound=1 / math.sqrt(n_in))


def _inputs(c, seed):
    """The tensors of a case, by name, from the seed alone."""
    r, k = _Make(seed), c["kind"]
    if k == "linear":
        w, b = r.layer(c["k"], c["n"])
        return {"x": r.normal(c["m"], c["k"]), "w": w, "b": b if c["bias"] else None}
    if k == "train":
        # activations, a weight [in, out], and the loss gradient of the output
        return {"a": r.normal(c["m"], c["k"]), "b": r.normal(c["k"], c["n"], std=0.02),
                "grad": r.normal(c["m"], c["n"], std=1.0 / c["m"])}
    if k == "bmm":
        return {"a": r.normal(c["b"], c["m"], c["k"]), "b": r.normal(c["b"], c["k"], c["n"])}
    if k in ("swiglu_f32", "swiglu_i8"):
        gate, up, down = r.layer(c["hidden"], c["inter"]), r.layer(c["hidden"], c["inter"]), r.layer(c["inter"], c["hidden"])
        return {"x": r.normal(c["m"], c["hidden"]), "gate": gate, "up": up, "down": down}
    if k == "qlinear":
        return {"x": r.normal(c["m"], c["k"]), "w": r.normal(c["n"], c["k"], std=0.02),
                "b": r.uniform(c["n"], bound=1 / math.sqrt(c["k"])) if c["bias"] else None}
    if k == "gemv_w8":
        return {"x": r.normal(c["b"], c["k"]), "w": r.normal(c["k"], c["n"], std=0.02)}
    if k == "sdpa":
        return {n: r.normal(c["b"], c["h"], c["s"], c["d"]) for n in "qkv"}
    if k in ("mha", "mha_step"):
        t = {"x": r.normal(c["b"], c["s"], c["e"]), "p": [v for _ in range(4) for v in r.layer(c["e"], c["e"])]}
        if k == "mha_step":
            # cached projections: what the layer itself gives for N(0, 1) inputs
            t["pk"], t["pv"] = (r.normal(c["b"], c["past"], c["e"], std=math.sqrt(2.0)) for _ in range(2))
        elif c["mask"]:
            t["mask"] = torch.ones(c["s"], c["s"], device="cuda").tril()
        return t
    return {n: r.normal(c["b"], c["s"], c["d"]) for n in "qkv"}


def prepare(case, seed):
    c, t = case, _inputs(case, seed)
    k = c["kind"]
    if k in ("swiglu_f32", "swiglu_i8"):
        layer = gh.SwiGLU(c["hidden"], c["inter"])
        (layer.gate_weight, layer.gate_bias), (layer.up_weight, layer.up_bias), (layer.down_weight, layer.down_bias) = \
            t["gate"], t["up"], t["down"]
        return {"kind": k, "x": t["x"], "layer": layer if k == "swiglu_f32" else layer.quantize()}
    if k == "qlinear":
        dq = gh.DynamicQuantization()
        dq.quantize_weights("w", t["w"])
        return {"kind": k, "x": t["x"], "dq": dq, "b": t["b"]}
    if k == "gemv_w8":
        q, s, z = gh.quantize_per_channel(t["w"], symmetric=True)
        return {"kind": k, "x": t["x"], "q": q, "s": s, "z": z}
    if k in ("mha", "mha_step"):
        layer = gh.MultiHeadAttention(c["e"], c["h"])
        (layer.q_weight, layer.q_bias, layer.k_weight, layer.k_bias, layer.v_weight, layer.v_bias, layer.out_weight,
         layer.out_bias) = t["p"]
        layer.eval()
        s = {"kind": k, "x": t["x"], "layer": layer, "mask": t.get("mask")}
        if k == "mha_step":
            cache = gh.KVCache(c["b"], c["past"] + c["s"], c["e"])
            cache.k[:, :c["past"]] = t["pk"]
            cache.v[:, :c["past"]] = t["pv"]
            s.update(cache=cache, past=c["past"])
        return s
    if k == "flash":
        cfg = gh.FlashAttentionConfig(block_size_m=c["block"], block_size_n=c["block"], causal=c["causal"],
                                      scale=1.0 / math.sqrt(c["d"]))
        return {"kind": k, "layer": gh.FlashAttention(cfg), **t}
    return {"kind": k, "causal": c.get("causal", False), **t}


def run(state):
    s, k = state, state["kind"]
    if k == "linear":
        return gh.linear(s["x"], s["w"], s["b"])
    if k == "train":
        y = gh.matmul(s["a"], s["b"])
        return (y, *gh.matmul_backward(s["grad"], s["a"], s["b"]))
    if k == "bmm":
        return gh.matmul(s["a"], s["b"])
    if k in ("swiglu_f32", "swiglu_i8"):
        return s["layer"](s["x"])
    if k == "qlinear":
        return s["dq"].quantized_linear("w", s["x"], s["b"])
    if k == "gemv_w8":
        return gh.gemv_w8(s["x"], s["q"], s["s"], s["z"])
    if k == "sdpa":
        return gh.sdpa(s["q"], s["k"], s["v"], causal=s["causal"])
    if k == "mha":
        return s["layer"].forward_with_cache(s["x"], s["x"], s["x"], mask=s["mask"])
    if k == "mha_step":
        # the cache is rewound to the same position before every pass
        cache, past = s["cache"], s["past"]
        cache.length = past
        y = s["layer"].step(s["x"], cache, causal=s["x"].shape[1] > 1)
        return y, cache.k[:, past:], cache.v[:, past:]
    return s["layer"](s["q"], s["k"], s["v"])


# ---- what a pass cannot do without ----------------------------------------------


def work(case):
    c, k = case, case["kind"]
    if k == "linear":
        m, kk, n = c["m"], c["k"], c["n"]
        return {"bytes": 4 * (m * kk + n * kk + m * n + (n if c["bias"] else 0)), "flops": 2 * m * n * kk}
    if k == "train":
        m, kk, n = c["m"], c["k"], c["n"]
        return {"bytes": 4 * (2 * m * kk + 2 * kk * n + 2 * m * n), "flops": 6 * m * n * kk}
    if k == "bmm":
        b, m, kk, n = c["b"], c["m"], c["k"], c["n"]
        return {"bytes": 4 * b * (m * kk + kk * n + m * n), "flops": 2 * b * m * n * kk}
    if k in ("swiglu_f32", "swiglu_i8"):
        m, hid, it = c["m"], c["hidden"], c["inter"]
        weights = 3 * hid * it * 4 if k == "swiglu_f32" else 3 * hid * it + 8 * (2 * it + hid)
        return {"bytes": weights + 4 * (2 * it + hid) + 8 * m * hid, "flops": 6 * m * hid * it}
    if k == "qlinear":
        m, kk, n = c["m"], c["k"], c["n"]
        return {"bytes": n * kk + 8 * n + 4 * m * kk + 4 * m * n + (4 * n if c["bias"] else 0), "flops": 2 * m * n * kk}
    if k == "gemv_w8":
        b, kk, n = c["b"], c["k"], c["n"]
        return {"bytes": kk * n + 5 * kk + 4 * b * (kk + n), "flops": 2 * b * kk * n}
    if k == "sdpa":
        b, h, s, d = c["b"], c["h"], c["s"], c["d"]
        pairs = s * (s + 1) // 2 if c["causal"] else s * s
        return {"bytes": 16 * b * h * s * d, "flops": 4 * b * h * pairs * d}
    if k == "mha":
        b, s, e, h = c["b"], c["s"], c["e"], c["h"]
        return {"bytes": 4 * (4 * (e * e + e) + 4 * b * s * e + b * h * s * s + (s * s if c["mask"] else 0)),
                "flops": 8 * b * s * e * e + 4 * b * s * s * e}
    if k == "mha_step":
        b, s, e, kv = c["b"], c["s"], c["e"], c["past"] + c["s"]
        return {"bytes": 4 * (4 * (e * e + e) + 2 * b * c["past"] * e + 4 * b * s * e),
                "flops": 8 * b * s * e * e + 4 * b * s * kv * e}
    b, s, d = c["b"], c["s"], c["d"]
    pairs = s * (s + 1) // 2 if c["causal"] else s * s
    return {"bytes": 16 * b * s * d, "flops": 4 * b * pairs * d}


def tolerance(case):
    # Sums of fp32 products: over these ranges the library's results lie up to
    # 1.9e-6 from the 64-bit ones (K = 8192), and another order of summation
    # as far.  int8: codes and int32 sums are whole numbers and only the fp32
    # epilogue rounds, but inside the block a last-bit difference of h moves
    # single codes of the next quantization.  flash: an element's error grows
    # with the power its block's correction is raised to.
    k = case["kind"]
    return {"rel": 3e-4 if k == "swiglu_i8" else 8e-6, "max": {"swiglu_i8": 1e-2, "flash": 1e-3}.get(k, 1e-4)}


# ---- the same results in 64 bits, as plain torch gives them ----------------------


def _linear64(x, w, b):
    y = x.double() @ w.double().t()
    return y if b is None else y + b.double()


def _div32(a, b):
    """The correctly rounded fp32 quotient."""
    return (a.double() / b).float()


def _round(v):
    """Half away from zero."""
    return torch.sign(v) * torch.floor(v.abs().double() + 0.5)


def _quant_rows(w):
    """Symmetric per-channel codes and scales (fp32 arithmetic)."""
    s = _div32(w.abs().amax(1), 127.0)
    return torch.clamp(_round(_div32(w, s.double()[:, None])), -128, 127), s


def _quant_tensor(x):
    """Asymmetric per-tensor codes, scale and zero point (fp32 arithmetic)."""
    mn, mx = x.min(), x.max()
    s = _div32(mx - mn, 255.0)
    zp = torch.clamp(_round(_div32(-mn, s.double()) - 128.0), -128, 127)
    return torch.clamp(_round(_div32(x, s.double())) + zp, -128, 127), s, zp


def _qlinear64(x, qw, sw, b):
    qx, sx, zx = _quant_tensor(x)
    y = ((qx - zx) @ qw.t()) * (sx * sw).double()
    return y if b is None else y + b.double()


def _attention64(q, k, v, keep, scale):
    s = (q @ k.transpose(-1, -2)).mul_(scale)
    if keep is not None:
        s.masked_fill_(~keep, -math.inf)
    w = torch.softmax(s, -1)
    return w @ v, w


def _mha64(t, c, past):
    wq, bq, wk, bk, wv, bv, wo, bo = t["p"]
    b, s, e = t["x"].shape
    h, d = c["h"], e // c["h"]
    q, kn, vn = (_linear64(t["x"], w, bias) for w, bias in ((wq, bq), (wk, bk), (wv, bv)))
    k, v = (kn, vn) if not past else (torch.cat([t["pk"].double(), kn], 1), torch.cat([t["pv"].double(), vn], 1))
    heads = lambda u: u.reshape(b, -1, h, d).transpose(1, 2).contiguous()  # noqa: E731
    keep = None
    if past and s > 1:
        keep = torch.ones(s, past + s, device="cuda", dtype=torch.bool).tril(past)
    elif t.get("mask") is not None:
        keep = t["mask"] > 0.5
    o, w = _attention64(heads(q), heads(k), heads(v), keep, 1.0 / math.sqrt(d))
    return _linear64(o.transpose(1, 2).reshape(b, s, e), wo, bo), w, kn, vn


def _flash64(t, c):
    """The blockwise recurrence, one key block after another: the correction
    of a risen maximum multiplies the output once per key of the block."""
    q, k, v = (t[n].double() for n in "qkv")
    b, s, d = q.shape
    bn = c["block"]
    m = torch.full((b, s, 1), -math.inf, device="cuda", dtype=torch.float64)
    total, o = torch.zeros_like(m), torch.zeros_like(q)
    rows = torch.arange(s, device="cuda")[:, None]
    scale = float(torch.tensor(1.0 / math.sqrt(d), dtype=torch.float32))
    for j in range(0, s, bn):
        n = min(bn, s - j)
        x = (q @ k[:, j:j + n].transpose(1, 2).contiguous()) * scale
        if c["causal"]:
            x.masked_fill_(torch.arange(j, j + n, device="cuda")[None, :] > rows, -math.inf)
        new = torch.maximum(m, x.amax(-1, keepdim=True))
        step = m - new
        left = torch.arange(n - 1, -1, -1, device="cuda", dtype=torch.float64)
        p = torch.exp(x - new)
        # the key with `left` keys after it is scaled by exp(step) that many times
        o = o * torch.exp(n * step) + (p * torch.where(left == 0, 1.0, torch.exp(left * step))) @ v[:, j:j + n]
        total = total * torch.exp(step) + p.sum(-1, keepdim=True)
        m = new
    return o / total


def exact(case, seed):
    c, t = case, _inputs(case, seed)
    k = c["kind"]
    if k == "linear":
        return _linear64(t["x"], t["w"], t["b"])
    if k == "train":
        a, b, g = (t[n].double() for n in ("a", "b", "grad"))
        return a @ b, g @ b.t(), a.t() @ g
    if k == "bmm":
        return t["a"].double() @ t["b"].double()
    if k == "swiglu_f32":
        x = t["x"]
        h = torch.nn.functional.silu(_linear64(x, *t["gate"])) * _linear64(x, *t["up"])
        return h @ t["down"][0].double().t() + t["down"][1].double()
    if k == "swiglu_i8":
        (wg, bg), (wu, bu), (wd, bd) = t["gate"], t["up"], t["down"]
        h = torch.nn.functional.silu(_qlinear64(t["x"], *_quant_rows(wg), bg)) * _qlinear64(t["x"], *_quant_rows(wu), bu)
        return _qlinear64(h.float(), *_quant_rows(wd), bd)
    if k == "qlinear":
        return _qlinear64(t["x"], *_quant_rows(t["w"]), t["b"])
    if k == "gemv_w8":
        q, s = _quant_rows(t["w"])
        return t["x"].double() @ (q * s.double()[:, None])
    if k == "sdpa":
        keep = torch.ones(c["s"], c["s"], device="cuda", dtype=torch.bool).tril() if c["causal"] else None
        return torch.stack([_attention64(*(t[n][i].double() for n in "qkv"), keep, 1.0 / math.sqrt(c["d"]))[0]
                            for i in range(c["b"])])
    if k == "mha":
        y, w, kn, vn = _mha64(t, c, 0)
        heads = lambda u: u.reshape(c["b"], c["s"], c["h"], -1).transpose(1, 2)  # noqa: E731
        return y, w, heads(kn), heads(vn)
    if k == "mha_step":
        y, _, kn, vn = _mha64(t, c, c["past"])
        return y, kn, vn
    return _flash64(t, c)
