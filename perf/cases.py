"""The calls that a user of this package makes, as timed cases.

A case is a dict of plain values whose ``"kind"`` names one public entry point:

* ``attention``   -- ``attention`` / ``rope_attention``: forward + backward as in
  training, or the forward alone as in evaluation and prefill;
* ``decode``      -- ``decode_attention``: one new token per sequence against a
  KV cache;
* ``norm``        -- ``add_rms_norm``: the residual add and the norm, forward +
  backward;
* ``head``        -- ``ops.fused_linear_cross_entropy``: the loss head, forward +
  backward;
* ``sample``      -- ``ops.topk_sample``: the draw after each generated token;
* ``train``       -- ``TradingModel.forward_with_loss`` under bf16 autocast and
  the gradient of every parameter;
* ``generate``    -- one generated token through the whole decoder with KV
  caches, recorded as a HIP graph and replayed, as ``TradingModel.generate``
  does for every token after the first.

``listed()`` are the sizes the package is run at; ``draw(rng)`` gives others of
the same ranges.  Inputs come from the seed alone and are made on the GPU.
"""

from __future__ import annotations

import importlib
import math

import torch
import torch.nn.functional as F

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_DEV = "cuda"
_EPS = 1e-5
_THETA = 500_000.0
# (query heads, KV heads): multi-head, and grouped-query with 2, 3, 4, 7 and 8 heads a group
_HEADS = ((4, 4), (4, 2), (6, 2), (8, 2), (16, 4), (32, 8), (14, 2), (16, 2))


def _pkg():
    return importlib.import_module("mega-trading_amd")


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # long-context training layer: 4096 tokens, 16 / 4 heads of 64 (the benchmark's headline shape)
        dict(name="train_t4096_d64", kind="attention", dtype="bf16", b=4, t=4096, hq=16, hkv=4, d=64, rope=True, train=True),
        # the widest training layer: 32 / 8 heads of 128
        dict(name="train_t2048_d128", kind="attention", dtype="bf16", b=8, t=2048, hq=32, hkv=8, d=128, rope=True, train=True),
        # a ragged batch of a model with three query heads a group, fp16, RoPE applied by the caller
        dict(name="train_ragged_fp16", kind="attention", dtype="fp16", b=5, t=777, hq=12, hkv=4, d=64, rope=False, train=True),
        # full-precision training and evaluation without autocast
        dict(name="train_fp32", kind="attention", dtype="fp32", b=8, t=512, hq=16, hkv=4, d=64, rope=True, train=True),
        # one short prompt: the smallest call, forward only
        dict(name="prompt_t200", kind="attention", dtype="bf16", b=1, t=200, hq=8, hkv=2, d=64, rope=True, train=False),
        # a token of 32 rollouts after a prompt of 512 tokens (the generation benchmark)
        dict(name="decode_32_rollouts", kind="decode", dtype="bf16", b=32, hq=8, hkv=2, d=64, capacity=1024, length=545),
        # a token of 16 long sequences of the widest model
        dict(name="decode_long", kind="decode", dtype="bf16", b=16, hq=32, hkv=8, d=128, capacity=8192, length=6001),
        # residual add + norm of a 1024-wide model, 64 sequences of 512 tokens
        dict(name="add_norm_1024", kind="norm", dtype="bf16", rows=32768, dim=1024),
        # loss head of the 8-layer model: 32 sequences of 1024 tokens, 16384 words
        dict(name="loss_head", kind="head", dtype="bf16", rows=32768, hidden=512, vocab=16384),
        # the draw of one token for each of 32 rollouts
        dict(name="sample_32", kind="sample", rows=32, vocab=16384, k=16),
        # a training step of four of the 8-layer model's blocks with embedding and head
        dict(name="train_step", kind="train", b=16, t=1024, layers=4, hidden=512, hq=8, hkv=2, ffn=1408, vocab=16384),
        # a generated token of the 8-layer model, 32 rollouts, fp32 weights
        dict(name="generate_token", kind="generate", b=32, layers=8, hidden=512, hq=8, hkv=2, ffn=1408, vocab=16384,
             capacity=1024, pos=600),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("attention", "attention", "attention", "attention", "decode", "decode", "norm", "head", "sample",
                       "train", "generate"))
    if kind == "attention":
        dtype = rng.choice(("bf16", "bf16", "bf16", "fp16", "fp32"))
        hq, hkv = rng.choice(_HEADS)
        d = rng.choice((32, 64, 64, 128))
        t = _log(rng, 64, 1024 if dtype == "fp32" else 4096)
        # batches from one sequence to what fills a training step, no dearer than the largest listed case
        most = (3e10 if dtype == "fp32" else 9e11) / (3.5 * 4 * hq * d * t * (t + 1) / 2)
        b = _log(rng, 1, max(1, min(32, int(most))))
        return dict(kind=kind, dtype=dtype, b=b, t=t, hq=hq, hkv=hkv, d=d, rope=rng.random() < 0.6, train=rng.random() < 0.75)
    if kind == "decode":
        hq, hkv = rng.choice(_HEADS)
        d = rng.choice((32, 64, 64, 128))
        capacity = 64 * _log(rng, 4, 128)
        most = 5e8 / (4 * hkv * d * capacity)
        b = _log(rng, 1, max(1, min(64, int(most))))
        return dict(kind=kind, dtype=rng.choice(("bf16", "fp16")), b=b, hq=hq, hkv=hkv, d=d, capacity=capacity,
                    length=rng.randint(capacity // 4, capacity))
    if kind == "norm":
        dim = 8 * _log(rng, 16, 512)
        return dict(kind=kind, dtype=rng.choice(("bf16", "fp32")), rows=_log(rng, 32, min(65536, 64_000_000 // dim)), dim=dim)
    if kind == "head":
        vocab = _log(rng, 2000, 16384)
        return dict(kind=kind, dtype=rng.choice(("bf16", "bf16", "fp16")), rows=_log(rng, 1024, 32768),
                    hidden=rng.choice((256, 384, 512)), vocab=vocab)
    if kind == "sample":
        return dict(kind=kind, rows=_log(rng, 1, 64), vocab=_log(rng, 1000, 32768), k=rng.choice((1, 16, 50)))
    hidden, hq, hkv = rng.choice(((256, 4, 2), (384, 6, 2), (512, 8, 2), (512, 8, 8), (768, 12, 4)))
    ffn = -(-8 * hidden // 3 // 16) * 16
    if kind == "train":
        return dict(kind=kind, b=_log(rng, 2, 16), t=_log(rng, 64, 1024), layers=rng.randint(2, 4), hidden=hidden, hq=hq,
                    hkv=hkv, ffn=ffn, vocab=_log(rng, 2000, 16384))
    capacity = 128 * rng.randint(2, 8)
    return dict(kind=kind, b=_log(rng, 1, 64), layers=rng.randint(2, 8), hidden=hidden, hq=hq, hkv=hkv, ffn=ffn,
                vocab=_log(rng, 2000, 16384), capacity=capacity, pos=rng.randint(capacity // 4, capacity - 1))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=_DEV).manual_seed(int(seed))


def _normal(g, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device=_DEV) * std).to(dtype)


def _heads(g, c, heads, dtype):
    """[B, H, T, D] view of a [B, T, H, D] projection output, as a decoder layer passes it."""
    return _normal(g, c["b"], c["t"], heads, c["d"], dtype=dtype).transpose(1, 2)


def _tables(rows, d):
    inv = 1.0 / (_THETA ** (torch.arange(0, d, 2, dtype=torch.float32) / d))
    freqs = torch.outer(torch.arange(rows, dtype=torch.float32), inv)
    return freqs.cos().view(1, 1, rows, d // 2).to(_DEV), freqs.sin().view(1, 1, rows, d // 2).to(_DEV)


def _zipf(g, shape, vocab):
    """Token ids with P(rank) ~ rank^-1.1, the order-flow vocabulary's shape."""
    p = torch.arange(1, vocab + 1, dtype=torch.float64, device=_DEV) ** -1.1
    cdf = torch.cumsum(p / p.sum(), 0)
    u = torch.rand(*shape, generator=g, device=_DEV, dtype=torch.float64)
    return torch.searchsorted(cdf, u).clamp_(max=vocab - 1)


def _weights(c, g):
    """Decoder weights by parameter name: N(0, 0.02) matrices, norms around one."""
    h, ffn, d = c["hidden"], c["ffn"], c["hidden"] // c["hq"]
    w = {"token_embedding.weight": _normal(g, c["vocab"], h, std=0.02), "norm.weight": 1 + _normal(g, h, std=0.1)}
    for i in range(c["layers"]):
        p = "blocks.%d." % i
        w[p + "attention_norm.weight"] = 1 + _normal(g, h, std=0.1)
        w[p + "ffn_norm.weight"] = 1 + _normal(g, h, std=0.1)
        w[p + "attention.q_proj.weight"] = _normal(g, h, h, std=0.04)
        w[p + "attention.k_proj.weight"] = _normal(g, c["hkv"] * d, h, std=0.04)
        w[p + "attention.v_proj.weight"] = _normal(g, c["hkv"] * d, h, std=0.04)
        w[p + "attention.o_proj.weight"] = _normal(g, h, h, std=0.02)
        w[p + "feed_forward.w1.weight"] = _normal(g, ffn, h, std=0.02)
        w[p + "feed_forward.w3.weight"] = _normal(g, ffn, h, std=0.02)
        w[p + "feed_forward.w2.weight"] = _normal(g, h, ffn, std=0.02)
    return w


def _inputs(c, seed):
    g = _gen(seed)
    kind = c["kind"]
    if kind == "attention":
        dt = _DTYPES[c["dtype"]]
        s = dict(q=_heads(g, c, c["hq"], dt), k=_heads(g, c, c["hkv"], dt), v=_heads(g, c, c["hkv"], dt))
        if c["train"]:
            s["do"] = _heads(g, c, c["hq"], dt)
        if c["rope"]:
            s["cos"], s["sin"] = _tables(c["t"], c["d"])
        return s
    if kind == "decode":
        dt = _DTYPES[c["dtype"]]
        cache = (c["b"], c["hkv"], c["capacity"], c["d"])
        return dict(q=_normal(g, c["b"], c["hq"], 1, c["d"], dtype=dt), k=_normal(g, *cache, dtype=dt),
                    v=_normal(g, *cache, dtype=dt))
    if kind == "norm":
        dt, n = _DTYPES[c["dtype"]], (c["rows"], c["dim"])
        return dict(x=_normal(g, *n, dtype=dt), r=_normal(g, *n, dtype=dt), w=(1 + _normal(g, c["dim"], std=0.1)).to(dt),
                    dr=_normal(g, *n, dtype=dt), dy=_normal(g, *n, dtype=dt))
    if kind == "head":
        dt = _DTYPES[c["dtype"]]
        return dict(h=_normal(g, c["rows"], c["hidden"], dtype=dt), w=_normal(g, c["vocab"], c["hidden"], std=0.05, dtype=dt),
                    labels=_zipf(g, (c["rows"],), c["vocab"]))
    if kind == "sample":
        n = (c["rows"], c["vocab"])
        return dict(x=_normal(g, *n, std=2.0), e=torch.empty(*n, device=_DEV).exponential_(1.0, generator=g))
    s = dict(weights=_weights(c, g))
    d = c["hidden"] // c["hq"]
    if kind == "train":
        ids = _zipf(g, (c["b"], c["t"] + 1), c["vocab"])
        s["ids"], s["labels"] = ids[:, :-1].contiguous(), ids[:, 1:].contiguous()
    else:
        s["token"] = _zipf(g, (c["b"], 1), c["vocab"])
        # [layer, key / value, B, Hkv, capacity, D]: keys rotated, values as projected
        s["caches"] = _normal(g, c["layers"], 2, c["b"], c["hkv"], c["capacity"], d, dtype=torch.bfloat16)
    return s


def _model(c, weights, rows):
    pkg = _pkg()
    with torch.device(_DEV):
        model = pkg.model.TradingModel(c["vocab"], rows, hidden_dim=c["hidden"], layers=c["layers"], attention_heads=c["hq"],
                                       kv_heads=c["hkv"], intermediate_dim=c["ffn"], dropout=0.0, rope_theta=_THETA,
                                       norm_eps=_EPS, attention_backend="hip")
    with torch.no_grad():
        for name, p in model.named_parameters():
            p.copy_(weights[name])
    return model


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    kind = case["kind"]
    if kind == "attention" and case["train"]:
        for n in ("q", "k", "v"):
            s[n].requires_grad_(True)
    elif kind == "norm":
        for n in ("x", "r", "w"):
            s[n].requires_grad_(True)
    elif kind == "head":
        for n in ("h", "w"):
            s[n].requires_grad_(True)
    elif kind == "train":
        s["model"] = _model(case, s.pop("weights"), case["t"]).train()
    elif kind == "generate":
        s["model"] = _model(case, s.pop("weights"), case["capacity"]).eval()
        s["pos"] = torch.full((1,), case["pos"], dtype=torch.int32, device=_DEV)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _decode_token(s)
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["logits"] = _decode_token(s)
    return s


@torch.no_grad()
def _decode_token(s):
    """The decoder on one token per sequence at position ``pos``: its keys and
    values go into the caches, the logits after it come back."""
    pkg, model = _pkg(), s["model"]
    length = s["pos"] + 1
    hidden = model.token_embedding(s["token"])
    normed = model.blocks[0].attention_norm(hidden)
    for i, block in enumerate(model.blocks):
        nxt = model.blocks[i + 1].attention_norm if i + 1 < len(model.blocks) else model.norm
        attended = block.attention.decode(normed, s["caches"][i, 0], s["caches"][i, 1], s["pos"], length)
        hidden, normed = pkg.add_rms_norm(attended, hidden, block.ffn_norm.weight, eps=_EPS)
        hidden, normed = pkg.add_rms_norm(block.feed_forward(normed), hidden, nxt.weight, eps=_EPS)
    return model.output(normed)[:, -1, :]


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    pkg, c = _pkg(), s["case"]
    kind = c["kind"]
    if kind == "attention":
        repeats = c["hq"] // c["hkv"]

        def call():
            if c["rope"]:
                return pkg.rope_attention(s["q"], s["k"], s["v"], s["cos"], s["sin"], repeats=repeats)
            return pkg.attention(s["q"], s["k"], s["v"], repeats=repeats)

        if not c["train"]:
            with torch.no_grad():
                return call()
        out = call()
        return (out, *torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["do"]))
    if kind == "decode":
        return pkg.decode_attention(s["q"], s["k"], s["v"], c["length"], repeats=c["hq"] // c["hkv"])
    if kind == "norm":
        res, y = pkg.add_rms_norm(s["x"], s["r"], s["w"], eps=_EPS)
        return (res, y, *torch.autograd.grad((res, y), (s["x"], s["r"], s["w"]), (s["dr"], s["dy"])))
    if kind == "head":
        loss = pkg.ops.fused_linear_cross_entropy(s["h"], s["w"], s["labels"])
        return (loss, *torch.autograd.grad(loss, (s["h"], s["w"])))
    if kind == "sample":
        return pkg.ops.topk_sample(s["x"], s["e"], min(c["k"], c["vocab"]))
    if kind == "train":
        with torch.autocast("cuda", dtype=torch.bfloat16):
            loss, _ = s["model"].forward_with_loss(s["ids"], s["labels"], return_logits=False)
        names, params = zip(*s["model"].named_parameters())
        return loss, dict(zip(names, torch.autograd.grad(loss, params)))
    s["graph"].replay()
    return s["logits"], s["caches"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _matrix_params(c):
    """Weights of the decoder's projections, without embedding and head."""
    d = c["hidden"] // c["hq"]
    return c["layers"] * c["hidden"] * (2 * c["hidden"] + 2 * c["hkv"] * d + 3 * c["ffn"])


def work(case):
    c, kind = case, case["kind"]
    if kind == "attention":
        q, kv, e = c["b"] * c["hq"] * c["t"] * c["d"], c["b"] * c["hkv"] * c["t"] * c["d"], _DTYPES[c["dtype"]].itemsize
        fwd = 4.0 * c["b"] * c["hq"] * c["d"] * c["t"] * (c["t"] + 1) / 2
        if c["train"]:  # q, k, v, dO in; O, dQ, dK, dV out
            return dict(bytes=e * (4 * q + 4 * kv), flops=3.5 * fwd)
        return dict(bytes=e * (2 * q + 2 * kv), flops=fwd)
    if kind == "decode":
        return dict(bytes=2 * (2 * c["b"] * c["hkv"] * c["length"] * c["d"] + 2 * c["b"] * c["hq"] * c["d"]),
                    flops=4.0 * c["b"] * c["hq"] * c["length"] * c["d"])
    if kind == "norm":
        n = c["rows"] * c["dim"]  # x, r, two gradients in; the sum, the norm and the (shared) gradient out
        return dict(bytes=7 * n * _DTYPES[c["dtype"]].itemsize, flops=16.0 * n)
    if kind == "head":
        n = c["rows"] * c["hidden"] + c["vocab"] * c["hidden"]
        return dict(bytes=2 * 2 * n + 8 * c["rows"], flops=6.0 * c["rows"] * c["vocab"] * c["hidden"])
    if kind == "sample":
        n = c["rows"] * c["vocab"]
        return dict(bytes=8 * n + 8 * c["rows"], flops=4.0 * n)
    mats, table, d = _matrix_params(c), c["vocab"] * c["hidden"], c["hidden"] // c["hq"]
    if kind == "train":
        rows = c["b"] * c["t"]
        att = 3.5 * 4.0 * c["layers"] * c["b"] * c["hidden"] * c["t"] * (c["t"] + 1) / 2
        return dict(bytes=8 * (mats + table) + 16 * rows, flops=6.0 * rows * (mats + table) + att)
    kv = 2 * 2 * c["layers"] * c["b"] * c["hkv"] * d * (c["pos"] + 1)
    return dict(bytes=4 * (mats + table) + kv + 4 * c["b"] * c["vocab"],
                flops=2.0 * c["b"] * (mats + table) + 4.0 * c["layers"] * c["b"] * c["hidden"] * (c["pos"] + 1))


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return "exact"  # whole numbers: no two p / E of a row are within a rounding of each other
    if kind == "attention" and case["dtype"] == "fp32":
        return dict(rel=1e-5)
    if kind in ("attention", "decode"):
        return dict(rel=2e-3 if case["dtype"] == "fp16" else 1.2e-2)  # P and dS rounded to 16 bits before their products
    if kind == "norm":
        return dict(rel=5e-6 if case["dtype"] == "fp32" else 1e-2)
    if kind == "head":
        return dict(rel=2e-3 if case["dtype"] == "fp16" else 1e-2)
    if kind == "train":
        return dict(rel=2.5e-2)  # 16-bit activations through the layers
    return dict(rel=1e-2)        # 16-bit queries, keys and values in every layer


# ---------------------------------------------------------------------------
# the same outputs in 64 bits
# ---------------------------------------------------------------------------
def _rotate(x, cos, sin):
    e, o = x[..., 0::2], x[..., 1::2]
    return torch.stack((e * cos - o * sin, e * sin + o * cos), dim=-1).flatten(-2)


def _attend(q, k, v):
    """Causal attention of one KV group: q [R, T, D], k and v [T, D]."""
    t = q.shape[-2]
    s = (q @ k.t()) / math.sqrt(q.shape[-1])
    s = s.masked_fill(torch.ones(t, t, dtype=torch.bool, device=q.device).triu(1), float("-inf"))
    return torch.softmax(s, dim=-1) @ v


def _attend_all(q, k, v):
    """_attend over [B, Hq, T, D] and [B, Hkv, T, D], a group at a time."""
    r = q.shape[1] // k.shape[1]
    return torch.stack([torch.cat([_attend(q[b, j * r:(j + 1) * r], k[b, j], v[b, j]) for j in range(k.shape[1])])
                        for b in range(q.shape[0])])


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + _EPS) * w


def _exact_attention(c, s):
    r = c["hq"] // c["hkv"]
    cos, sin = (s[n][0, 0].double() for n in ("cos", "sin")) if c["rope"] else (None, None)
    full = [torch.empty(s[n].shape, dtype=torch.float64, device=_DEV) for n in ("q", "q", "k", "v")]
    for b in range(c["b"]):
        for j in range(c["hkv"]):
            h = slice(j * r, (j + 1) * r)
            q, k, v = s["q"][b, h].double(), s["k"][b, j].double(), s["v"][b, j].double()
            for x in (q, k, v):
                x.requires_grad_(c["train"])
            out = _attend(*((_rotate(q, cos, sin), _rotate(k, cos, sin)) if c["rope"] else (q, k)), v)
            full[0][b, h] = out.detach()
            if c["train"]:
                full[1][b, h], full[2][b, j], full[3][b, j] = torch.autograd.grad(out, (q, k, v), s["do"][b, h].double())
    return tuple(full) if c["train"] else full[0]


def _exact_layers(c, w, hidden, attend):
    d = c["hidden"] // c["hq"]
    for i in range(c["layers"]):
        p = "blocks.%d." % i
        n = _rms(hidden, w[p + "attention_norm.weight"])
        q, k, v = (n @ w[p + "attention.%s_proj.weight" % x].t() for x in "qkv")
        q, k, v = (x.view(*x.shape[:-1], -1, d).transpose(1, 2) for x in (q, k, v))
        a = attend(i, q, k, v).transpose(1, 2).reshape(hidden.shape)
        hidden = hidden + a @ w[p + "attention.o_proj.weight"].t()
        n = _rms(hidden, w[p + "ffn_norm.weight"])
        gate = F.silu(n @ w[p + "feed_forward.w1.weight"].t()) * (n @ w[p + "feed_forward.w3.weight"].t())
        hidden = hidden + gate @ w[p + "feed_forward.w2.weight"].t()
    return _rms(hidden, w["norm.weight"])


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "sample":
        return None
    s = _inputs(c, seed)
    if kind == "attention":
        return _exact_attention(c, s)
    if kind == "decode":
        n, r = c["length"], c["hq"] // c["hkv"]
        q = s["q"].double().view(c["b"], c["hkv"], r, c["d"])
        p = torch.softmax(q @ s["k"][:, :, :n].double().transpose(2, 3) / math.sqrt(c["d"]), dim=-1)
        return (p @ s["v"][:, :, :n].double()).view(c["b"], c["hq"], 1, c["d"])
    if kind == "norm":
        x, r, w = (s[n].double().requires_grad_(True) for n in ("x", "r", "w"))
        res = x + r
        y = _rms(res, w)
        grads = torch.autograd.grad((res, y), (x, r, w), (s["dr"].double(), s["dy"].double()))
        return (res.detach(), y.detach(), *grads)
    if kind == "head":
        h, w = (s[n].double().requires_grad_(True) for n in ("h", "w"))
        loss = F.cross_entropy(h @ w.t(), s["labels"])
        return (loss.detach(), *torch.autograd.grad(loss, (h, w)))
    w = {n: x.double() for n, x in s["weights"].items()}
    d = c["hidden"] // c["hq"]
    if kind == "train":
        for x in w.values():
            x.requires_grad_(True)
        cos, sin = (x[0, 0].double() for x in _tables(c["t"], d))
        hidden = w["token_embedding.weight"][s["ids"]]
        normed = _exact_layers(c, w, hidden, lambda i, q, k, v: _attend_all(_rotate(q, cos, sin), _rotate(k, cos, sin), v))
        loss = F.cross_entropy(normed.reshape(-1, c["hidden"]) @ w["token_embedding.weight"].t(), s["labels"].reshape(-1))
        return loss.detach(), dict(zip(w, torch.autograd.grad(loss, list(w.values()))))
    cos, sin = (x[0, 0, c["pos"]].double() for x in _tables(c["capacity"], d))
    caches = s["caches"].double()
    n, r = c["pos"] + 1, c["hq"] // c["hkv"]

    def attend(i, q, k, v):
        caches[i, 0, :, :, c["pos"]], caches[i, 1, :, :, c["pos"]] = _rotate(k, cos, sin)[:, :, 0], v[:, :, 0]
        q = _rotate(q, cos, sin).reshape(c["b"], c["hkv"], r, d)
        p = torch.softmax(q @ caches[i, 0, :, :, :n].transpose(2, 3) / math.sqrt(d), dim=-1)
        return (p @ caches[i, 1, :, :, :n]).view(c["b"], c["hq"], 1, d)

    normed = _exact_layers(c, w, w["token_embedding.weight"][s["token"]], attend)
    return normed[:, -1, :] @ w["token_embedding.weight"].t(), caches
