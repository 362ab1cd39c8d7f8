"""Performance cases: the calls a program makes of this package, with their inputs, work and exact values.

A case is a plain dict.  ``op`` is the call sequence:

* ``gemm``: ``api.gemm(a, b)``, bf16 in and out.  Activations are N(0, 1)
  and weights N(0, 1) / sqrt(K), the scale an initialised linear layer has.
* ``attention``: ``api.attention_forward(q, k, v, causal)`` -> (O, LSE), a
  prefill or an inference layer.
* ``train``: the forward and ``api.attention_backward`` on its outputs, one
  attention layer of a training step -> (O, LSE, dQ, dK, dV).

Attention inputs are N(0, 1) ``[batch, heads, seq, dim]`` with ``kv_heads``
key/value heads.  ``layout`` is how they lie in memory: ``bhsd`` dense, or
``packed``, transposed views of one ``[batch, seq, 3, heads, dim]`` tensor,
as a fused QKV projection writes it.
"""
import math

import torch

from warpir_amd import api


def _gemm(m, n, k, **more):
    return {"op": "gemm", "m": m, "n": n, "k": k, **more}


def _attn(op, batch, heads, kv_heads, seq, dim, causal, layout="bhsd", **more):
    return {"op": op, "batch": batch, "heads": heads, "kv_heads": kv_heads, "seq": seq, "dim": dim,
            "causal": causal, "layout": layout, **more}


def listed():
    return [
        # a small layer (a router, an adapter, a toy model): the call itself is most of the time
        _gemm(256, 256, 256, name="gemm_small"),
        # a decode step over a large weight: 128 sequences, one token each
        _gemm(128, 8192, 8192, name="gemm_decode_m128"),
        # a chunk of a prompt through a down projection: few output tiles and a long reduction
        _gemm(512, 4096, 8192, name="gemm_chunk"),
        # packed variable-length tokens against sizes that are no multiple of a tile
        _gemm(3000, 4104, 4040, name="gemm_ragged"),
        # the square products of a training step: one output tile per compute unit, and four
        _gemm(4096, 4096, 4096, name="gemm_4096"),
        _gemm(8192, 8192, 8192, name="gemm_8192"),
        # one short sequence through a small encoder
        _attn("attention", 1, 8, 8, 512, 64, False, name="attention_small"),
        # a large non-causal layer (image or audio encoder, diffusion)
        _attn("attention", 16, 16, 16, 4096, 128, False, name="attention_d128"),
        # a long causal context with 64-wide heads
        _attn("attention", 8, 32, 32, 8192, 64, True, name="attention_causal_d64"),
        # one prompt's prefill with grouped key/value heads, its length a multiple of 64 and of nothing larger
        _attn("attention", 1, 32, 8, 4160, 128, True, name="attention_gqa_prefill"),
        # a causal training layer
        _attn("train", 16, 16, 16, 4096, 128, True, name="train_causal_d128"),
        # an encoder's training layer on views of a packed QKV projection
        _attn("train", 8, 12, 12, 1024, 64, False, layout="packed", name="train_packed_d64"),
    ]


MAX_FLOPS = {"gemm": 2.0 * 8192 ** 3, "attention": 2.0 * 8 * 32 * 8192 ** 2 * 64,
             "train": 7.0 * 16 * 16 * 4096 ** 2 * 128}


def _log(rng, lo, hi, step):
    """A multiple of ``step`` in [lo, hi], spread evenly over its logarithm."""
    x = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(x / step)) * step))


def draw(rng):
    if rng.random() < 0.5:
        while True:
            kind = rng.choice(("small", "decode", "chunk", "large"))
            step = rng.choice((8, 64, 64, 128))   # hidden sizes are mostly round, vocabularies and experts are not
            if kind == "small":
                c = _gemm(rng.randint(1, 512), _log(rng, 64, 1024, step), _log(rng, 64, 2048, step))
            elif kind == "decode":
                c = _gemm(rng.randint(1, 256), _log(rng, 1024, 16384, step), _log(rng, 1024, 16384, step))
            elif kind == "chunk":
                c = _gemm(_log(rng, 256, 2048, 1), _log(rng, 1024, 16384, step), _log(rng, 1024, 16384, step))
            else:
                c = _gemm(_log(rng, 2048, 16384, rng.choice((1, 64, 256))), _log(rng, 1024, 16384, step),
                          _log(rng, 1024, 16384, step))
            if work(c)["flops"] <= MAX_FLOPS["gemm"]:
                return c
    op = rng.choice(("attention", "train"))
    while True:
        heads = rng.choice((8, 12, 16, 24, 32))
        kv_heads = heads // rng.choice((1, 1, 2, 4))
        layout = rng.choice(("bhsd", "packed")) if kv_heads == heads else "bhsd"
        c = _attn(op, _log(rng, 1, 16, 1), heads, kv_heads, _log(rng, 128, 8192, 64), rng.choice((64, 128)),
                  rng.random() < 0.6, layout)
        if work(c)["flops"] <= MAX_FLOPS[op]:
            return c


def _normal(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.bfloat16)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["op"] == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"op": "gemm", "a": _normal(gen, m, k), "b": _normal(gen, k, n) * k ** -0.5}
    b, h, s, d = case["batch"], case["heads"], case["seq"], case["dim"]
    if case["layout"] == "packed":
        q, k, v = _normal(gen, b, s, 3, h, d).permute(2, 0, 3, 1, 4)
    else:
        q = _normal(gen, b, h, s, d)
        k, v = (_normal(gen, b, case["kv_heads"], s, d) for _ in range(2))
    state = {"op": case["op"], "q": q, "k": k, "v": v, "causal": case["causal"]}
    if case["op"] == "train":
        state["do"] = _normal(gen, b, h, s, d)
    return state


def run(state):
    if state["op"] == "gemm":
        return api.gemm(state["a"], state["b"])
    q, k, v, causal = state["q"], state["k"], state["v"], state["causal"]
    o, lse = api.attention_forward(q, k, v, causal=causal)
    if state["op"] == "attention":
        return o, lse
    return (o, lse, *api.attention_backward(q, k, v, o, lse, state["do"], causal=causal))


def work(case):
    if case["op"] == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2.0 * (m * k + k * n + m * n), "flops": 2.0 * m * n * k}
    b, h, s, d = case["batch"], case["heads"], case["seq"], case["dim"]
    q, kv, stat = 2.0 * b * h * s * d, 2.0 * b * case["kv_heads"] * s * d, 4.0 * b * h * s
    product = 2.0 * b * h * s * s * d / (2 if case["causal"] else 1)
    if case["op"] == "attention":
        return {"bytes": 2 * q + 2 * kv + stat, "flops": 2 * product}
    # q, k, v, dO in; O, LSE, dQ, dK, dV out; two products forward, five backward
    return {"bytes": 4 * q + 4 * kv + stat, "flops": 7 * product}


def tolerance(case):
    # Four times what these kernels show against ``exact`` (2-norm: gemm
    # 1.7e-3, O 2.3e-3, gradients 2.5e-3), which is the bf16 rounding of the
    # outputs, and of the probabilities and score gradients that enter a
    # product.  "max" covers single elements.
    if case["op"] == "gemm":
        return {"rel": 7e-3, "max": 0.02}
    return {"rel": 1e-2, "max": 0.05}


def exact(case, seed):
    state = prepare(case, seed)
    if case["op"] == "gemm":
        return state["a"].double() @ state["b"].double()
    b, h, s, d = case["batch"], case["heads"], case["seq"], case["dim"]
    group, scale, train = h // case["kv_heads"], d ** -0.5, case["op"] == "train"
    q, k, v = state["q"], state["k"], state["v"]
    future = torch.ones(s, s, dtype=torch.bool, device="cuda").triu(1) if case["causal"] else None

    def zeros(like):
        return torch.zeros(like.shape, dtype=torch.float64, device="cuda")

    o, lse = zeros(q), torch.zeros(b, h, s, dtype=torch.float64, device="cuda")
    dq, dk, dv = (zeros(q), zeros(k), zeros(v)) if train else (None, None, None)
    for i in range(b):
        for j in range(h):
            g = j // group
            qh, kh, vh = q[i, j].double(), k[i, g].double(), v[i, g].double()
            p = (qh @ kh.T).mul_(scale)
            if future is not None:
                p.masked_fill_(future, -math.inf)
            lse[i, j] = torch.logsumexp(p, -1)
            p.sub_(lse[i, j, :, None]).exp_()
            o[i, j] = p @ vh
            if train:
                doh = state["do"][i, j].double()
                dv[i, g] += p.T @ doh
                ds = (doh @ vh.T).sub_((doh * o[i, j]).sum(-1, keepdim=True)).mul_(p).mul_(scale)
                dq[i, j] = ds @ kh
                dk[i, g] += ds.T @ qh
    return (o, lse, dq, dk, dv) if train else (o, lse)
