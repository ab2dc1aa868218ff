"""Performance cases of the MI355X MoE decode library: what a program built on it runs.

Each case is one pass through the public entry points of ``kanjoos_amd`` at the
Qwen3-30B-A3B geometry (hidden 2048, 32/4 heads x 128, 128 experts top-8 of width
768) or, for drawn cases, at other shapes the entry points take.  Weights are
random Q4_K / Q6_K / bf16 / f32 tensors of standard deviation 0.02 made on the
GPU from the seed; ``exact`` recomputes a pass in float64 with plain torch.

Kinds:

* ``gemv``      -- one weight matrix applied to one vector (``gemv``)
* ``moe_token`` -- one token through a few MoE layers (``moe_decode_layer``)
* ``moe_batch`` -- one MoE layer over many tokens (``moe_batch_layer``)
* ``attn``      -- one decode token's attention block (``attention_step``)
* ``decode``    -- greedy decode of one sequence on a whole model (``Model``)
* ``prompt``    -- a prompt through a whole model in one call (``Model.forward``)
* ``batch``     -- lockstep decode of several sequences (``Batch``)

The whole-model cases run a few layers of the 48-layer model over a smaller
vocabulary; every layer is alike, so their share per layer is the full model's.
A prompt's rows meet f16 cache slots and routing in every layer, and a last-bit
difference that flips either grows from layer to layer, so prompts run two.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import kanjoos_amd as K

STD = 0.02
EPS = 1e-6
ROPE_BASE = 1e6
TYPES = {"q4_k": K.TYPE_Q4_K, "q6_k": K.TYPE_Q6_K, "bf16": K.TYPE_BF16, "f32": K.TYPE_F32}

A3B = dict(n_embd=2048, n_ff=768, n_expert=128, k=8)
HEADS = dict(n_head=32, n_head_kv=4, head_dim=128)


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # the fused QKV projection of one token with its RMSNorm: the smallest launch a
        # decode step makes, latency-bound
        dict(name="gemv_qkv", kind="gemv", type="q4_k", n_in=2048, n_out=5120, norm=True, resid=False),
        # a Q6_K LM head (Q4_K_M-style files) over the whole vocabulary: one long stream
        dict(name="gemv_head_q6k", kind="gemv", type="q6_k", n_in=2048, n_out=151936, norm=True, resid=False),
        # one token's MoE FFN, layer after layer, as a decode loop of a caller's own calls it
        dict(name="moe_token", kind="moe_token", layers=8, down="q4_k", **A3B),
        # one MoE layer over a short prompt or a large decode batch: a few tokens per expert
        dict(name="moe_batch_77", kind="moe_batch", n_tokens=77, down="q4_k", **A3B),
        # one MoE layer over a 512-token prompt chunk
        dict(name="moe_batch_512", kind="moe_batch", n_tokens=512, down="q4_k", **A3B),
        # a longer ragged chunk with Q6_K expert down
        dict(name="moe_batch_1000_q6k", kind="moe_batch", n_tokens=1000, down="q6_k", **A3B),
        # one token's attention at a 4K context and at a 32K context
        dict(name="attn_4k", kind="attn", pos=4100, n_ctx=4352, **HEADS),
        dict(name="attn_32k", kind="attn", pos=32770, n_ctx=33024, **HEADS),
        # greedy decode at a 4K context: 32 tokens of one sequence
        dict(name="decode_4k", kind="decode", layers=6, vocab=32768, pos=4096, steps=32, down="q4_k", head="bf16"),
        # a 512-token prompt into an empty cache
        dict(name="prompt_512", kind="prompt", layers=2, vocab=32768, pos=0, n=512, down="q4_k", head="bf16"),
        # a long ragged prompt that continues a conversation, Q6_K expert down and head
        dict(name="prompt_1500_q6k", kind="prompt", layers=2, vocab=32768, pos=1000, n=1500, down="q6_k", head="q6_k"),
        # 32 sequences decoded together at a 2K context: 16 steps, logits of the last
        dict(name="batch_32x2k", kind="batch", layers=4, vocab=32768, n_seq=32, pos=2048, steps=16, down="q4_k",
             head="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "moe_token", "moe_batch", "moe_batch", "attn", "decode", "prompt", "prompt", "batch"])
    quant = rng.choice(["q4_k", "q6_k"])
    if kind == "gemv":
        t = rng.choice(["q4_k", "q4_k", "q6_k", "bf16", "f32"])
        n_in = 256 * rng.randint(2, 24)
        most = min(151936, int(320e6 / _row_bytes(t, n_in)))
        return dict(kind=kind, type=t, n_in=n_in, n_out=_log(rng, 100, most), norm=rng.random() < 0.5,
                    resid=rng.random() < 0.5)
    shape = dict(A3B)
    if rng.random() < 0.3:
        shape = dict(n_embd=256 * rng.randint(4, 12), n_ff=256 * rng.randint(1, 5), n_expert=rng.randint(8, 128),
                     k=rng.randint(2, 8))
    if kind == "moe_token":
        return dict(kind=kind, layers=rng.randint(2, 8), down=quant, **shape)
    if kind == "moe_batch":
        return dict(kind=kind, n_tokens=_log(rng, 2, 1000), down=quant, **shape)
    if kind == "attn":
        heads = rng.choice([(32, 4, 128), (32, 4, 128), (32, 8, 128), (16, 4, 128), (8, 2, 64), (16, 2, 64)])
        pos = _log(rng, 20, 32770)
        return dict(kind=kind, pos=pos, n_ctx=pos + rng.randint(1, 300), n_head=heads[0], n_head_kv=heads[1],
                    head_dim=heads[2])
    head = rng.choice(["bf16", "q6_k"])
    layers, vocab = rng.randint(2, 3), rng.randint(8, 32) * 1024 + rng.choice([0, 0, 32, 96])
    if kind == "decode":
        return dict(kind=kind, layers=layers, vocab=vocab, pos=_log(rng, 400, 16000), steps=rng.randint(4, 32), down=quant,
                    head=head)
    if kind == "prompt":
        return dict(kind=kind, layers=2, vocab=vocab, pos=rng.choice([0, 0, _log(rng, 20, 4000)]),
                    n=_log(rng, 16, 1500), down=quant, head=head)
    return dict(kind=kind, layers=layers, vocab=vocab, n_seq=rng.randint(2, 40), pos=_log(rng, 200, 2500),
                steps=rng.randint(2, 16), down=quant, head=head)


# ------------------------------------------------------------------ inputs

def _row_bytes(t, n):
    return {"q4_k": n // 256 * 144, "q6_k": n // 256 * 210, "bf16": 2 * n, "f32": 4 * n}[t]


def _gen(seed, *more):
    g = torch.Generator(device="cuda")
    s = seed & 0xFFFFFFFF
    for m in more:
        s = (s * 1000003 + m + 1) & 0x7FFFFFFFFFFF
    g.manual_seed(s)
    return g


def _bytes(g, shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g)


def _f16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(*v.shape, 2)


def _q4k(g, rows, n_in, std):
    """Q4_K rows: bell-shaped codes 0..14 around 7, 6-bit scales, mins that centre them."""
    nb = n_in // 256
    r = _bytes(g, (rows, nb, 4, 2, 32))
    q = (r & 7) + ((r >> 3) & 7)
    qs = (q[:, :, :, 0] | (q[:, :, :, 1] << 4)).reshape(rows, nb, 128)
    t = _bytes(g, (rows, nb, 8, 2))
    sc = 24 + (t[..., 0] >> 3)
    mn = (sc - 2 + (t[..., 1] & 3)).clamp(0, 63)
    packed = torch.cat([sc[..., :4] | ((sc[..., 4:] >> 4) << 6), mn[..., :4] | ((mn[..., 4:] >> 4) << 6),
                        (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], dim=-1)
    d = std / (3.24 * 40) * (0.8 + 0.4 * torch.rand((rows, nb), device="cuda", generator=g))
    return torch.cat([_f16_bytes(d), _f16_bytes(7 * d), packed, qs], dim=-1).reshape(rows, nb * 144)


def _q6k(g, rows, n_in, std):
    """Q6_K rows: bell-shaped codes -31..31, int8 scales of both signs."""
    nb = n_in // 256
    r = torch.randint(0, 1024, (rows, nb, 2, 4, 32), dtype=torch.int16, device="cuda", generator=g)
    q = ((r & 31) + (r >> 5) + 1).to(torch.uint8)
    lo, hi = q & 15, q >> 4
    ql = (lo[:, :, :, :2] | (lo[:, :, :, 2:] << 4)).reshape(rows, nb, 128)
    qh = (hi[:, :, :, 0] | (hi[:, :, :, 1] << 2) | (hi[:, :, :, 2] << 4) | (hi[:, :, :, 3] << 6)).reshape(rows, nb, 64)
    t = _bytes(g, (rows, nb, 16))
    sc = (64 + (t >> 2)).to(torch.int8) * (1 - 2 * (t & 1).to(torch.int8))
    d = std / (13.0 * 95) * (0.8 + 0.4 * torch.rand((rows, nb), device="cuda", generator=g))
    return torch.cat([ql, qh, sc.view(torch.uint8), _f16_bytes(d)], dim=-1).reshape(rows, nb * 210)


def _weight(g, t, rows, n_in, std=STD):
    """`rows` rows of type `t` as bytes [rows][row_bytes], made in pieces that bound the temporaries."""
    if t in ("bf16", "f32"):
        w = torch.randn((rows, n_in), device="cuda", generator=g) * std
        return (w.to(torch.bfloat16) if t == "bf16" else w).view(torch.uint8)
    out = torch.empty((rows, _row_bytes(t, n_in)), dtype=torch.uint8, device="cuda")
    step = max(1, (1 << 27) // n_in)
    for i in range(0, rows, step):
        n = min(step, rows - i)
        out[i:i + n] = (_q4k if t == "q4_k" else _q6k)(g, n, n_in, std)
    return out


def _norm_weight(g, n):
    return 1.0 + 0.1 * torch.randn(n, device="cuda", generator=g)


def _moe_weights(g, c):
    """Router, its norm, and the expert slabs of one layer."""
    H, F, E = c["n_embd"], c["n_ff"], c["n_expert"]
    return dict(norm=_norm_weight(g, H), router=_weight(g, "f32", E, H), gate=_weight(g, "q4_k", E * F, H),
                up=_weight(g, "q4_k", E * F, H), down=_weight(g, c["down"], E * H, F))


def _tokens(g, n, width):
    """n rows of a residual stream: rows of one text share part of their direction."""
    return torch.randn((n, width), device="cuda", generator=g) + 0.5 * torch.randn(width, device="cuda", generator=g)


def _model_shape(c):
    return dict(A3B, **HEADS, down=c["down"], head=c["head"], layers=c["layers"], vocab=c["vocab"])


def _model_tensors(c, seed):
    """The tensors of a whole model in image order, one (name, bytes) pair at a time."""
    H, F, E = A3B["n_embd"], A3B["n_ff"], A3B["n_expert"]
    D, QD, KVD = HEADS["head_dim"], HEADS["n_head"] * HEADS["head_dim"], HEADS["n_head_kv"] * HEADS["head_dim"]
    yield "embd", _weight(_gen(seed, 1), "bf16", c["vocab"], H, 1.0)
    for il in range(c["layers"]):
        g = _gen(seed, 2, il)
        for name, n in (("attn_norm", H), ("ffn_norm", H), ("q_norm", D), ("k_norm", D)):
            yield name, _norm_weight(g, n).view(torch.uint8)
        yield "wqkv", _weight(g, "q4_k", QD + 2 * KVD, H)
        yield "wo", _weight(g, "q4_k", H, QD)
        yield "router", _weight(g, "f32", E, H)
        yield "gate", _weight(g, "q4_k", E * F, H)
        yield "up", _weight(g, "q4_k", E * F, H)
        yield "down", _weight(g, c["down"], E * H, F)
    yield "out_norm", _norm_weight(_gen(seed, 3), H).view(torch.uint8)
    yield "head", _weight(_gen(seed, 4), c["head"], c["vocab"], H)


def _n_ctx(c):
    return {"decode": lambda: c["pos"] + c["steps"], "prompt": lambda: c["pos"] + c["n"],
            "batch": lambda: c["pos"] + c["steps"]}[c["kind"]]() + 64


def _model(c, seed):
    cfg = K.qwen3_30b_a3b(n_layer=c["layers"], n_vocab=c["vocab"], n_ctx=_n_ctx(c), rms_eps=EPS, rope_base=ROPE_BASE,
                          type_down=TYPES[c["down"]], type_head=TYPES[c["head"]])
    parts, size = [], 0
    for _, w in _model_tensors(c, seed):
        n = w.numel()
        parts.append(w.reshape(-1))
        size += n
        if n % 256:
            parts.append(torch.zeros(256 - n % 256, dtype=torch.uint8, device="cuda"))
            size += 256 - n % 256
    image = np.empty(size, np.uint8)
    at = 0
    for p in parts:
        torch.from_numpy(image[at:at + p.numel()]).copy_(p)
        at += p.numel()
    return K.Model.from_image(cfg, image)


def _history(c, seed, seq):
    """K and V of the slots before `pos`, f16 [layer][kv head][slot][dim] on the GPU."""
    g = _gen(seed, 5, seq)
    shape = (c["layers"], HEADS["n_head_kv"], _n_ctx(c), HEADS["head_dim"])
    kv = [torch.randn(shape, device="cuda", generator=g).to(torch.float16) for _ in range(2)]
    for t in kv:
        t[:, :, c["pos"]:] = 0
    return kv


def _ids(seed, n, vocab):
    return np.random.default_rng([seed, 6]).integers(0, vocab, n).astype(np.int32)


def _attn_inputs(c, seed):
    g = _gen(seed, 7)
    D, nh, nk = c["head_dim"], c["n_head"], c["n_head_kv"]
    s = dict(q=torch.randn((nh, D), device="cuda", generator=g), k=torch.randn((nk, D), device="cuda", generator=g),
             v=torch.randn((nk, D), device="cuda", generator=g), q_norm=_norm_weight(g, D), k_norm=_norm_weight(g, D))
    for name in ("k_cache", "v_cache"):
        t = torch.randn((nk, c["n_ctx"], D), device="cuda", generator=g).to(torch.float16)
        t[:, c["pos"]:] = 0
        s[name] = t
    return s


def _gemv_inputs(c, seed):
    g = _gen(seed, 8)
    return dict(w=_weight(g, c["type"], c["n_out"], c["n_in"]), x=torch.randn(c["n_in"], device="cuda", generator=g),
                norm=_norm_weight(g, c["n_in"]) if c["norm"] else None,
                resid=torch.randn(c["n_out"], device="cuda", generator=g) if c["resid"] else None)


def _moe_inputs(c, seed):
    n = c.get("n_tokens", 1)
    return dict(x=_tokens(_gen(seed, 9), n, c["n_embd"]),
                layers=[_moe_weights(_gen(seed, 10, i), c) for i in range(c.get("layers", 1))])


def prepare(case, seed):
    c, kind = case, case["kind"]
    K.open_device(0)
    if kind == "gemv":
        s = _gemv_inputs(c, seed)
        s["y"] = torch.empty(c["n_out"], device="cuda")
    elif kind in ("moe_token", "moe_batch"):
        s = _moe_inputs(c, seed)
        n, E, k = c.get("n_tokens", 1), c["n_expert"], c["k"]
        for w in s["layers"]:
            w["out"] = torch.empty((n, c["n_embd"]), device="cuda")
            w["logits"] = torch.empty((n, E), device="cuda")
            w["idx"] = torch.empty((n, k), dtype=torch.int32, device="cuda")
            w["w"] = torch.empty((n, k), device="cuda")
    elif kind == "attn":
        s = _attn_inputs(c, seed)
        s["out"] = torch.empty((c["n_head"], c["head_dim"]), device="cuda")
    else:
        m = _model(c, seed)
        s = dict(model=m)
        if kind == "batch":
            b = K.Batch(m, c["n_seq"], _n_ctx(c))
            for i in range(c["n_seq"]):
                b.kv_upload(i, *[t.cpu().numpy().view(np.uint16) for t in _history(c, seed, i)])
            s.update(batch=b, first=_ids(seed, c["n_seq"], c["vocab"]))
        else:
            if c["pos"]:
                m.kv_upload(*[t.cpu().numpy().view(np.uint16) for t in _history(c, seed, 0)])
            s["ids"] = _ids(seed, c.get("n", 1), c["vocab"])
    s["case"] = c
    torch.cuda.synchronize()
    return s


# ------------------------------------------------------------------ one pass

def _p(t):
    return None if t is None else t.data_ptr()


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "gemv":
        K.gemv(TYPES[c["type"]], _p(s["w"]), c["n_in"], c["n_out"], _p(s["x"]), _p(s["y"]), norm_w=_p(s["norm"]), eps=EPS,
               resid=_p(s["resid"]))
        return s["y"]
    if kind == "moe_token":
        x = s["x"]
        for w in s["layers"]:
            K.moe_decode_layer(_p(x), _p(w["router"]), _p(w["gate"]), _p(w["up"]), _p(w["down"]), c["n_embd"], c["n_ff"],
                               c["n_expert"], c["k"], _p(w["out"]), _p(w["logits"]), _p(w["idx"]), _p(w["w"]),
                               norm_w=_p(w["norm"]), eps=EPS, resid=_p(x), type_down=TYPES[c["down"]])
            x = w["out"]
        return [{n: w[n] for n in ("out", "logits", "idx", "w")} for w in s["layers"]]
    if kind == "moe_batch":
        w = s["layers"][0]
        K.moe_batch_layer(_p(s["x"]), _p(w["router"]), _p(w["gate"]), _p(w["up"]), _p(w["down"]), c["n_tokens"],
                          c["n_embd"], c["n_ff"], c["n_expert"], c["k"], _p(w["out"]), _p(w["logits"]), _p(w["idx"]),
                          _p(w["w"]), norm_w=_p(w["norm"]), eps=EPS, resid=_p(s["x"]), type_down=TYPES[c["down"]])
        return [{n: w[n] for n in ("out", "logits", "idx", "w")}]
    if kind == "attn":
        K.attention_step(_p(s["q"]), _p(s["k"]), _p(s["v"]), _p(s["q_norm"]), _p(s["k_norm"]), EPS, ROPE_BASE, c["pos"],
                         c["n_head"], c["n_head_kv"], c["head_dim"], c["n_ctx"], _p(s["k_cache"]), _p(s["v_cache"]),
                         _p(s["out"]))
        return {n: s[n] for n in ("out", "k_cache", "v_cache")}
    if kind == "decode":
        m = s["model"]
        m.set_pos(c["pos"])
        tokens = m.decode_greedy(int(s["ids"][0]), c["steps"])
        return {"tokens": tokens, "logits": m.logits()}
    if kind == "prompt":
        m = s["model"]
        m.set_pos(c["pos"])
        return {"logits": m.forward(s["ids"])}
    b = s["batch"]
    b.set_pos(c["pos"])
    tokens = b.decode_greedy(s["first"], c["steps"] - 1)
    return {"tokens": tokens, "logits": b.forward(tokens[-1])}


# ------------------------------------------------------------------ what a pass cannot do without

def _distinct(n_tokens, c):
    """Experts that n_tokens tokens reach when routing is even."""
    return c["n_expert"] * (1.0 - (1.0 - c["k"] / c["n_expert"]) ** n_tokens)


def _moe_work(n, c):
    H, F, E, k = c["n_embd"], c["n_ff"], c["n_expert"], c["k"]
    expert = 2 * _row_bytes("q4_k", H) * F + _row_bytes(c["down"], F) * H
    return (_distinct(n, c) * expert + 4 * E * H + n * (12 * H + 4 * E + 8 * k),
            2.0 * n * (E * H + 3 * k * H * F))


def work(case):
    c, kind = case, case["kind"]
    if kind == "gemv":
        rb = _row_bytes(c["type"], c["n_in"])
        return dict(bytes=rb * c["n_out"] + 4 * (c["n_in"] * (1 + c["norm"]) + c["n_out"] * (1 + c["resid"])),
                    flops=2.0 * c["n_in"] * c["n_out"])
    if kind in ("moe_token", "moe_batch"):
        b, f = _moe_work(c.get("n_tokens", 1), c)
        layers = c.get("layers", 1)
        return dict(bytes=b * layers, flops=f * layers)
    if kind == "attn":
        D = c["head_dim"]
        return dict(bytes=4 * D * c["n_head_kv"] * (c["pos"] + 1) + 4 * D * (2 * c["n_head"] + 2 * c["n_head_kv"]),
                    flops=4.0 * c["n_head"] * D * (c["pos"] + 1))
    m = _model_shape(c)
    H, QD, KVD = m["n_embd"], m["n_head"] * m["head_dim"], m["n_head_kv"] * m["head_dim"]
    attn_w = _row_bytes("q4_k", H) * (QD + 2 * KVD) + _row_bytes("q4_k", QD) * H
    attn_f = 2.0 * (H * (QD + 2 * KVD) + QD * H)
    head_w, head_f = _row_bytes(m["head"], H) * m["vocab"], 2.0 * H * m["vocab"]
    if kind == "prompt":
        n, rows = c["n"], 1
        slots = n * c["pos"] + n * (n + 1) // 2
        kv = 4 * KVD * (c["pos"] + 2 * n)
        passes = 1
    else:
        n = rows = c.get("n_seq", 1)
        slots = n * (c["pos"] + c["steps"] // 2)
        kv = 4 * KVD * slots
        passes = c["steps"]
    moe_b, moe_f = _moe_work(n, m)
    return dict(bytes=passes * (m["layers"] * (attn_w + kv + moe_b) + head_w + 2 * H * n + 4 * rows * m["vocab"]),
                flops=passes * (m["layers"] * (n * attn_f + moe_f + 4.0 * QD * slots) + rows * head_f))


def tolerance(case):
    kind = case["kind"]
    if kind == "gemv":
        return {"rel": 5e-6}
    if kind in ("moe_token", "moe_batch"):
        # a near-tie of two router logits may swap two experts
        return {"rel": 1e-5, "max": 1e-3, "differ": 2e-3}
    if kind == "attn":
        # the appended key and value are rounded to f16: a last-bit difference flips one
        return {"rel": 1e-5, "max": 2e-3}
    # f16 cache slots flip by one ulp on last-bit differences, in every layer
    return {"rel": 4e-4, "max": 4e-3, "differ": 1e-2}


# ------------------------------------------------------------------ the same in float64

def _dequant(t, w, n_in):
    """Weights [rows][n_in] in float64 from their bytes."""
    if t in ("bf16", "f32"):
        return w.view(torch.bfloat16 if t == "bf16" else torch.float32).reshape(-1, n_in).double()
    nb = n_in // 256
    w = w.reshape(-1, nb, 144 if t == "q4_k" else 210)
    rows = w.shape[0]

    def f16(a):
        return a.contiguous().view(torch.float16).double()

    if t == "q4_k":
        s = w[..., 4:16]
        sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], dim=-1)
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], dim=-1)
        qs = w[..., 16:].reshape(rows, nb, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], dim=3).reshape(rows, nb, 8, 32).double()
        v = (f16(w[..., 0:2]) * sc)[..., None] * q - (f16(w[..., 2:4]) * mn)[..., None]
        return v.reshape(rows, n_in)
    ql = w[..., :128].reshape(rows, nb, 2, 2, 32)
    qh = w[..., 128:192].reshape(rows, nb, 2, 32)
    q = torch.stack([(ql[..., t & 1, :] >> (4 * (t >> 1)) & 15) | ((qh >> (2 * t) & 3) << 4) for t in range(4)], dim=3)
    sc = w[..., 192:208].contiguous().view(torch.int8).double() * f16(w[..., 208:210])
    v = (q.double() - 32).reshape(rows, nb, 16, 16) * sc[..., None]
    return v.reshape(rows, n_in)


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _moe64(x, w, c):
    """One MoE layer over rows x (float64): its outputs, and the rows plus the experts' sum."""
    H, F, E, k = c["n_embd"], c["n_ff"], c["n_expert"], c["k"]
    h = _rms(x, w["norm"])
    logits = h @ _dequant("f32", w["router"], H).T
    p = torch.softmax(logits, -1)
    order = torch.sort(p, dim=-1, descending=True, stable=True)
    idx, top = order.indices[:, :k], order.values[:, :k]
    top = top / top.sum(-1, keepdim=True)
    out = x.clone()
    for e in torch.unique(idx).tolist():
        t, j = (idx == e).nonzero(as_tuple=True)
        a = h[t]
        gate = a @ _dequant("q4_k", w["gate"][e * F:(e + 1) * F], H).T
        up = a @ _dequant("q4_k", w["up"][e * F:(e + 1) * F], H).T
        y = (gate * torch.sigmoid(gate) * up) @ _dequant(c["down"], w["down"][e * H:(e + 1) * H], F).T
        out[t] += top[t, j, None] * y
    return dict(out=out, logits=logits, idx=idx.to(torch.int32), w=top)


def _rope_tables(pos, D):
    """cos and sin [n][D/2] of positions `pos`: the angle is a float32 product, as the path defines it."""
    inv = np.power(ROPE_BASE, -2.0 * np.arange(D // 2) / D).astype(np.float32)
    th = np.asarray(pos, np.float32)[:, None] * inv[None, :]
    th = torch.from_numpy(th.astype(np.float64)).cuda()
    return torch.cos(th), torch.sin(th)


def _rope(x, cos, sin):
    """Rows x [n][heads][D] rotated in pairs (i, i + D/2)."""
    a, b = x.chunk(2, dim=-1)
    cos, sin = cos[:, None, :], sin[:, None, :]
    return torch.cat([a * cos - b * sin, a * sin + b * cos], dim=-1)


def _attend(q, kc, vc, n_slots):
    """q [heads][D] over the first n_slots of caches [kv heads][slots][D]."""
    nk, D = kc.shape[0], q.shape[-1]
    G = q.shape[0] // nk
    out = torch.empty_like(q)
    for h in range(nk):
        kk, vv = kc[h, :n_slots].double(), vc[h, :n_slots].double()
        a = torch.softmax(q[h * G:(h + 1) * G] @ kk.T / math.sqrt(D), -1)
        out[h * G:(h + 1) * G] = a @ vv
    return out


def _attn64(q, k, v, q_norm, k_norm, pos, kc, vc):
    """Attention of rows at positions pos.. (q [n][heads][D]); the caches take every row's K and V in f16."""
    n = q.shape[0]
    cos, sin = _rope_tables(range(pos, pos + n), q.shape[-1])
    q, k = _rope(_rms(q, q_norm), cos, sin), _rope(_rms(k, k_norm), cos, sin)
    kc[:, pos:pos + n] = k.transpose(0, 1).to(torch.float16)
    vc[:, pos:pos + n] = v.transpose(0, 1).to(torch.float16)
    if n == 1:
        return _attend(q[0], kc, vc, pos + 1)[None]
    nk, D = kc.shape[0], q.shape[-1]
    G = q.shape[1] // nk
    out = torch.empty_like(q)
    seen = torch.arange(pos + n, device="cuda")[None, :] <= torch.arange(pos, pos + n, device="cuda")[:, None]
    for h in range(q.shape[1]):
        s = q[:, h] @ kc[h // G, :pos + n].double().T / math.sqrt(D)
        out[:, h] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ vc[h // G, :pos + n].double()
    return out


class _Exact:
    """A whole model in float64: rows of several sequences, each with its own cache."""

    def __init__(self, c, seed):
        self.c, self.m = c, _model_shape(c)
        self.layers, self.t = [], {}
        for name, w in _model_tensors(c, seed):
            if name in ("embd", "out_norm", "head"):
                self.t[name] = w
            else:
                if name == "attn_norm":
                    self.layers.append({})
                self.layers[-1][name] = w
        self.kv = [_history(c, seed, i) for i in range(c.get("n_seq", 1))]

    def forward(self, tokens, pos):
        """tokens [sequences][rows]; logits of every sequence's last row."""
        m, H = self.m, self.m["n_embd"]
        ids = torch.as_tensor(np.asarray(tokens, np.int64), device="cuda")
        n_seq, rows = ids.shape
        x = self.t["embd"].view(torch.bfloat16).reshape(-1, H)[ids.reshape(-1)].double()
        nh, nk, D = m["n_head"], m["n_head_kv"], m["head_dim"]
        for il, w in enumerate(self.layers):
            h = _rms(x, w["attn_norm"].view(torch.float32))
            qkv = (h @ _dequant("q4_k", w["wqkv"], H).T).reshape(n_seq, rows, nh + 2 * nk, D)
            ctx = [_attn64(qkv[i, :, :nh], qkv[i, :, nh:nh + nk], qkv[i, :, nh + nk:], w["q_norm"].view(torch.float32),
                           w["k_norm"].view(torch.float32), pos, self.kv[i][0][il], self.kv[i][1][il])
                   for i in range(n_seq)]
            x = x + torch.cat(ctx).reshape(n_seq * rows, nh * D) @ _dequant("q4_k", w["wo"], nh * D).T
            x = _moe64(x, dict(w, norm=w["ffn_norm"].view(torch.float32)), m)["out"]
        last = _rms(x.reshape(n_seq, rows, H)[:, -1], self.t["out_norm"].view(torch.float32))
        return last @ _dequant(m["head"], self.t["head"], H).T


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "gemv":
        s = _gemv_inputs(c, seed)
        x = s["x"].double()
        if s["norm"] is not None:
            x = _rms(x, s["norm"])
        step = max(1, (1 << 28) // c["n_in"])
        y = torch.cat([_dequant(c["type"], s["w"][i:i + step], c["n_in"]) @ x for i in range(0, c["n_out"], step)])
        return y if s["resid"] is None else y + s["resid"].double()
    if kind in ("moe_token", "moe_batch"):
        s = _moe_inputs(c, seed)
        x, out = s["x"].double(), []
        for w in s["layers"]:
            out.append(_moe64(x, w, c))
            x = out[-1]["out"]
        return out
    if kind == "attn":
        s = _attn_inputs(c, seed)
        kc, vc = s["k_cache"], s["v_cache"]
        out = _attn64(s["q"].double()[None], s["k"].double()[None], s["v"].double()[None], s["q_norm"], s["k_norm"],
                      c["pos"], kc, vc)
        return dict(out=out[0], k_cache=kc.double(), v_cache=vc.double())
    x = _Exact(c, seed)
    if kind == "prompt":
        return {"logits": x.forward([_ids(seed, c["n"], c["vocab"])], c["pos"])[0]}
    n_seq = c.get("n_seq", 1)
    t, tokens = _ids(seed, n_seq, c["vocab"]), []
    for i in range(c["steps"]):
        logits = x.forward(t[:, None], c["pos"] + i)
        t = logits.argmax(-1).cpu().numpy().astype(np.int32)
        tokens.append(t)
    if kind == "decode":
        return {"tokens": np.concatenate(tokens), "logits": logits[0]}
    return {"tokens": np.stack(tokens[:-1]), "logits": logits}
