"""What this library's users have it compute, as measurable cases.

A case is one call (or the few calls that belong together) through the public
entry points of llm_core_amd: the quantized products of a decode step, of
multi-sequence decode and of a prefill, the two attentions, a decoder step and
whole generations.  listed() gives one of each at the sizes of this
repository's benchmark and model shapes; draw() gives more over the ranges they
stand for, ragged and odd sizes included.

Weights are N(0, 0.02) in GGUF blocks, activations N(0, 1), all made on the GPU
from the seed.  exact() restates each case in 64-bit torch.
"""
import math
import types

import numpy as np
import torch

from llm_core_amd import hip
from llm_core_amd.model import Hparams, LlamaHip

DEV = "cuda"
F32, F16, Q5_0, Q8_0, Q4_K, Q6_K = 0, 1, 6, 8, 12, 14
TYPES = {"f16": F16, "q5_0": Q5_0, "q8_0": Q8_0, "q4_k": Q4_K, "q6_k": Q6_K}
BITS = {F16: 16.0, Q5_0: 5.5, Q8_0: 8.5, Q4_K: 4.5, Q6_K: 6.5625}
K_QUANTS = (Q4_K, Q6_K)

_ctx = None


def _context():
    """The program's one device context (one in-order stream), as the decoder keeps it."""
    global _ctx
    if _ctx is None:
        _ctx = hip.Context(0)
    return _ctx


# --------------------------------------------------------------------------- cases


def listed():
    return [
        # the smallest product of a decode step: the key projection of a hidden-2048
        # layer with 2 KV heads; two launches, so latency is all there is
        {"name": "matmul k-proj T1", "op": "matmul", "type": "q4_k", "act": "q8", "rows": 256,
         "cols": 2048, "tokens": 1},
        # Q4_K times fp32 activations, batch 1 (benchmark config 1)
        {"name": "matmul f32 T1", "op": "matmul", "type": "q4_k", "act": "f32", "rows": 4096,
         "cols": 4096, "tokens": 1},
        # output head of a 151936-token vocabulary and the greedy pick (config 2)
        {"name": "head 151936 greedy", "op": "head", "type": "q6_k", "rows": 151936, "cols": 2048},
        # FFN up projection for 16 sequences decoded together (config 4)
        {"name": "matmul ffn T16", "op": "matmul", "type": "q4_k", "act": "q8", "rows": 11008,
         "cols": 4096, "tokens": 16},
        # FFN down projection of a short prompt or of 64 sequences
        {"name": "matmul down T64", "op": "matmul", "type": "q6_k", "act": "q8", "rows": 4096,
         "cols": 11008, "tokens": 64},
        # FFN up projection of one whole prefill chunk
        {"name": "matmul ffn T512", "op": "matmul", "type": "q4_k", "act": "q8", "rows": 11008,
         "cols": 4096, "tokens": 512},
        # the 32-block types' prefill product (hidden 896 is no multiple of 256), ragged tokens
        {"name": "matmul q5_0 T200", "op": "matmul", "type": "q5_0", "act": "f32", "rows": 4864,
         "cols": 896, "tokens": 200},
        # one decoded token's attention over an odd, grown cache with shared KV heads
        {"name": "attn decode 3005", "op": "attn_decode", "heads": 32, "kv_heads": 8,
         "head_dim": 128, "seq": 3005},
        # the last chunk of a 2048-token prompt
        {"name": "attn prefill 512@1536", "op": "attn_prefill", "heads": 32, "kv_heads": 32,
         "head_dim": 128, "tokens": 512, "pos": 1536},
        # one layer's decode step at position 1024, hidden 2048, 16/2 heads (config 3): a
        # caller that picks its own tokens reads the logits of every step
        {"name": "step 2048 @1024", "op": "step", "layers": 1, "embd": 2048, "heads": 16,
         "kv_heads": 2, "ffn": 11008, "vocab": 512, "ctx": 1088, "pos": 1024, "mix": "k",
         "theta": 1e6, "bias": False},
        # 512-token prompt and 128 greedy tokens at the 4096-wide shape (config 5), 2 of its layers
        {"name": "greedy 4096 512+128", "op": "generate", "layers": 2, "embd": 4096, "heads": 32,
         "kv_heads": 32, "ffn": 11008, "vocab": 32000, "ctx": 2048, "prompt": 512, "gen": 128,
         "mix": "k", "sampled": False, "theta": 1e4, "bias": False},
        # a sampled answer of the 896-wide shape (14/2 heads, biases, the fallback types of that
        # width), 4 of its layers: penalty, top-k and top-p on every token
        {"name": "sampled 896 200+64", "op": "generate", "layers": 4, "embd": 896, "heads": 14,
         "kv_heads": 2, "ffn": 4864, "vocab": 151936, "ctx": 1024, "prompt": 200, "gen": 64,
         "mix": "fallback", "sampled": True, "theta": 1e6, "bias": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["matmul", "matmul", "matmul", "matmul", "head", "attn_decode", "attn_prefill",
                     "step", "generate", "generate"])
    if op == "matmul":
        t = rng.choice(["q4_k", "q4_k", "q4_k", "q6_k", "q6_k", "q5_0", "q8_0", "f16"])
        k_quant = t in ("q4_k", "q6_k")
        cols = 256 * _log(rng, 2, 43) if k_quant else 32 * _log(rng, 8, 160)
        tokens = 1 if rng.random() < 0.3 else _log(rng, 2, 640)
        act = "q8" if k_quant and (tokens > 1 or rng.random() < 0.7) else "f32"
        if act == "f32" and k_quant:  # one token; its fp32 row is staged whole
            cols = 256 * _log(rng, 2, 43)
        rows = _log(rng, 128, 14000)
        if rng.random() < 0.5:  # half of all matrices have the usual whole row tiles
            rows = max(128, rows // 128 * 128)
        return {"op": op, "type": t, "act": act, "rows": rows, "cols": cols, "tokens": tokens}
    if op == "head":
        return {"op": op, "type": rng.choice(["q6_k", "q6_k", "q4_k"]),
                "rows": _log(rng, 8000, 152000), "cols": 256 * rng.randint(4, 16)}
    head_dim = rng.choice([64, 128, 128])
    group = rng.choice([1, 1, 2, 4, 7, 8])
    kv_heads = rng.choice([2, 4, 8])
    if op == "attn_decode":
        return {"op": op, "heads": kv_heads * group, "kv_heads": kv_heads, "head_dim": head_dim,
                "seq": _log(rng, 16, 12000)}
    if op == "attn_prefill":
        return {"op": op, "heads": kv_heads * group, "kv_heads": kv_heads, "head_dim": head_dim,
                "tokens": _log(rng, 2, 512), "pos": rng.choice([0, rng.randint(1, 2500)])}
    # models: hidden sizes with head_dim 64 or 128, up to 8 query heads per KV head
    embd, heads, kv, ffn, mix = rng.choice([
        (896, 14, 2, 4864, "fallback"), (1024, 16, 8, 2816, "k"), (1536, 12, 2, 8960, "k"),
        (2048, 16, 2, 11008, "k"), (2048, 32, 8, 5632, "k"), (2304, 18, 18, 5888, "k"),
        (3072, 24, 8, 8192, "k"), (4096, 32, 8, 11008, "k")])
    vocab = rng.choice([4099, 32000, 32003])
    theta = rng.choice([1e4, 1e6])
    c = {"op": op, "layers": rng.randint(1, 2), "embd": embd, "heads": heads, "kv_heads": kv,
         "ffn": ffn, "vocab": vocab, "mix": mix, "theta": theta, "bias": rng.random() < 0.5}
    if op == "step":
        pos = _log(rng, 4, 2000)
        return dict(c, ctx=pos + 64, pos=pos)
    prompt, gen = _log(rng, 1, 600), _log(rng, 16, 128)
    return dict(c, ctx=prompt + gen + rng.randint(0, 900), prompt=prompt, gen=gen,
                sampled=rng.random() < 0.4)


# --------------------------------------------------------------------------- GGUF blocks


class _Draws:
    """Normal draws on the GPU, each call another stream of the same seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed) * 7919 + 17)

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.g, device=DEV) * std + mean

    def ints(self, n, high):
        return torch.randint(0, high, (n,), generator=self.g, device=DEV)


def _bytes(t):
    return t.contiguous().view(torch.uint8)


def _quantize(x, qtype):
    """fp32 [rows, cols] as GGUF rows: uint8 [rows, row bytes]."""
    rows, cols = x.shape
    if qtype == F16:
        return _bytes(x.to(torch.float16)).reshape(rows, -1)
    if qtype == Q8_0:
        b = x.reshape(rows, cols // 32, 32)
        d = (b.abs().amax(2) / 127).to(torch.float16)
        q = torch.round(b / d.float().clamp_min(1e-12)[..., None]).clamp(-127, 127).to(torch.int8)
        return torch.cat([_bytes(d[..., None]), _bytes(q)], 2).reshape(rows, -1)
    if qtype == Q5_0:
        b = x.reshape(rows, cols // 32, 32)
        m = b.gather(2, b.abs().argmax(2, keepdim=True))
        d = (m[..., 0] / -16).to(torch.float16)
        df = d.float()[..., None]
        q = torch.floor(b / torch.where(df == 0, 1, df) + 16.5).clamp(0, 31).to(torch.int32)
        qs = (q[..., :16] & 15) | ((q[..., 16:] & 15) << 4)
        at = torch.arange(32, device=x.device)
        qh = ((q >> 4).to(torch.int64) << at).sum(2, keepdim=True)
        qh = torch.cat([(qh >> s) & 255 for s in (0, 8, 16, 24)], 2)
        return torch.cat([_bytes(d[..., None]), qh.to(torch.uint8), qs.to(torch.uint8)],
                         2).reshape(rows, -1)
    out = torch.empty(rows, cols // 256 * (144 if qtype == Q4_K else 210), dtype=torch.uint8,
                      device=x.device)
    step = max(1, (1 << 26) // cols)
    for r in range(0, rows, step):
        b = x[r:r + step].reshape(-1, 256)
        out[r:r + step] = (_q4_k if qtype == Q4_K else _q6_k)(b).reshape(-1, out.shape[1])
    return out


def _q4_k(b):
    s = b.reshape(-1, 8, 32)
    m = (-s.amin(2)).clamp_min(0)
    scale = (s.amax(2) + m) / 15
    d = (scale.amax(1, keepdim=True) / 63).to(torch.float16)
    dm = (m.amax(1, keepdim=True) / 63).to(torch.float16)
    df, dmf = d.float().clamp_min(1e-12), dm.float().clamp_min(1e-12)
    sc = torch.round(scale / df).clamp(0, 63).to(torch.int32)
    mn = torch.round(m / dmf).clamp(0, 63).to(torch.int32)
    step = (df * sc).clamp_min(1e-12)[..., None]
    q = torch.round((s + (dmf * mn)[..., None]) / step).clamp(0, 15).to(torch.int32)
    packed = torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), mn[:, :4] | ((mn[:, 4:] >> 4) << 6),
                        (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)
    q = q.reshape(-1, 4, 2, 32)
    qs = (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(-1, 128)
    return torch.cat([_bytes(d), _bytes(dm), packed.to(torch.uint8), qs.to(torch.uint8)], 1)


def _q6_k(b):
    s = b.reshape(-1, 16, 16)
    scale = s.abs().amax(2) / 31
    d = (scale.amax(1, keepdim=True) / 127).to(torch.float16)
    df = d.float().clamp_min(1e-12)
    sc = torch.round(scale / df).clamp(0, 127)
    q = torch.round(s / (df * sc).clamp_min(1e-12)[..., None]).clamp(-32, 31).to(torch.int32) + 32
    q = q.reshape(-1, 2, 4, 32)  # half, quarter, weight
    ql = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4),
                    (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2).reshape(-1, 128)
    h = q >> 4
    qh = (h[:, :, 0] | (h[:, :, 1] << 2) | (h[:, :, 2] << 4) | (h[:, :, 3] << 6)).reshape(-1, 64)
    return torch.cat([ql.to(torch.uint8), qh.to(torch.uint8), _bytes(sc.to(torch.int8)), _bytes(d)],
                     1)


def _weights64(w, qtype, cols):
    """GGUF rows (uint8) as float64 [rows, cols]."""
    rows = w.shape[0]

    def half(t):
        return t.contiguous().view(torch.float16).double()

    if qtype == F16:
        return half(w).reshape(rows, cols)
    if qtype == Q8_0:
        b = w.reshape(rows, cols // 32, 34)
        return (half(b[..., :2]) * b[..., 2:].contiguous().view(torch.int8).double()).reshape(rows, cols)
    if qtype == Q5_0:
        b = w.reshape(rows, cols // 32, 22)
        n = b.to(torch.int64)
        qh = n[..., 2:3] | (n[..., 3:4] << 8) | (n[..., 4:5] << 16) | (n[..., 5:6] << 24)
        bit = (qh >> torch.arange(32, device=w.device)) & 1
        q = torch.cat([n[..., 6:] & 15, n[..., 6:] >> 4], 2) | (bit << 4)
        return (half(b[..., :2]) * (q - 16).double()).reshape(rows, cols)
    if qtype == Q4_K:
        b = w.reshape(-1, 144)
        n = b.to(torch.int16)
        a, m, z = n[:, 4:8], n[:, 8:12], n[:, 12:16]
        sc = torch.cat([a & 63, (z & 15) | ((a >> 6) << 4)], 1).double()
        mn = torch.cat([m & 63, (z >> 4) | ((m >> 6) << 4)], 1).double()
        qs = n[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
        v = (half(b[:, 0:2]) * sc)[..., None] * q - (half(b[:, 2:4]) * mn)[..., None]
        return v.reshape(rows, cols)
    b = w.reshape(-1, 210)
    ql = b[:, :128].to(torch.int16).reshape(-1, 2, 64)
    qh = b[:, 128:192].to(torch.int16).reshape(-1, 2, 1, 32)
    lo = torch.stack([ql[..., :32] & 15, ql[..., 32:] & 15, ql[..., :32] >> 4, ql[..., 32:] >> 4], 2)
    hi = torch.cat([qh & 3, (qh >> 2) & 3, (qh >> 4) & 3, (qh >> 6) & 3], 2)
    q = ((lo | (hi << 4)) - 32).reshape(-1, 16, 16).double()
    sc = b[:, 192:208].contiguous().view(torch.int8).double()
    return (half(b[:, 208:210])[..., None] * sc[..., None] * q).reshape(rows, cols)


def _product64(x, w, qtype, cols):
    """float64 x [T, cols] times the rows of w, a slice of rows at a time."""
    step = max(1, (1 << 27) // cols)
    return torch.cat([x @ _weights64(w[r:r + step], qtype, cols).T
                      for r in range(0, w.shape[0], step)], 1)


def _q8_64(x):
    """x rounded to Q8_0 blocks of 32 (scale max|x| / 127), as values.  The whole
    numbers are picked as the format does, from 32-bit products x * (127 / max|x|):
    which side a tie falls to is no matter of precision."""
    b = x.reshape(-1, 32)
    most = b.abs().amax(1, keepdim=True)
    m = most.float().clamp_min(1e-30)
    q = torch.round(b.float() * torch.div(torch.full_like(m, 127.0), m))
    return (q.double() * (most / 127)).reshape(x.shape)


# --------------------------------------------------------------------------- models


def _types(case):
    """Weight type of each matrix: the Q4_K_M mix, or its fallbacks where the
    hidden size is no multiple of 256."""
    if case["mix"] == "k":
        t = {"q": Q4_K, "k": Q4_K, "v": Q6_K, "output": Q4_K, "gate": Q4_K, "up": Q4_K, "down": Q6_K}
        return t, Q4_K, Q6_K
    t = {"q": Q5_0, "k": Q5_0, "v": Q8_0, "output": Q5_0, "gate": Q5_0, "up": Q5_0, "down": Q6_K}
    return t, Q8_0, Q8_0


def _shapes(case):
    e, f = case["embd"], case["ffn"]
    kv = e // case["heads"] * case["kv_heads"]
    return {"q": (e, e), "k": (kv, e), "v": (kv, e), "output": (e, e), "gate": (f, e),
            "up": (f, e), "down": (e, f)}


def _shift(case):
    """Each token's confident successor is this much further round the vocabulary."""
    v = case["vocab"]
    return next(s for s in range(v // 3 + 1, v) if math.gcd(s, v) == 1)


def _tensors(case, r):
    """GGUF name -> (type, uint8 or float rows on the GPU).  The head's rows are the
    embeddings of the token before each, so that the pick is as clear as a
    trained model's and does not hang on the last bit of a logit."""
    t, emb_type, head_type = _types(case)
    e, v = case["embd"], case["vocab"]
    emb = r.normal(v, e)
    out = {"token_embd.weight": (emb_type, _quantize(emb, emb_type))}
    out["output.weight"] = (head_type, _quantize(emb.roll(_shift(case), 0) * 0.04, head_type))
    del emb
    out["output_norm.weight"] = (F32, r.normal(e, std=0.05, mean=1.0))
    for l in range(case["layers"]):
        b = "blk.%d." % l
        for n in ("attn_norm", "ffn_norm"):
            out[b + n + ".weight"] = (F32, r.normal(e, std=0.05, mean=1.0))
        for k, (rows, cols) in _shapes(case).items():
            name = b + ("attn_" if k in ("q", "k", "v", "output") else "ffn_") + k
            out[name + ".weight"] = (t[k], _quantize(r.normal(rows, cols, std=0.02), t[k]))
            if case["bias"] and k in ("q", "k", "v"):
                out[name + ".bias"] = (F32, r.normal(rows, std=0.02))
    return out


def _kv_rows(case, r):
    kv = case["embd"] // case["heads"] * case["kv_heads"]
    return [(r.normal(case["pos"], kv), r.normal(case["pos"], kv)) for _ in range(case["layers"])]


def _hparams(case):
    return Hparams(n_layer=case["layers"], n_embd=case["embd"], n_heads=case["heads"],
                   n_kv_heads=case["kv_heads"], ffn_dim=case["ffn"], n_vocab=case["vocab"],
                   n_ctx=case["ctx"], rms_eps=1e-6, rope_theta=case["theta"])


class _Model:
    """A loaded decoder that gives its device memory back with the state."""

    def __init__(self, case, tensors):
        host = {n: (t, w.cpu().numpy().reshape(-1)) for n, (t, w) in tensors.items()}
        self.dec = LlamaHip(_context(), types.SimpleNamespace(hp=_hparams(case), tensors=host))

    def __del__(self):
        dec = getattr(self, "dec", None)
        if dec is not None:
            dec.close()


def _rope64(x, pos, theta):
    """Rotate-half RoPE of x [T, heads, head_dim] at positions pos [T]."""
    half = x.shape[2] // 2
    freq = theta ** (-torch.arange(half, device=x.device, dtype=torch.float64) * 2 / x.shape[2])
    a = pos.double()[:, None, None] * freq
    c, s = a.cos(), a.sin()
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat([lo * c - hi * s, hi * c + lo * s], 2)


def _attention64(q, k, v, pos0):
    """Causal attention of q [T, heads, hd] at positions pos0.. over k, v [n, kv_heads, hd]."""
    t, heads, hd = q.shape
    group = heads // k.shape[1]
    hidden = torch.arange(k.shape[0], device=q.device)[None, :] > torch.arange(t, device=q.device)[:, None] + pos0
    out = torch.empty_like(q)
    for h in range(heads):
        s = q[:, h] @ k[:, h // group].T / math.sqrt(hd)
        out[:, h] = torch.softmax(s.masked_fill(hidden, -math.inf), 1) @ v[:, h // group]
    return out


def _forward64(case, w, tokens, pos0, n_batch, cache=None):
    """The last row's logits for `tokens` at positions pos0.., the first n_batch of them as one
    prefill batch and the others one by one.  The two differ for Q8_0 matrices only: a batch gives
    them its fp32 rows, a single token its Q8_0 blocks.  cache: K, V rows before pos0."""
    e, heads, kvh = case["embd"], case["heads"], case["kv_heads"]
    hd, t = e // heads, len(tokens)
    pos = torch.arange(pos0, pos0 + t, device=DEV)
    batch = (torch.arange(t, device=DEV) < n_batch)[:, None]

    def norm(x, name):
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-6) * w[name][1].double()

    def times(x, name, rows=None):
        qt, m = w[name + ".weight"]
        if qt in K_QUANTS:
            x = _q8_64(x)
        elif qt == Q8_0:
            x = torch.where(batch if rows is None else rows, x, _q8_64(x))
        y = _product64(x, m, qt, x.shape[1])
        return y + w[name + ".bias"][1].double() if name + ".bias" in w else y

    qt, emb = w["token_embd.weight"]
    x = _weights64(emb[tokens], qt, e)
    for l in range(case["layers"]):
        b = "blk.%d." % l
        n = norm(x, b + "attn_norm.weight")
        q = _rope64(times(n, b + "attn_q").reshape(t, heads, hd), pos, case["theta"])
        k = _rope64(times(n, b + "attn_k").reshape(t, kvh, hd), pos, case["theta"])
        v = times(n, b + "attn_v").reshape(t, kvh, hd)
        if cache is not None:
            k = torch.cat([cache[l][0].double().reshape(-1, kvh, hd), k])
            v = torch.cat([cache[l][1].double().reshape(-1, kvh, hd), v])
        x = x + times(_attention64(q, k, v, pos0).reshape(t, e), b + "attn_output")
        n = norm(x, b + "ffn_norm.weight")
        g = times(n, b + "ffn_gate")
        x = x + times(g * torch.sigmoid(g) * times(n, b + "ffn_up"), b + "ffn_down")
    # the head takes one row, whichever way it came
    return times(norm(x[-1:], "output_norm.weight"), "output",
                 torch.zeros(1, 1, dtype=torch.bool, device=DEV))[0]


def _prompt(case, r):
    return r.ints(case["prompt"], case["vocab"])


# --------------------------------------------------------------------------- inputs


def _tables(positions, head_dim, theta=10000.0):
    freq = theta ** (-torch.arange(head_dim // 2, device=DEV, dtype=torch.float64) * 2 / head_dim)
    a = torch.arange(positions, device=DEV, dtype=torch.float64)[:, None] * freq
    return a.cos().float(), a.sin().float()


def _inputs(case, seed):
    """Everything a case is given, on the GPU."""
    r, op = _Draws(seed), case["op"]
    if op in ("matmul", "head"):
        qt = TYPES[case["type"]]
        return {"w": _quantize(r.normal(case["rows"], case["cols"], std=0.02), qt),
                "x": r.normal(case.get("tokens", 1), case["cols"])}
    if op in ("attn_decode", "attn_prefill"):
        n = case["seq"] if op == "attn_decode" else case["pos"] + case["tokens"]
        hd = case["head_dim"]
        i = {"q": r.normal(case.get("tokens", 1), case["heads"] * hd),
             "k": r.normal(n, case["kv_heads"] * hd), "v": r.normal(n, case["kv_heads"] * hd)}
        if op == "attn_prefill":
            i["cos"], i["sin"] = _tables(n, hd)
        return i
    i = {"tensors": _tensors(case, r)}
    if op == "step":
        i["token"], i["kv"] = int(r.ints(1, case["vocab"])[0]), _kv_rows(case, r)
    else:
        i["prompt"] = _prompt(case, r)
    return i


def prepare(case, seed):
    i, op = _inputs(case, seed), case["op"]
    s = {"case": case, "ctx": _context()}
    if op in ("matmul", "head"):
        t = case.get("tokens", 1)
        s.update(i, y=torch.zeros(t, case["rows"], device=DEV), qtype=TYPES[case["type"]],
                 row_bytes=hip.row_bytes(TYPES[case["type"]], case["cols"]),
                 xq8=torch.zeros(t * (case["cols"] // 32) * hip.Q8_0_BYTES, dtype=torch.uint8,
                                 device=DEV))
        if op == "head":
            s["token"] = torch.zeros(1, dtype=torch.int32, device=DEV)
    elif op in ("attn_decode", "attn_prefill"):
        n = case["heads"] * case["head_dim"]
        t = case.get("tokens", 1)
        s.update(i, y=torch.zeros(t, n, device=DEV),
                 yq8=torch.zeros(t * (n // 32) * hip.Q8_0_BYTES, dtype=torch.uint8, device=DEV))
    else:
        s["model"] = _Model(case, i["tensors"])
        if op == "step":
            s["token"] = i["token"]
            for l, (k, v) in enumerate(i["kv"]):
                s["model"].dec.set_kv(l, k.cpu().numpy(), v.cpu().numpy(), case["pos"])
        else:
            s["prompt"] = i["prompt"].cpu().numpy().astype(np.int32)
    torch.cuda.synchronize()
    return s


# --------------------------------------------------------------------------- one pass


def run(s):
    case, ctx = s["case"], s["ctx"]
    op = case["op"]
    if op == "matmul":
        return _run_matmul(s, case, ctx)
    if op == "head":
        rows, cols = case["rows"], case["cols"]
        ctx.gemv_f32(s["qtype"], s["y"].data_ptr(), s["w"].data_ptr(), s["x"].data_ptr(), rows, cols,
                     s["row_bytes"])
        ctx.argmax(s["token"].data_ptr(), s["y"].data_ptr(), rows)
        return s["y"], s["token"]
    if op == "attn_decode":
        ctx.attn_decode(s["y"].data_ptr(), s["yq8"].data_ptr(), s["q"].data_ptr(), s["k"].data_ptr(),
                        s["v"].data_ptr(), case["seq"], case["heads"], case["kv_heads"],
                        case["head_dim"])
        return s["y"]
    if op == "attn_prefill":
        hip._ffi.call("axf_hip_attn_prefill", ctx.handle, s["y"].data_ptr(), s["yq8"].data_ptr(),
                      s["q"].data_ptr(), case["heads"] * case["head_dim"], None, s["k"].data_ptr(),
                      s["v"].data_ptr(), case["pos"], case["tokens"], case["heads"],
                      case["kv_heads"], case["head_dim"], s["cos"].data_ptr(), s["sin"].data_ptr(), 0)
        return s["y"]
    dec = s["model"].dec
    if op == "step":
        dec.forward_token(s["token"], case["pos"])
        return dec.logits()
    if case["sampled"]:
        tokens = dec.generate_sampled(s["prompt"], case["gen"], temperature=0.8, top_k=40, top_p=0.95,
                                      rep_penalty=1.1, rep_penalty_last_n=64)
    else:
        tokens = dec.generate(s["prompt"], case["gen"])
    return tokens, dec.logits()


def _run_matmul(s, case, ctx):
    rows, cols, t, qt = case["rows"], case["cols"], case["tokens"], s["qtype"]
    y, w, x, rb = s["y"].data_ptr(), s["w"].data_ptr(), s["x"].data_ptr(), s["row_bytes"]
    if qt in K_QUANTS and case["act"] == "q8":
        xq8 = s["xq8"].data_ptr()
        ctx.quantize_q8_0(xq8, x, t * cols)
        if t == 1:
            ctx.gemv_q8(qt, y, w, xq8, rows, cols, rb)
        elif qt == Q4_K:
            ctx.gemm_q4k_q8(y, w, xq8, rows, t, cols, rb)
        else:
            ctx.gemm_q6k_q8(y, w, xq8, rows, t, cols, rb)
    elif qt in K_QUANTS:
        ctx.gemv_f32(qt, y, w, x, rows, cols, rb)
    elif t > 1:
        hip._ffi.call("axf_hip_gemm_misc_f32", ctx.handle, qt, y, w, x, rows, t, cols, rb, 0)
    elif qt == F16:
        hip._ffi.call("axf_hip_gemv_f16_f32", ctx.handle, y, w, x, None, rows, cols)
    else:
        hip._ffi.call("axf_hip_gemv_q8_0w_f32" if qt == Q8_0 else "axf_hip_gemv_q5_0_f32", ctx.handle,
                      y, w, x, rows, cols, rb)
    return s["y"]


# --------------------------------------------------------------------------- what it takes


def _model_work(case, rows, first_pos, heads_read):
    """(weight bytes of one reading of the layers, head bytes, flops, KV bytes) of `rows` new rows."""
    t, emb_type, head_type = _types(case)
    w = sum(a * b * BITS[t[k]] / 8 for k, (a, b) in _shapes(case).items()) * case["layers"]
    n = sum(a * b for a, b in _shapes(case).values()) * case["layers"]
    head = case["vocab"] * case["embd"] * BITS[head_type] / 8
    seen = sum(first_pos + i + 1 for i in range(rows))
    flops = 2.0 * n * rows + 4.0 * seen * case["embd"] * case["layers"]
    flops += 2.0 * case["vocab"] * case["embd"] * heads_read
    kv_row = 8.0 * case["embd"] // case["heads"] * case["kv_heads"] * case["layers"]
    return w, head, flops, kv_row, seen


def work(case):
    op = case["op"]
    if op in ("matmul", "head"):
        rows, cols, t = case["rows"], case["cols"], case.get("tokens", 1)
        return {"bytes": rows * cols * BITS[TYPES[case["type"]]] / 8 + 4.0 * t * (rows + cols),
                "flops": 2.0 * rows * cols * t}
    if op in ("attn_decode", "attn_prefill"):
        t = case.get("tokens", 1)
        pos = case["seq"] - 1 if op == "attn_decode" else case["pos"]
        n, hd = pos + t, case["head_dim"]
        seen = sum(pos + i + 1 for i in range(t))
        # the output as fp32 rows and as Q8_0 blocks
        return {"bytes": 8.0 * n * case["kv_heads"] * hd + (4 + 4 + 36 / 32) * t * case["heads"] * hd,
                "flops": 4.0 * seen * case["heads"] * hd}
    if op == "step":
        w, head, flops, kv_row, seen = _model_work(case, 1, case["pos"], 1)
        return {"bytes": w + head + kv_row * seen + 4.0 * case["vocab"], "flops": flops}
    p, g = case["prompt"], case["gen"]
    w, head, flops, kv_row, _ = _model_work(case, p, 0, 1)
    _, _, f2, _, seen = _model_work(case, g - 1, p, g - 1)
    return {"bytes": (w + head) * g + kv_row * (p + seen), "flops": flops + f2}


def tolerance(case):
    op = case["op"]
    if op in ("matmul", "head"):
        # 32-bit sums: 1e-7 to 3e-7 off 64 bits
        return {"rel": 1.5e-6, "max": 2e-5, "differ": 0.0}
    if op in ("attn_decode", "attn_prefill"):
        return {"rel": 2e-6, "max": 2e-5}
    # each layer rounds its activations to Q8_0 four times: a last bit that falls the
    # other way moves a value by 1/127 of its block's largest, and those after it;
    # 64-bit arithmetic is up to 2e-3 off after a step, 5e-3 to 14e-3 after a generation
    return {"rel": 8e-3 if op == "step" else 3e-2, "max": 8e-2 if op == "step" else 0.3,
            "differ": 0.0}


# --------------------------------------------------------------------------- 64 bits


def exact(case, seed):
    i, op = _inputs(case, seed), case["op"]
    if op in ("matmul", "head"):
        x = i["x"].double()
        if op == "matmul" and case["act"] == "q8":
            x = _q8_64(x)
        y = _product64(x, i["w"], TYPES[case["type"]], case["cols"])
        return (y, None) if op == "head" else y
    if op in ("attn_decode", "attn_prefill"):
        hd, kvh = case["head_dim"], case["kv_heads"]
        q, k, v = i["q"].double().reshape(-1, case["heads"], hd), i["k"].double(), i["v"].double()
        pos = case["pos"] if op == "attn_prefill" else case["seq"] - 1
        if op == "attn_prefill":
            c, s = (i[n][pos:].double()[:, None, :] for n in ("cos", "sin"))
            lo, hi = q[..., :hd // 2], q[..., hd // 2:]
            q = torch.cat([lo * c - hi * s, hi * c + lo * s], 2)
        y = _attention64(q, k.reshape(-1, kvh, hd), v.reshape(-1, kvh, hd), pos)
        return y.reshape(-1, case["heads"] * hd)
    if op == "step":
        tokens = torch.tensor([i["token"]], device=DEV)
        return _forward64(case, i["tensors"], tokens, case["pos"], 0, i["kv"])
    # every picked token is its predecessor's successor; the logits are the last step's
    prompt, v = i["prompt"], case["vocab"]
    made = [(int(prompt[-1]) + n * _shift(case)) % v for n in range(1, case["gen"])]
    tokens = torch.cat([prompt, torch.tensor(made, device=DEV, dtype=prompt.dtype)])
    logits = _forward64(case, i["tensors"], tokens, 0, case["prompt"] if case["prompt"] > 1 else 0)
    if case["sampled"]:  # the last pick's penalty stays in the logits, once for each occurrence
        for t in tokens[-64:].tolist():
            logits[t] = logits[t] / 1.1 if logits[t] > 0 else logits[t] * 1.1
    return None, logits
