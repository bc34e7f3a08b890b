"""The calls that a program serving old-KV partial attention makes, as cases that can be timed and compared.

A case is one call of the device-resident path on one stream: the partial attention of one layer over paged, quantized
K/V (decode, verify and prefill row counts; the (O, m, l) partial or the reply format), the acceptance of a draft block
over its logits, or the append of new keys. Bytes and operations in work() are what the call cannot do without: K/V, Q
and results once, and the multiply-adds of QK and PV.
"""
import math

import numpy as np
import torch

import backburner_amd as bb

FMT = {"f16": bb.FMT_F16, "q8_0": bb.FMT_Q8_0, "q4_0": bb.FMT_Q4_0}
QMODE = {"ggml": bb.QMODE_GGML, "f16": bb.QMODE_F16}
BLOCK = {"f16": 64, "q8_0": 34, "q4_0": 18}          # bytes per 32 values

_ws = None


def _workspace():
    """One workspace for the one stream that the calls run on, as a serving loop keeps it."""
    global _ws
    if _ws is None:
        _ws = bb.Workspace()
    return _ws


def _attn(name, op, fmt, qmode, heads, rows, hd, keys, page=bb.PAGE):
    return {"name": name, "op": op, "fmt": fmt, "qmode": qmode, "heads": heads, "rows": rows, "hd": hd, "keys": keys,
            "page": page}


def listed():
    return [
        # one token x GQA 8 over a single page: the smallest call, where launches and latency count
        _attn("decode 4k q8_0", "attn", "q8_0", "ggml", 8, 8, 128, 4096),
        # the headline: one token over a 128k cache
        _attn("decode 128k q8_0", "attn", "q8_0", "ggml", 8, 8, 128, 131072),
        # the 4-bit cache of a 140k context, answered in the reply format that goes back to the sender
        _attn("decode 140k q4_0 reply", "reply", "q4_0", "ggml", 8, 8, 128, 143360),
        # a 16-token draft block verified over 96k keys
        _attn("verify 16 tokens 96k q8_0", "attn", "q8_0", "ggml", 8, 128, 128, 98304),
        # a short draft (5 tokens) over a cache that ends inside a page and inside a tile
        _attn("verify 5 tokens ragged q4_0 reply", "reply", "q4_0", "ggml", 8, 40, 128, 33333),
        # a 512-token prefill chunk over 64k keys: the largest call
        _attn("prefill 512 tokens 64k q8_0", "attn", "q8_0", "ggml", 8, 4096, 128, 65536),
        # a 250-token chunk in the reference engines' query rounding over a 16k 4-bit cache (rows not a multiple of a block)
        _attn("prefill 250 tokens 16k q4_0", "attn", "q4_0", "f16", 8, 2000, 128, 16384),
        # the reference engines' own shape: 8 tokens x GQA 6, head dim 256, f16 queries
        _attn("head 256 verify 64k q8_0", "attn", "q8_0", "f16", 4, 48, 256, 65536),
        # its prefill call: 256 tokens over 16k 4-bit keys
        _attn("head 256 prefill 16k q4_0", "attn", "q4_0", "f16", 4, 1536, 256, 16384),
        # decode over pages that the server stored as f16
        _attn("decode 32k f16", "attn", "f16", "ggml", 8, 8, 128, 32768),
        # the verify step's tail: greedy acceptance of 16 drafted tokens over the vocabulary
        {"name": "accept 16 drafts", "op": "accept", "rows": 17, "vocab": 151936},
        # the sender's side of a prefill chunk: 512 new tokens of fp32 K/V quantized into their pages
        {"name": "append 512 tokens q8_0", "op": "append", "fmt": "q8_0", "heads": 8, "hd": 128, "tokens": 512, "pos": 3900,
         "page": bb.PAGE},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["attn", "attn", "attn", "attn", "reply", "reply", "accept", "append"])
    if op == "accept":
        return {"op": "accept", "rows": rng.randint(2, 33), "vocab": _log(rng, 32000, 262144)}
    if op == "append":
        return {"op": "append", "fmt": rng.choice(["q8_0", "q4_0", "f16"]), "heads": rng.choice([4, 8]),
                "hd": rng.choice([128, 256]), "tokens": _log(rng, 1, 2048), "pos": rng.randint(0, 8191), "page": bb.PAGE}
    hd = rng.choice([128, 128, 128, 256])
    heads = 8 if hd == 128 else 4
    gqa = 8 if hd == 128 else 6
    kind = rng.choice(["decode", "verify", "prefill"])
    tokens = 1 if kind == "decode" else rng.randint(2, 16) if kind == "verify" else _log(rng, 17, 512)
    fmt = rng.choice(["q8_0", "q8_0", "q4_0", "q4_0", "f16"])
    keys = _log(rng, 300, 65536 if kind == "prefill" or fmt == "f16" else 131072)
    if rng.random() < 0.5:
        keys = max(256, keys // 4096 * 4096)
    return {"op": op, "fmt": fmt, "qmode": rng.choice(["ggml", "ggml", "f16"]), "heads": heads, "rows": tokens * gqa, "hd": hd,
            "keys": keys, "page": bb.PAGE}


# ---------------------------------------------------------------- inputs
def _quantize(x, fmt):
    """fp32 [n, 32] on the device -> block bytes [n, 34 / 18 / 64], by ggml's reference rules."""
    if fmt == "f16":
        return x.half().view(torch.uint8)
    if fmt == "q8_0":
        d = x.abs().amax(1, keepdim=True) / 127.0
        q = torch.where(d > 0, x * (1.0 / d.clamp_min(1e-30)), torch.zeros_like(x))
        q = (torch.sign(q) * torch.floor(q.abs() + 0.5)).to(torch.int8).view(torch.uint8)
        return torch.cat([d.half().view(torch.uint8), q], 1)
    i = x.abs().argmax(1, keepdim=True)
    d = x.gather(1, i) / -8.0
    q = torch.where(d != 0, x / torch.where(d != 0, d, torch.ones_like(d)), torch.zeros_like(x))
    q = torch.floor(q + 8.5).clamp(0, 15).to(torch.uint8)
    return torch.cat([d.half().view(torch.uint8), q[:, :16] | (q[:, 16:] << 4)], 1)


def _rows(gen, keys, heads, hd, fmt, outliers):
    """K or V rows of N(0,1) values, as bytes [keys, heads * head bytes]; K with 4 channels per head scaled by 8, the outlier
    channels of real keys."""
    out = torch.empty(keys, heads * hd // 32 * BLOCK[fmt], dtype=torch.uint8, device="cuda")
    gain = torch.ones(heads, hd, device="cuda")
    if outliers:
        at = torch.rand(heads, hd, generator=gen, device="cuda").argsort(1)[:, :4]
        gain.scatter_(1, at, 8.0)
    for k0 in range(0, keys, 16384):
        n = min(16384, keys - k0)
        x = torch.randn(n, heads, hd, generator=gen, device="cuda") * gain
        out[k0:k0 + n] = _quantize(x.reshape(-1, 32), fmt).reshape(n, -1)
    return out


def _pages(K, V, page):
    n, rs = K.shape
    starts = range(0, n, page)
    return bb.Pages([K.data_ptr() + s * rs for s in starts], [V.data_ptr() + s * rs for s in starts],
                    [min(page, n - s) for s in starts], [])


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    s = {"case": case, "stream": torch.cuda.current_stream().cuda_stream, "ws": _workspace()}
    if case["op"] == "accept":
        n, vocab = case["rows"], case["vocab"]
        s["logits"] = torch.randn(n, vocab, generator=gen, device="cuda") * 2.0
        best = s["logits"].argmax(1).to(torch.int32)
        s["draft"] = best[:n - 1].clone()
        hit = n // 2                                        # the draft goes wrong half way through
        s["draft"][hit:] = (s["draft"][hit:] + 1) % vocab
        s["out"] = torch.zeros(2 + n, dtype=torch.int32, device="cuda")
        return s
    heads, hd, fmt = case["heads"], case["hd"], case["fmt"]
    if case["op"] == "append":
        n, pos, page = case["tokens"], case["pos"], case["page"]
        s["K"] = torch.randn(n, heads, hd, generator=gen, device="cuda")
        s["V"] = torch.randn(n, heads, hd, generator=gen, device="cuda")
        s["shape"] = bb.make_shape(heads, 8, hd, FMT[fmt])
        n_pages = (pos + n + page - 1) // page
        s["k"] = torch.zeros(n_pages * page, s["shape"].rs, dtype=torch.uint8, device="cuda")
        s["v"] = torch.zeros_like(s["k"])
        s["pages"] = _pages(s["k"], s["v"], page)
        return s
    rows = heads * case["rows"]
    s["k"] = _rows(gen, case["keys"], heads, hd, fmt, True)
    s["v"] = _rows(gen, case["keys"], heads, hd, fmt, False)
    s["q"] = torch.randn(rows, hd, generator=gen, device="cuda")
    s["shape"] = bb.make_shape(heads, case["rows"], hd, FMT[fmt], QMODE[case["qmode"]])
    s["pages"] = _pages(s["k"], s["v"], case["page"])
    if case["op"] == "reply":
        s["Oh"] = torch.zeros(rows, hd, dtype=torch.float16, device="cuda")
        s["lse"] = torch.zeros(rows, device="cuda")
    else:
        s["O"] = torch.zeros(rows, hd, device="cuda")
        s["m"] = torch.zeros(rows, device="cuda")
        s["l"] = torch.zeros(rows, device="cuda")
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    case = s["case"]
    op = case["op"]
    if op == "attn":
        s["ws"].attn(s["shape"], s["pages"], s["q"].data_ptr(), s["O"].data_ptr(), s["m"].data_ptr(), s["l"].data_ptr(),
                     s["stream"])
        return {"O": s["O"], "m": s["m"], "l": s["l"]}
    if op == "reply":
        s["ws"].attn_reply(s["shape"], s["pages"], s["q"].data_ptr(), s["Oh"].data_ptr(), s["lse"].data_ptr(), s["stream"])
        return {"Oh": s["Oh"], "lse": s["lse"]}
    if op == "accept":
        s["ws"].accept(s["logits"].data_ptr(), case["rows"], case["vocab"], s["draft"].data_ptr(), s["out"].data_ptr(),
                       s["stream"])
        return s["out"]
    bb.append_f32(s["shape"], s["pages"], case["page"], case["pos"], s["K"].data_ptr(), s["V"].data_ptr(), case["tokens"],
                  s["stream"])
    return {"k": s["k"], "v": s["v"]}


def work(case):
    op = case["op"]
    if op == "accept":
        n = case["rows"] * case["vocab"]
        return {"bytes": 4 * n + 4 * (2 * case["rows"] + 1), "flops": n}
    row = case["heads"] * case["hd"] // 32 * BLOCK[case["fmt"]]
    if op == "append":
        values = 2 * case["tokens"] * case["heads"] * case["hd"]
        return {"bytes": 4 * values + 2 * case["tokens"] * row, "flops": 4 * values}
    rows, hd = case["heads"] * case["rows"], case["hd"]
    result = rows * (2 * hd + 4) if op == "reply" else rows * (4 * hd + 8)
    return {"bytes": 2 * case["keys"] * row + 4 * rows * hd + result, "flops": 4 * rows * case["keys"] * hd}


def tolerance(case):
    if case["op"] in ("accept", "append"):
        return "exact"
    # probabilities and V (f16 queries: K too) enter the matrix cores as fp16, sums are fp32: against 64 bits 2e-4 to 6e-4
    # on O, up to 4e-4 on l, below 1e-4 on m
    return {"rel": 2.4e-3, "max": 2.4e-2}


# ---------------------------------------------------------------- the same in 64 bits
def _values(rows, fmt, heads, hd, h):
    """Head h of the row bytes as fp64 [keys, hd]."""
    nb, bb_ = hd // 32, BLOCK[fmt]
    b = rows.reshape(rows.shape[0], heads, nb, bb_)[:, h].contiguous()
    if fmt == "f16":
        return b.view(torch.float16).reshape(-1, hd).double()
    d = b[..., :2].contiguous().view(torch.float16).double()
    if fmt == "q8_0":
        return (d * b[..., 2:].contiguous().view(torch.int8).double()).reshape(-1, hd)
    q = b[..., 2:]
    return (d * (torch.cat([q & 15, q >> 4], -1).double() - 8.0)).reshape(-1, hd)


def _query(q, case, scale):
    """The query rounding that the call asks for (part of its definition), then 64 bits; scale included."""
    if case["qmode"] == "f16":
        return (q * scale).half().double()
    if case["fmt"] == "f16":
        return q.half().double() * scale
    x = q.reshape(-1, 32)
    d = x.abs().amax(1, keepdim=True) / 127.0
    t = x * torch.where(d > 0, 1.0 / d, torch.zeros_like(d))
    t = torch.sign(t) * torch.floor(t.abs() + 0.5)
    return (d.half().double() * t.double()).reshape(q.shape) * scale


def exact(case, seed):
    s = prepare(case, seed)
    if case["op"] == "accept":
        best = s["logits"].double().argmax(1).cpu().numpy()
        draft = s["draft"].cpu().numpy()
        k = 0
        while k < len(draft) and best[k] == draft[k]:
            k += 1
        return torch.from_numpy(np.concatenate([[k, best[k]], best]).astype(np.int32))
    if case["op"] == "append":
        return None
    heads, n, hd, fmt = case["heads"], case["rows"], case["hd"], case["fmt"]
    Q = _query(s["q"], case, s["shape"].scale).reshape(heads, n, hd)
    O = torch.zeros(heads, n, hd, dtype=torch.float64, device="cuda")
    m = torch.full((heads, n), -math.inf, dtype=torch.float64, device="cuda")
    l = torch.zeros(heads, n, dtype=torch.float64, device="cuda")
    for h in range(heads):
        K, V = _values(s["k"], fmt, heads, hd, h), _values(s["v"], fmt, heads, hd, h)
        step = max(4096, 2 ** 27 // max(n, 1))
        for k0 in range(0, case["keys"], step):
            S = Q[h] @ K[k0:k0 + step].t().contiguous()
            mn = torch.maximum(m[h], S.amax(1))
            w = torch.exp(m[h] - mn)
            P = torch.exp(S - mn[:, None])
            O[h] = O[h] * w[:, None] + P @ V[k0:k0 + step]
            l[h] = l[h] * w + P.sum(1)
            m[h] = mn
    O, m, l = O.reshape(-1, hd), m.reshape(-1), l.reshape(-1)
    if case["op"] == "reply":
        return {"Oh": O / l[:, None], "lse": m + l.log()}
    return {"O": O, "m": m, "l": l}
