"""The operator calls whose speed is watched, and how their results are checked.

A case is one call of the public operator API as an attention layer makes it:
varlen-packed q [tokens, Hq, D] and k / v [tokens, Hkv, D] (or a paged cache), a
relative bias, and the layer's options.  Sizes are this repository's own
(benchmark, test and serving workloads: Hq 8 / Hkv 2 or Hq = Hkv = 4, head_dim
128 and 64, extents 128 / 512 / 1024, block size 16) or odd and ragged ones of
the same ranges.

Fields of a case:
  op         "prefill", "rproj" (prefill, bias from low-rank factors), "decode"
             (contiguous cache), "paged" (block tables)
  batch, q_lo, q_hi, past_lo, past_hi, len_seed
             sequences; sequence b holds U[q_lo, q_hi] new tokens over a cache of
             U[past_lo, past_hi] older keys plus the new tokens' own
  hq, hkv, d, dtype, kv ("same" or "fp8"), block (paged: tokens per block)
  rel        "table": one row per head shared by every token (token stride 0);
             "token": a row per token and head; rel_dtype, extent
             (rproj: the dtype of r; W is fp32 [16, extent])
  causal, window (-1: none), bottom_right, scale ("head_dim": the operator's
             default 1/d; "sqrt": 1/sqrt(d)), lse (return the LSE too)
"""
import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.getcwd(), "inkling-fa4-relative-attention_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from inkling_fa4 import (inkling_fa4_rel_attention, inkling_fa4_rel_attention_decode,  # noqa: E402
                         inkling_fa4_rel_attention_decode_paged,
                         inkling_fa4_rel_attention_rproj)

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_BASE = dict(op="prefill", batch=1, q_lo=1, q_hi=1, past_lo=0, past_hi=0, len_seed=1,
             hq=8, hkv=2, d=128, dtype="bf16", kv="same", block=0, rel="token",
             rel_dtype="bf16", extent=1024, causal=True, window=-1, bottom_right=False,
             scale="head_dim", lse=False)


def _case(name=None, **kw):
    c = dict(_BASE, **kw)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # The reference's own benchmark call: one sequence over 4 heads, per-token
        # bias of extent 1024, timed at 64 .. 4096 tokens; here a short prompt.
        _case("prompt_512", q_lo=512, q_hi=512, hq=4, hkv=4),
        # The throughput workload: a full batch of long prompts, one bias table.
        _case("prefill_8x4096", batch=8, q_lo=4096, q_hi=4096, rel="table", rel_dtype="fp32",
              extent=128),
        # A packed batch of prompts of very unequal lengths, with the LSE a caller
        # needs to merge contexts.
        _case("ragged_prompts", batch=16, q_lo=17, q_hi=1900, len_seed=3, lse=True),
        # Chunked prefill of a global layer in the serving convention: the next
        # few hundred tokens of long prompts over their cached keys.
        _case("chunk_global", batch=3, q_lo=333, q_hi=512, past_lo=3000, past_hi=9000,
              len_seed=4, bottom_right=True, lse=True),
        # The same on a local layer: window and bias extent 512.
        _case("chunk_local", batch=6, q_lo=200, q_hi=900, past_lo=100, past_hi=4000, len_seed=5,
              bottom_right=True, window=511, extent=512),
        # head_dim 64 in fp16 (the small-model configuration), 1/sqrt(d) scale.
        _case("prefill_d64", batch=6, q_lo=700, q_hi=2048, len_seed=6, hq=8, hkv=8, d=64,
              dtype="fp16", rel="table", rel_dtype="fp32", extent=128, scale="sqrt"),
        # Prefill with the relative-logit projection fused in, extent 1024.
        _case("rproj_prompts", op="rproj", batch=2, q_lo=900, q_hi=2100, len_seed=7,
              rel_dtype="bf16"),
        # A serving decode step of a global layer: 64 caches of 1K .. 16K keys.
        _case("decode_64", op="decode", batch=64, past_lo=1023, past_hi=16383, len_seed=8,
              bottom_right=True),
        # The same on a paged fp8 cache.
        _case("decode_paged_fp8", op="paged", batch=40, past_lo=500, past_hi=8000, len_seed=9,
              kv="fp8", block=16, bottom_right=True),
        # A single user's decode step on a long context.
        _case("decode_one_32k", op="decode", batch=1, past_lo=32767, past_hi=32767,
              rel="table", rel_dtype="fp32", extent=128, causal=False),
        # A decode step of a local layer: window 512 of a paged cache.
        _case("decode_window", op="paged", batch=24, past_lo=200, past_hi=6000, len_seed=10,
              block=16, bottom_right=True, window=511, extent=512),
        # A few query tokens per sequence over long caches (draft verification,
        # the tail of chunked prompts): the decode entry with more than one token.
        _case("decode_multi", op="decode", batch=12, q_lo=2, q_hi=5, past_lo=1000, past_hi=8000,
              len_seed=11, bottom_right=True, lse=True),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _span(rng, lo, hi):
    """Two sizes lo <= a <= b <= hi, spread over the logarithm."""
    a, b = _log_int(rng, lo, hi), _log_int(rng, lo, hi)
    return (a, b) if a <= b else (b, a)


_HEADS = ((4, 4), (8, 2), (8, 2), (8, 4), (16, 4), (8, 1), (6, 3), (16, 2))


def _draw(rng):
    kind = rng.choice(["prompt", "prompt", "chunk", "chunk", "rproj", "decode", "decode", "paged",
                       "paged", "multi"])
    c = _case(len_seed=rng.randrange(1 << 20))
    c["hq"], c["hkv"] = rng.choice(_HEADS)
    c["d"] = rng.choice([128, 128, 128, 64])
    c["dtype"] = rng.choice(["bf16", "bf16", "fp16"])
    c["scale"] = rng.choice(["head_dim", "sqrt"])
    c["lse"] = rng.random() < 0.3
    c["extent"] = rng.choice([128, 512, 1024])
    c["rel_dtype"] = rng.choice([c["dtype"], "fp32"])
    if rng.random() < 0.3:
        c["rel"] = "table"
    if kind == "prompt":
        c["batch"] = _log_int(rng, 1, 16)
        c["q_lo"], c["q_hi"] = _span(rng, 33, 4096)
        if rng.random() < 0.25:
            c["window"] = c["extent"] - 1
        c["causal"] = rng.random() < 0.9
    elif kind == "chunk":
        c["batch"] = _log_int(rng, 1, 8)
        c["q_lo"], c["q_hi"] = _span(rng, 40, 1024)
        c["past_lo"], c["past_hi"] = _span(rng, 64, 8192)
        c["bottom_right"] = True
        if rng.random() < 0.5:
            c["window"] = c["extent"] - 1
    elif kind == "rproj":
        c["op"], c["rel"] = "rproj", "token"
        c["rel_dtype"] = rng.choice(["bf16", "fp32"])
        c["batch"] = _log_int(rng, 1, 6)
        c["q_lo"], c["q_hi"] = _span(rng, 50, 3000)
        c["bottom_right"] = rng.random() < 0.5
        if c["bottom_right"]:
            c["past_lo"], c["past_hi"] = _span(rng, 16, 2048)
    elif kind == "multi":
        c["op"] = "decode"
        c["batch"] = _log_int(rng, 1, 24)
        c["q_lo"], c["q_hi"] = 2, rng.randint(2, 8)
        c["past_lo"], c["past_hi"] = _span(rng, 200, 8192)
        c["bottom_right"] = True
    else:
        c["op"] = kind
        c["batch"] = _log_int(rng, 1, 64)
        c["past_lo"], c["past_hi"] = _span(rng, 100, 16384)
        c["bottom_right"] = rng.random() < 0.75
        c["causal"] = c["bottom_right"]
        if c["bottom_right"] and rng.random() < 0.35:
            c["window"] = c["extent"] - 1
        if kind == "paged":
            c["block"] = rng.choice([16, 16, 32, 64])
        if rng.random() < 0.35:
            c["kv"] = "fp8"
    return c


def draw(rng):
    most = [work(c) for c in listed()]
    flops, nbytes = max(w["flops"] for w in most), max(w["bytes"] for w in most)
    while True:
        c = _draw(rng)
        w = work(c)
        if w["flops"] / flops + w["bytes"] / nbytes <= 1.0:
            return c


def _lens(c):
    """(queries, keys) of each sequence."""
    r = random.Random(c["len_seed"])
    lq = [r.randint(c["q_lo"], c["q_hi"]) for _ in range(c["batch"])]
    return lq, [n + r.randint(c["past_lo"], c["past_hi"]) for n in lq]


def _geometry(c, lq, lk, i):
    """Of queries i (a tensor) of one sequence: first and last visible key (lo,
    hi exclusive), and the distance of key 0 (dist(i, j) = d0 - j)."""
    pos = i + (lk - lq if c["bottom_right"] else 0)
    hi = torch.clamp(pos + 1, 0, lk) if c["causal"] else torch.full_like(i, lk)
    lo = torch.clamp(pos - c["window"], min=0) if c["window"] >= 0 else torch.zeros_like(i)
    return lo, hi, i + (lk - lq if c["bottom_right"] else lq - lk)


def work(case):
    """Queries, outputs and every visible key once, the bias a visible pair needs
    once; 4 d flops per visible pair and head (and the projection's products)."""
    c = case
    lqs, lks = _lens(c)
    pairs = band = keys = 0
    for lq, lk in zip(lqs, lks):
        i = torch.arange(lq)
        lo, hi, d0 = _geometry(c, lq, lk, i)
        pairs += int(torch.clamp(hi - lo, min=0).sum())
        b0 = torch.maximum(lo, d0 - c["extent"] + 1)
        band += int(torch.clamp(torch.minimum(hi, d0 + 1) - b0, min=0).sum())
        keys += max(0, int(hi.max()) - int(lo.min()))
    tq = sum(lqs)
    esize, rsize = (1 if c["kv"] == "fp8" else 2), (4 if c["rel_dtype"] == "fp32" else 2)
    nbytes = 2 * tq * c["hq"] * c["d"] * 2 + 2 * keys * c["hkv"] * c["d"] * esize
    flops = 4 * c["d"] * pairs * c["hq"]
    if c["op"] == "rproj":
        nbytes += tq * c["hq"] * 16 * rsize + 16 * c["extent"] * 4
        flops += 2 * 16 * band * c["hq"]
    elif c["rel"] == "table":
        nbytes += c["hq"] * c["extent"] * rsize
    else:
        nbytes += band * c["hq"] * rsize
    if c["block"]:
        nbytes += 4 * sum(-(-n // c["block"]) for n in lks)
    if c["lse"]:
        nbytes += 4 * tq * c["hq"]
    return {"bytes": nbytes, "flops": flops}


_FP8_SCALE = 1.0 / 64  # N(0, 1) keys and values stay inside e4m3's +-448


def _cu(lens):
    out = [0]
    for n in lens:
        out.append(out[-1] + n)
    return torch.tensor(out, dtype=torch.int32, device="cuda")


def prepare(case, seed):
    c = case
    g = torch.Generator("cuda").manual_seed(seed)

    def randn(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    lqs, lks = _lens(c)
    tq, tk = sum(lqs), sum(lks)
    dtype, rdtype = _DTYPES[c["dtype"]], _DTYPES[c["rel_dtype"]]
    s = {"case": c, "q": randn(tq, c["hq"], c["d"]).to(dtype), "cu_q": _cu(lqs), "cu_k": _cu(lks),
         "max_q": max(lqs), "max_k": max(lks)}
    rows = (tk,)
    if c["op"] == "paged":
        bs = c["block"]
        nblk = [-(-n // bs) for n in lks]
        rows = (sum(nblk), bs)
        order = torch.randperm(sum(nblk), generator=g, device="cuda").to(torch.int32)
        table = torch.zeros(c["batch"], max(nblk), dtype=torch.int32, device="cuda")
        at = 0
        for b, n in enumerate(nblk):
            table[b, :n] = order[at:at + n]
            at += n
        s["table"] = table
        s["used"] = torch.tensor(lks, dtype=torch.int32, device="cuda")
    for name in ("k", "v"):
        x = randn(*rows, c["hkv"], c["d"])
        s[name] = ((x / _FP8_SCALE).to(torch.float8_e4m3fn) if c["kv"] == "fp8" else x.to(dtype))
    if c["op"] == "rproj":
        s["r"] = (0.3 * randn(tq, c["hq"], 16)).to(rdtype)
        s["w"] = 0.3 * randn(16, c["extent"])
    elif c["rel"] == "table":
        table = (0.5 * randn(c["hq"], c["extent"])).to(rdtype)
        s["rel"] = table.unsqueeze(0).expand(tq, c["hq"], c["extent"])
    else:
        s["rel"] = (0.5 * randn(tq, c["hq"], c["extent"])).to(rdtype)
    return s


def run(state):
    s, c = state, state["case"]
    kw = dict(causal=c["causal"], window_size=(c["window"], 0) if c["window"] >= 0 else (-1, -1),
              softmax_scale=None if c["scale"] == "head_dim" else 1.0 / math.sqrt(c["d"]),
              return_lse=c["lse"], bottom_right=c["bottom_right"])
    if c["kv"] == "fp8":
        kw.update(k_scale=_FP8_SCALE, v_scale=_FP8_SCALE)
    if c["op"] == "paged":
        out = inkling_fa4_rel_attention_decode_paged(
            s["q"], s["k"], s["v"], s["rel"], s["cu_q"], s["used"], s["table"], s["max_q"],
            s["max_k"], c["extent"], **kw)
    elif c["op"] == "rproj":
        out = inkling_fa4_rel_attention_rproj(
            s["q"], s["k"], s["v"], s["r"], s["w"], s["cu_q"], s["cu_k"], s["max_q"], s["max_k"],
            c["extent"], **kw)
    else:
        op = inkling_fa4_rel_attention_decode if c["op"] == "decode" else inkling_fa4_rel_attention
        out = op(s["q"], s["k"], s["v"], s["rel"], s["cu_q"], s["cu_k"], s["max_q"], s["max_k"],
                 c["extent"], **kw)
    return {"out": out[0], "lse": out[1]} if c["lse"] else {"out": out}


def exact(case, seed):
    """The same call in fp64: dense scores of a sequence and head, row blocks."""
    c = case
    s = prepare(case, seed)
    lqs, lks = _lens(c)
    f64 = torch.float64
    scale = 1.0 / c["d"] if c["scale"] == "head_dim" else 1.0 / math.sqrt(c["d"])
    mul = _FP8_SCALE if c["kv"] == "fp8" else 1.0
    out = torch.zeros(sum(lqs), c["hq"], c["d"], dtype=f64, device="cuda")
    lse = torch.zeros(c["hq"], sum(lqs), dtype=f64, device="cuda")
    qs = ks = 0
    for b, (lq, lk) in enumerate(zip(lqs, lks)):
        if c["op"] == "paged":
            at = s["table"][b, :-(-lk // c["block"])].long()
            kv = [s[n][at].float().reshape(-1, c["hkv"], c["d"])[:lk] for n in ("k", "v")]
        else:
            kv = [s[n][ks:ks + lk].float() for n in ("k", "v")]
        key = torch.arange(lk, device="cuda")
        for h in range(c["hq"]):
            kh, vh = (x[:, h // (c["hq"] // c["hkv"])].to(f64) * mul for x in kv)
            for i0 in range(0, lq, 1024):
                i = torch.arange(i0, min(lq, i0 + 1024), device="cuda")
                lo, hi, d0 = (x.unsqueeze(1) for x in _geometry(c, lq, lk, i))
                x = s["q"][qs + i, h].to(f64) @ kh.t() * scale
                if c["op"] == "rproj":
                    rel = s["r"][qs + i, h].to(f64) @ s["w"].to(f64)
                else:
                    rel = s["rel"][qs + i, h].to(f64)
                dist = d0 - key
                bias = rel.gather(1, dist.clamp(0, c["extent"] - 1))
                x += torch.where((dist >= 0) & (dist < c["extent"]), bias, 0.0)
                x.masked_fill_((key < lo) | (key >= hi), -math.inf)
                lse[h, qs + i] = torch.logsumexp(x, 1)
                out[qs + i, h] = torch.softmax(x, 1) @ vh
        qs += lq
        ks += lk
    return {"out": out, "lse": lse} if c["lse"] else {"out": out}


def tolerance(case):
    """Outputs are rounded to the query type and P to it before P V: bf16 keeps 8
    bits, fp16 11.  About four times the error against exact() (measured: bf16
    1.9e-3 .. 2.4e-3, fp16 2.6e-4 .. 2.8e-4)."""
    if case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 6e-2}
    return {"rel": 1.2e-3, "max": 1e-2}
