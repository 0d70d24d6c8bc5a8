"""Performance cases of the attention path: what a program that serves or
evaluates a transformer asks of this package, through its public entry points.

A case is a flat dict:

  kind    attn         flash_attn over contiguous K/V (whole sequences, no cache)
          prefill      flash_attn_paged, a chunk of M new tokens per sequence
          decode       flash_attn_paged, 1 query row per sequence (or a few:
                       the drafted tokens of speculative decoding)
          step         flash_attn_paged_append: one token appended, then attended
          append       paged_kv_append of M new tokens per sequence
          token_major  decode_token_major over the INT8 engine's cache layout
  B, Hq, Hk, D, M      batch, query heads, KV heads, head dim, query rows (new tokens)
  N                    attn: keys; token_major: cached rows
  page, pool           tokens per page; one shared pool with a block table (True)
                       or a page array per sequence without one (False)
  lo, hi, mix          tokens each sequence has cached before the call: uniform
                       in [lo, hi], drawn from `mix` (a plain number of the case)
  ragged               prefill: sequence b brings only some of the M rows (q_lens)
  rope                 rotary embedding fused into the call
  f32, causal          element type (attn) and mask

Q, K and V are N(0, 1), as in the package's benchmark workloads.
"""
from __future__ import annotations

import math
import random

import torch

from hrm_flashrenderer_amd import (build_rope_cache, flash_attn, flash_attn_paged,
                                   flash_attn_paged_append, paged_kv_append)
from hrm_flashrenderer_amd.token_major import decode_token_major

DEVICE = "cuda"


def _case(kind, **kw):
    c = dict(kind=kind, B=1, Hq=8, Hk=8, D=128, M=1, N=0, page=16, pool=True, lo=0, hi=0, mix=0,
             ragged=False, rope=False, f32=False, causal=True)
    c.update(kw)
    return c


def listed():
    return [
        # the smallest call: one short sequence of a small MHA model, fp16
        _case("attn", name="attn_small_f16", Hq=8, Hk=8, D=64, M=512, N=512),
        # fp32 attention of whole sequences (evaluation, checks against fp16), an odd length
        _case("attn", name="attn_odd_f32", B=2, Hq=16, Hk=16, D=128, M=1000, N=1000, f32=True),
        # a batch of prompts prefilled at once, 40/8 heads
        _case("prefill", name="prefill_batch", B=4, Hq=40, Hk=8, M=2048),
        # a ragged chunk of several requests with small pages, per-sequence
        # page arrays and 64-wide heads
        _case("prefill", name="prefill_ragged_page8", B=5, Hq=32, Hk=8, D=64, M=777, page=8,
              pool=False, hi=1500, mix=4, ragged=True, rope=True),
        # one user's prompt chunk over a long conversation, 64/8 heads
        _case("prefill", name="chunk_single", B=1, Hq=64, Hk=8, M=512, lo=16000, hi=16000, rope=True),
        # chunked prefill of a full batch over contexts of up to 32K tokens (the largest call)
        _case("prefill", name="chunk_batch", B=16, Hq=64, Hk=8, M=512, hi=32768, mix=5),
        # one user's next token over a short conversation: latency
        _case("decode", name="decode_single", B=1, Hq=40, Hk=8, lo=1500, hi=1500, causal=False),
        # the next token of a mid-sized batch, 40/8 heads
        _case("decode", name="decode_batch", B=32, Hq=40, Hk=8, lo=511, hi=8191, mix=3, causal=False),
        # verification of drafted tokens: five query rows per sequence, large pages
        _case("decode", name="decode_verify", B=24, Hq=64, Hk=8, M=5, page=128, lo=1024, hi=8192,
              mix=6),
        # a whole decode step (append, then attention) of a large batch, 64/8 heads
        _case("step", name="step_batch", B=64, Hq=64, Hk=8, lo=1024, hi=16384, mix=7, rope=True,
              causal=False),
        # a prompt chunk's keys and values written into their pages
        _case("append", name="append_chunk", B=16, Hk=8, M=512, hi=4096, mix=8, rope=True),
        # one layer's decode step of the INT8 engine on its token-major cache
        _case("token_major", name="token_major_32k", Hq=40, Hk=8, N=32768, causal=False),
    ]


_HEADS = ((8, 8), (16, 16), (32, 8), (40, 8), (64, 8))


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(("attn", "prefill", "prefill", "decode", "decode", "step", "append",
                           "token_major"))
        Hq, Hk = rng.choice(_HEADS)
        D = rng.choice((64, 128, 128))
        page = rng.choice((8, 16, 16, 32, 64, 128))
        c = _case(kind, Hq=Hq, Hk=Hk, D=D, page=page, pool=rng.random() < 0.7,
                  mix=rng.randrange(1 << 20))
        if kind == "attn":
            c["f32"] = rng.random() < 0.3
            c["B"] = _logint(rng, 1, 8)
            c["M"] = c["N"] = _logint(rng, 64, 2048 if c["f32"] else 4096)
            c["causal"] = rng.random() < 0.75
            most = 1.6e10 if c["f32"] else 2e11
        elif kind == "prefill":
            c["B"] = _logint(rng, 1, 16)
            c["M"] = _logint(rng, 32, 2048)
            c["hi"] = rng.choice((0, _logint(rng, 64, 4096 if page == 8 else 32768)))
            c["lo"] = c["hi"] // rng.choice((1, 4, 16))
            c["ragged"] = rng.random() < 0.4
            c["rope"] = rng.random() < 0.5
            most = 1e11 if page == 8 else 1.2e12
        elif kind in ("decode", "step"):
            c["B"] = _logint(rng, 1, 96)
            c["M"] = 1 if kind == "step" or rng.random() < 0.6 else rng.randint(2, 8)
            c["hi"] = _logint(rng, 128, 32768)
            c["lo"] = c["hi"] // rng.choice((1, 4, 16))
            c["rope"] = rng.random() < 0.5
            c["causal"] = c["M"] > 1
            most = 4e11
        elif kind == "append":
            c["B"] = _logint(rng, 1, 32)
            c["M"] = _logint(rng, 1, 2048)
            c["hi"] = rng.choice((0, _logint(rng, 64, 4096)))
            c["rope"] = rng.random() < 0.5
            most = 1e12
        else:
            c["Hq"], c["Hk"], c["D"] = rng.choice(((40, 8, 128), (64, 8, 128), (32, 32, 64),
                                                   (28, 4, 128)))
            c["N"] = _logint(rng, 256, 65536)
            c["causal"] = False
            most = 1e12
        w = work(c)
        if w["flops"] <= most and w["bytes"] <= (1.2e9 if page == 8 else 2.3e9) and _pool_bytes(c) <= 3e9:
            return c


# ------------------------------------------------------------------ sizes ---

def _lengths(c):
    """(tokens cached before the call, new tokens) of each sequence."""
    rng = random.Random(1000 + c["mix"])
    prior = [rng.randint(c["lo"], c["hi"]) for _ in range(c["B"])]
    new = [rng.randint(max(1, c["M"] // 8), c["M"]) if c["ragged"] else c["M"] for _ in range(c["B"])]
    return prior, new


def _pool_bytes(c):
    if c["kind"] in ("attn", "token_major"):
        return 0
    prior, _ = _lengths(c)
    most = max(prior) + c["M"]
    tokens = sum(p + c["M"] for p in prior) if c["pool"] else c["B"] * most
    return 4 * c["Hk"] * c["D"] * tokens


def work(c):
    B, Hq, Hk, D, M = (c[k] for k in ("B", "Hq", "Hk", "D", "M"))
    if c["kind"] == "attn":
        size = 4 if c["f32"] else 2
        pairs = sum(min(c["N"], i + 1) if c["causal"] else c["N"] for i in range(M))
        return {"bytes": size * D * (2 * B * Hq * M + 2 * B * Hk * c["N"]),
                "flops": 4 * D * B * Hq * pairs}
    if c["kind"] == "token_major":
        return {"bytes": 2 * 2 * c["N"] * Hk * D + 2 * 4 * Hq * D, "flops": 4 * D * Hq * c["N"]}
    prior, new = _lengths(c)
    tables = 2 * 2 * sum(new) * D // 2 if c["rope"] else 0
    if c["kind"] == "append":
        return {"bytes": 2 * 2 * 2 * B * Hk * M * D + tables, "flops": 6 * B * Hk * M * D // 2 if c["rope"] else 0}
    pages = sum(-(-(p + n) // c["page"]) for p, n in zip(prior, new)) if c["pool"] else 0
    kv = sum(p + n for p, n in zip(prior, new)) * 2 * 2 * Hk * D
    q = 2 * Hq * D * sum(new)
    o = 2 * Hq * D * B * M
    pairs = sum(sum(p + i + 1 for i in range(n)) if c["causal"] else n * (p + n)
                for p, n in zip(prior, new))
    extra = 2 * 2 * B * Hk * D if c["kind"] == "step" else 0
    return {"bytes": kv + q + o + 4 * pages + tables + extra, "flops": 4 * D * Hq * pairs}


# ----------------------------------------------------------------- inputs ---

def _randn(g, *shape, dtype=torch.float16):
    return torch.randn(shape, generator=g, device=DEVICE, dtype=dtype)


def _ints(values):
    return torch.tensor(values, dtype=torch.int32, device=DEVICE)


def prepare(c, seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    B, Hq, Hk, D, M = (c[k] for k in ("B", "Hq", "Hk", "D", "M"))
    s = dict(case=c)
    if c["kind"] == "attn":
        dt = torch.float32 if c["f32"] else torch.float16
        s["q"] = _randn(g, B, Hq, M, D, dtype=dt)
        s["k"] = _randn(g, B, Hk, c["N"], D, dtype=dt)
        s["v"] = _randn(g, B, Hk, c["N"], D, dtype=dt)
        return s
    if c["kind"] == "token_major":
        s["q"] = _randn(g, Hq, D, dtype=torch.float32)
        s["k"] = _randn(g, c["N"], Hk, D)
        s["v"] = _randn(g, c["N"], Hk, D)
        return s
    prior, new = _lengths(c)
    total = [p + n for p, n in zip(prior, new)]
    # pages are mapped for a whole chunk, real rows or not
    pages = [-(-(p + M) // c["page"]) for p in prior]
    if c["pool"]:
        rows, per = 1, sum(pages)
        ids = torch.randperm(per, generator=torch.Generator().manual_seed(seed)).tolist()
        table = torch.full((B, max(pages)), -1, dtype=torch.int32)
        at = 0
        for b, n in enumerate(pages):
            table[b, :n] = torch.tensor(ids[at:at + n], dtype=torch.int32)
            at += n
        s["table"] = table.to(DEVICE)
    else:
        rows, per = B, max(pages)
        s["table"] = None
    s["k"] = _randn(g, rows, Hk, per, c["page"], D)
    s["v"] = _randn(g, rows, Hk, per, c["page"], D)
    s["rope"] = build_rope_cache(max(prior) + M, D) if c["rope"] else None
    s["seqlen"] = _ints(total)
    s["prior"] = _ints(prior)
    s["uniform"] = c["hi"] == 0
    if c["kind"] != "append":
        s["q"] = _randn(g, B, Hq, M, D)
        s["head_map"] = _ints([h // (Hq // Hk) for h in range(Hq)])
    if c["kind"] in ("append", "step"):
        s["k_new"] = _randn(g, B, Hk, M, D)
        s["v_new"] = _randn(g, B, Hk, M, D)
    s["q_lens"] = _ints(new) if c["ragged"] else None
    return s


def run(s):
    c = s["case"]
    if c["kind"] == "attn":
        return flash_attn(s["q"], s["k"], s["v"], c["causal"])
    if c["kind"] == "token_major":
        return decode_token_major(s["q"], s["k"], s["v"], c["N"] - 1)
    start = 0 if s["uniform"] else s["prior"]
    if c["kind"] == "append":
        paged_kv_append(s["k"], s["v"], s["k_new"], s["v_new"], start, c["page"],
                        block_table=s["table"], rope=s["rope"])
        return s["k"], s["v"]
    if c["kind"] == "step":
        o = flash_attn_paged_append(s["q"], s["k"], s["v"], s["k_new"], s["v_new"], s["seqlen"],
                                    c["page"], s["head_map"], c["causal"], start, start_pos=start,
                                    block_table=s["table"], rope=s["rope"])
        return o, s["k"], s["v"]
    # causal rows sit after the cached tokens; without a mask only the rotary
    # embedding reads the offset
    offset = start if c["causal"] or c["rope"] else 0
    return flash_attn_paged(s["q"], s["k"], s["v"], s["seqlen"], c["page"], s["head_map"],
                            c["causal"], offset, block_table=s["table"], rope=s["rope"],
                            q_lens=s["q_lens"])


# ---------------------------------------------------------------- results ---

def tolerance(c):
    if c["kind"] == "append":
        return "exact"  # copies, and a rotation whose every rounding is fixed
    # about four times the error against 64 bits of one correct implementation
    # (2-norm, largest) over the ranges above
    if c["f32"]:
        return {"rel": 8e-7, "max": 2e-5}    # 1.8e-7, 4e-6
    if c["kind"] == "token_major":
        return {"rel": 8e-4, "max": 4e-3}    # 2e-4, 9e-4: fp32 in and out, softmax weights in fp16
    if c["rope"]:
        return {"rel": 1.8e-3, "max": 2.8e-2}  # 4.2e-4, 6.8e-3: fp16 rotation, then as below
    return {"rel": 1.2e-3, "max": 1.6e-2}    # 2.9e-4, 4.1e-3: fp16 in and out


def _attend(q, k, v, limits):
    """softmax(q k^T / sqrt(D)) v in fp64: q [G, M, D] heads of one KV head,
    k, v [N, D], row i of every head sees keys j < limits[i]."""
    G, M, D = q.shape
    s = (q.reshape(G * M, D).double() @ k.double().t().contiguous()).view(G, M, -1)
    s.mul_(1.0 / math.sqrt(D))
    hide = torch.arange(k.size(0), device=k.device)[None, :] >= limits[:, None]
    s.masked_fill_(hide[None], -math.inf)
    p = torch.softmax(s, dim=-1)
    return (p.view(G * M, -1) @ v.double()).view(G, M, D)


def _rotate(x, rope, pos):
    """Half-split rotation of x [..., T, D] at positions pos [T], in fp64."""
    cos, sin = rope[0][pos].double(), rope[1][pos].double()
    h = x.size(-1) // 2
    a, b = x[..., :h].double(), x[..., h:].double()
    return torch.cat((a * cos - b * sin, a * sin + b * cos), dim=-1)


def exact(c, seed):
    s = prepare(c, seed)
    B, Hq, Hk, D, M = (c[k] for k in ("B", "Hq", "Hk", "D", "M"))
    G = Hq // Hk
    ar = torch.arange(M, device=DEVICE)
    if c["kind"] == "attn":
        lim = (ar + 1).clamp(max=c["N"]) if c["causal"] else torch.full_like(ar, c["N"])
        out = torch.empty(B, Hq, M, D, dtype=torch.float64, device=DEVICE)
        for b in range(B):
            for h in range(Hk):
                out[b, h * G:(h + 1) * G] = _attend(s["q"][b, h * G:(h + 1) * G], s["k"][b, h],
                                                    s["v"][b, h], lim)
        return out
    if c["kind"] == "token_major":
        # query head h reads KV head h % Hk
        out = torch.empty(Hq, D, dtype=torch.float64, device=DEVICE)
        lim = torch.tensor([c["N"]], device=DEVICE)
        for h in range(Hk):
            out[h::Hk] = _attend(s["q"][h::Hk, None], s["k"][:, h], s["v"][:, h], lim)[:, 0]
        return out
    prior, new = _lengths(c)
    written = {}
    for b in range(B if c["kind"] in ("append", "step") else 0):
        pos = prior[b] + ar
        kn = _rotate(s["k_new"][b], s["rope"], pos) if c["rope"] else s["k_new"][b].double()
        written[b] = (pos, kn, s["v_new"][b].double())

    def place(b, pos):
        page = pos // c["page"]
        return (0, s["table"][b][page].long(), pos % c["page"]) if c["pool"] else (b, page, pos % c["page"])

    pages = None
    if written:
        pages = (s["k"].double(), s["v"].double())
        for b, (pos, kn, vn) in written.items():
            row, page, slot = place(b, pos)
            pages[0][row][:, page, slot] = kn
            pages[1][row][:, page, slot] = vn
    if c["kind"] == "append":
        return pages
    k_src, v_src = pages if pages is not None else (s["k"], s["v"])
    out = torch.zeros(B, Hq, M, D, dtype=torch.float64, device=DEVICE)
    for b in range(B):
        n = prior[b] + new[b]
        row, page, slot = place(b, torch.arange(n, device=DEVICE))
        live = ar[:new[b]]
        lim = (prior[b] + live + 1) if c["causal"] else torch.full_like(live, n)
        for h in range(Hk):
            q = s["q"][b, h * G:(h + 1) * G, :new[b]]
            if c["rope"]:
                q = _rotate(q, s["rope"], prior[b] + live)
            k, v = k_src[row, h][page, slot], v_src[row, h][page, slot]
            out[b, h * G:(h + 1) * G, :new[b]] = _attend(q, k, v, lim)
    return (out,) + pages if pages is not None else out
