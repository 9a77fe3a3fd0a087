"""The calls that a serving program makes on the paged KV-cache path, as measurable cases.

A serving engine runs, per attention layer, one of two sequences of calls on one layer's cache:
  decode step   qknorm_rope_append (or store_kvcache) for the new tokens, then gqa_decode_paged_fn
  prefill chunk qknorm_rope_append (or store_kvcache) for the chunk, then gqa_prefill_paged_fn
Each case is one of these calls, or a decode layer's pair, over the sizes that the repository's own
workloads, tests and benchmark use: 24 query / 4 KV heads of 256 (and that model's tensor-parallel
shards, 12/2 and 6/1), 32/8 heads of 128, bf16 and fp16, pages of 8, 16 and 32 tokens, one short
sequence up to 64 sequences of 32,768 tokens, chunks of a few tokens up to thousands.

Kinds of case (the `kind` entry):
  layer    qknorm_rope_append of the step's tokens, then the gated decode: one decode layer
  decode   gqa_decode_paged_fn alone (`append`: with the step's append fused into it)
  prefix   the decode of a batch whose tables share a prefix's pages (`keyword`: stated by the caller)
  prefill  gqa_prefill_paged_fn of packed chunks (first chunks, or continuations over cached tokens)
  inputs   qknorm_rope_append of a chunk: the input side of a prefill layer
  append   store_kvcache of a chunk
"""
import math
import random

import torch

from tileinfer_amd.kernels import (gqa_decode_paged_fn, gqa_prefill_paged_fn, qknorm_rope_append,
                                   store_kvcache)

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
ROTARY = 64  # rotated dimensions of each head
EPS = 1e-6


def _case(name, kind, hq=24, hkv=4, d=256, dtype="bf16", page=16, **kw):
    case = {"kind": kind, "hq": hq, "hkv": hkv, "d": d, "dtype": dtype, "page": page, **kw}
    return {"name": name, **case} if name else case


def listed():
    return [
        # One short interactive session: launch and latency bound.
        _case("layer_1x512", "layer", batch=1, lo=512, hi=512, lens=1),
        # A small server's decode layer, ragged contexts.
        _case("layer_16x8k", "layer", batch=16, lo=512, hi=8192, lens=2),
        # The headline workload: long contexts at batch 64, one layer.
        _case("decode_64x32k", "decode", batch=64, lo=32768, hi=32768, lens=3, append=False),
        # Chat traffic: many sequences of up to two thousand tokens, the append fused in.
        _case("decode_64x2k", "decode", batch=64, lo=64, hi=2048, lens=4, append=True),
        # Another model family's heads, fp16, small pages, odd batch.
        _case("decode_33_d128", "decode", hq=32, hkv=8, d=128, dtype="fp16", page=8, batch=33,
              lo=1, hi=6000, lens=5, append=False),
        # A batch behind one system prompt, which the scheduler shares through the prefix cache.
        _case("prefix_128x8k", "prefix", batch=128, prefix=8192, lo=1, hi=1023, lens=6,
              keyword=True),
        # The first chunk of a prompt, gate in the epilogue.
        _case("prefill_first_2k", "prefill", seqs=1, q_lo=2048, q_hi=2048, c_lo=0, c_hi=0, lens=7,
              gate=True),
        # A later chunk of a long prompt.
        _case("prefill_2k_on_6k", "prefill", seqs=1, q_lo=2048, q_hi=2048, c_lo=6144, c_hi=6144,
              lens=8, gate=False),
        # Short prompts batched into one prefill, odd lengths.
        _case("prefill_24_short", "prefill", seqs=24, q_lo=17, q_hi=700, c_lo=0, c_hi=0, lens=9,
              gate=True),
        # Another model family's heads, fp16: chunks of several prompts with cached context.
        _case("prefill_5_d128", "prefill", hq=32, hkv=8, d=128, dtype="fp16", seqs=5, q_lo=200,
              q_hi=1500, c_lo=0, c_hi=6000, lens=10, gate=False),
        # The input side of a mixed step: a 2,048-token chunk and 32 decode tokens.
        _case("inputs_2080", "inputs", tokens=2080),
        # A bulk append: many chunks written at once.
        _case("append_16k", "append", tokens=16384),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    heads = rng.choice([(24, 4, 256)] * 4 + [(12, 2, 256), (6, 1, 256), (32, 8, 128), (32, 4, 128)])
    hq, hkv, d = heads
    common = {"hq": hq, "hkv": hkv, "d": d, "dtype": rng.choice(["bf16", "bf16", "fp16"]),
              "page": rng.choice([16, 16, 16, 8, 32]), "lens": rng.randrange(1 << 20)}
    kind = rng.choice(["layer", "decode", "decode", "prefix", "prefill", "prefill", "prefill",
                       "inputs", "append"])
    if kind in ("inputs", "append"):
        return _case(None, kind, tokens=_log_int(rng, 16, 16384), **common)
    while True:
        if kind in ("layer", "decode"):
            hi = _log_int(rng, 64, 32768)
            lo = rng.choice([1, max(1, hi // 16), hi])
            more = {"append": rng.random() < 0.5} if kind == "decode" else {}
            case = _case(None, kind, batch=_log_int(rng, 1, 256), lo=lo, hi=hi, **more, **common)
        elif kind == "prefix":
            hi = _log_int(rng, 32, 2048)
            case = _case(None, kind, batch=_log_int(rng, 8, 192), lo=1, hi=hi,
                         prefix=32 * _log_int(rng, 32, 512), keyword=rng.random() < 0.7, **common)
        else:
            seqs = _log_int(rng, 1, 48)
            q_hi = _log_int(rng, 16, 6000)
            c_hi = rng.choice([0, 0, _log_int(rng, 64, 24000)])
            case = _case(None, kind, seqs=seqs, q_lo=rng.choice([q_hi, max(1, q_hi // 20)]),
                         q_hi=q_hi, c_lo=rng.choice([0, c_hi]), c_hi=c_hi,
                         gate=rng.random() < 0.5, **common)
        w = work(case)
        held = _pool(case) * case["page"] * hkv * d * 4  # bytes of both caches
        if max(w["bytes"], w["flops"] / 50) <= 6e9 and held <= 6e9:
            return case



def _lens(case):
    """(query tokens, context tokens) of every sequence; a function of the case alone."""
    rng = random.Random(case.get("lens", 0))
    kind = case["kind"]
    if kind in ("layer", "decode"):
        ctx = [rng.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]
        return [1] * len(ctx), ctx
    if kind == "prefix":
        ctx = [case["prefix"] + rng.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]
        return [1] * len(ctx), ctx
    if kind == "prefill":
        q = [rng.randint(case["q_lo"], case["q_hi"]) for _ in range(case["seqs"])]
        return q, [n + rng.randint(case["c_lo"], case["c_hi"]) for n in q]
    return [case["tokens"]], [case["tokens"]]


def _pages(case):
    return [-(-c // case["page"]) for c in _lens(case)[1]]


def _pool(case):
    """Pages of the cache: a quarter more than the sequences hold, as a pool in use has."""
    need = sum(_pages(case))
    if case["kind"] == "prefix":
        need -= (case["batch"] - 1) * (case["prefix"] // case["page"])
    return math.ceil(1.25 * need)


def _visible(q_len, kv_len):
    """(query, key) pairs of a causal chunk."""
    return q_len * (kv_len - q_len) + q_len * (q_len + 1) // 2


def work(case):
    q_lens, ctx = _lens(case)
    hq, hkv, d, kind = case["hq"], case["hkv"], case["d"], case["kind"]
    tokens = sum(q_lens)
    row_q, row_kv = 2 * hq * d, 2 * hkv * d  # bytes of a token's q (or output), and of its k (or v)
    pages, flops = sum(_pages(case)), 0
    if kind == "append":
        return {"bytes": 4 * row_kv * tokens + 4 * tokens, "flops": 0}
    inputs = (2 * row_q + 4 * row_kv + 4 * ROTARY + 4) * tokens + 4 * d
    if kind == "inputs":
        return {"bytes": inputs, "flops": 10 * (hq + hkv) * d * tokens}
    held = sum(ctx)
    if kind == "prefix":
        held -= (case["batch"] - 1) * case["prefix"]
    nbytes = 2 * row_kv * held + 2 * row_q * tokens + 4 * pages + 8 * len(ctx)
    flops = 4 * hq * d * sum(_visible(a, b) for a, b in zip(q_lens, ctx))
    if case.get("gate") or kind == "layer":
        nbytes += row_q * tokens
    if kind == "layer":
        nbytes += inputs - 2 * row_kv * tokens  # the appended rows are read within the contexts
    elif case.get("append"):
        nbytes += 2 * row_kv * tokens
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Copies are exact. The attention kinds round P to 16 bits before P.V and the output to 16
    bits (`layer` rounds its query twice more, after the norm and after the rotation), `inputs` the
    normalised and the rotated row. Relative errors measured against `exact`: attention 2.1e-3 to
    3.3e-3 in bf16 and 2.7e-4 to 2.9e-4 in fp16, `inputs` 1.8e-3 in bf16; about four times those."""
    kind = case["kind"]
    if kind == "append":
        return "exact"
    coarse = case["dtype"] == "bf16"
    if kind == "inputs":
        return {"rel": 7e-3, "max": 4e-2} if coarse else {"rel": 1e-3, "max": 5e-3}
    return {"rel": 1.2e-2, "max": 6e-2} if coarse else {"rel": 1.4e-3, "max": 8e-3}


def _randn(shape, gen, dt):
    return torch.empty(shape, dtype=dt, device="cuda").normal_(generator=gen)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    dt, page = DTYPES[case["dtype"]], case["page"]
    hq, hkv, d, kind = case["hq"], case["hkv"], case["d"], case["kind"]
    q_lens, ctx = _lens(case)
    pages, pool, tokens = _pages(case), _pool(case), sum(q_lens)
    st = {"case": case}
    # The cache holds earlier tokens' K/V; a sequence's pages lie anywhere in the pool.
    st["k_cache"] = _randn((pool, page, hkv, d), gen, dt)
    st["v_cache"] = _randn((pool, page, hkv, d), gen, dt)
    perm = torch.randperm(pool, generator=gen, device="cuda", dtype=torch.int32)
    width = max(pages)
    table = torch.full((len(ctx), width), -1, dtype=torch.int32, device="cuda")
    shared = case["prefix"] // page if kind == "prefix" else 0
    at = shared
    for i, n in enumerate(pages):
        table[i, :shared] = perm[:shared]
        table[i, shared:n] = perm[at:at + n - shared]
        at += n - shared
    st["table"] = table
    st["seqlen"] = torch.tensor(ctx, dtype=torch.int32, device="cuda")
    st["q"] = _randn((tokens, hq, d), gen, dt)
    if case.get("gate") or kind == "layer":
        st["gate"] = _randn((1, tokens, hq * d), gen, dt)
    if kind == "prefill":
        cu = [0]
        for n in q_lens:
            cu.append(cu[-1] + n)
        st["cu_q"] = torch.tensor(cu, dtype=torch.int32, device="cuda")
        st["max_q"], st["max_k"] = max(q_lens), max(ctx)
    if kind in ("layer", "inputs", "append") or case.get("append"):
        st["k"] = _randn((tokens, hkv, d), gen, dt)
        st["v"] = _randn((tokens, hkv, d), gen, dt)
        # The new tokens are their sequences' last ones.
        row, pos = [], []
        for i, (n, c) in enumerate(zip(q_lens, ctx)):
            row += [i] * n
            pos += range(c - n, c)
        row, pos = torch.tensor(row, device="cuda"), torch.tensor(pos, device="cuda")
        st["slots"] = (table[row, pos // page].long() * page + pos % page).to(torch.int32)
        st["k_rows"], st["v_rows"] = (st[n].view(-1, hkv * d) for n in ("k_cache", "v_cache"))
    if kind in ("layer", "inputs"):
        st["q_w"], st["k_w"] = (0.1 * _randn((d,), gen, dt) for _ in range(2))
        freq = 1e6 ** (-torch.arange(0, ROTARY, 2, device="cuda", dtype=torch.float32) / ROTARY)
        angle = pos.float()[:, None] * torch.cat([freq, freq])[None]
        st["cos"], st["sin"] = angle.cos().to(dt), angle.sin().to(dt)
    return st


def run(st):
    case = st["case"]
    kind, page = case["kind"], case["page"]
    if kind == "append":
        store_kvcache(st["k"], st["v"], st["k_rows"], st["v_rows"], st["slots"])
        return {"k_cache": st["k_cache"], "v_cache": st["v_cache"]}
    q = st["q"]
    if kind in ("layer", "inputs"):
        q = qknorm_rope_append(q, st["k"], st["v"], st["q_w"], st["k_w"], st["cos"], st["sin"],
                               st["k_rows"], st["v_rows"], st["slots"], EPS)
        if kind == "inputs":
            return {"q": q, "k_cache": st["k_cache"], "v_cache": st["v_cache"]}
    caches = (st["k_cache"], st["v_cache"], st["table"])
    if kind == "prefill":
        return {"out": gqa_prefill_paged_fn(q, *caches, st["cu_q"], st["seqlen"], st["max_q"], page,
                                            max_seqlen_k=st["max_k"], gate=st.get("gate"))}
    if kind == "layer":
        out = gqa_decode_paged_fn(q, *caches, st["seqlen"], page, gate=st["gate"])
    elif kind == "prefix":
        prefix = case["prefix"] if case["keyword"] else 0
        return {"out": gqa_decode_paged_fn(q, *caches, st["seqlen"], page,
                                           shared_prefix_tokens=prefix)}
    elif case["append"]:
        out = gqa_decode_paged_fn(q, *caches, st["seqlen"], page,
                                  append=(st["k"], st["v"], st["slots"]))
    else:
        return {"out": gqa_decode_paged_fn(q, *caches, st["seqlen"], page)}
    return {"out": out, "k_cache": st["k_cache"], "v_cache": st["v_cache"]}


def _norm_rope64(x, w, cos, sin):
    """RMSNorm with (1 + w), then rotate-half RoPE of the first ROTARY dimensions."""
    x = x.double()
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * (1 + w.double())
    c, s = (t.double()[:, None, :] for t in (cos, sin))
    head, tail = x[..., :ROTARY], x[..., ROTARY:]
    half = torch.cat([-head[..., ROTARY // 2:], head[..., :ROTARY // 2]], -1)
    return torch.cat([head * c + half * s, tail], -1)


def _attend64(st, q, k_rows, v_rows):
    """Causal attention of the packed queries over their sequences' pages, in 64 bits."""
    case = st["case"]
    page, hkv, d = case["page"], case["hkv"], case["d"]
    group = case["hq"] // hkv
    out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
    at = 0
    for b, (n, c) in enumerate(zip(*_lens(case))):
        pos = torch.arange(c, device="cuda")
        rows = st["table"][b, pos // page].long() * page + pos % page
        k, v = (t.view(-1, hkv, d)[rows].double() for t in (k_rows, v_rows))
        for h in range(case["hq"]):
            kv = h // group
            for i in range(0, n, 2048):
                m = min(2048, n - i)
                s = (q[at + i:at + i + m, h].double() @ k[:, kv].t().contiguous()) / math.sqrt(d)
                if n > 1:
                    own = c - n + i + torch.arange(m, device="cuda")
                    s.masked_fill_(pos[None] > own[:, None], -math.inf)
                out[at + i:at + i + m, h] = torch.softmax(s, -1) @ v[:, kv].contiguous()
        at += n
    return out


def exact(case, seed):
    st = prepare(case, seed)
    kind, hkv, d = case["kind"], case["hkv"], case["d"]
    if kind == "append":
        return None  # a copy: compared bit for bit
    caches = {n: st[n] for n in ("k_cache", "v_cache")}
    q = st["q"]
    if "slots" in st:
        new_k = st["k"].double()
        if kind in ("layer", "inputs"):
            new_k = _norm_rope64(st["k"], st["k_w"], st["cos"], st["sin"])
            q = _norm_rope64(q, st["q_w"], st["cos"], st["sin"])
        slots = st["slots"].long()
        for name, rows in (("k_cache", new_k), ("v_cache", st["v"].double())):
            wide = caches[name].double()
            wide.view(-1, hkv, d)[slots] = rows
            caches[name] = wide
        if kind == "inputs":
            return {"q": q, **caches}
    out = _attend64(st, q, caches["k_cache"], caches["v_cache"])
    if "gate" in st:
        out = out * torch.sigmoid(st["gate"].double()).view(out.shape)
    return {"out": out, **caches} if "slots" in st else {"out": out}
