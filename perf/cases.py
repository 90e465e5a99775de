"""Performance cases of the paged-attention path: the calls a serving program makes.

Each case is one pass of a kind of work (its "work" field):

  layer    one layer of an eager decode step, as a model runner without graphs makes it:
           write_kv of the new token, then forward, with an int64 block table and
           Python-list lengths
  graph    one whole decode step of a model through GraphedDecodeRunner (append and
           attention of every layer, page lists from the host's scheduler)
  decode   one layer's decode call over device-resident tables and lengths
  prefix   the same over block tables that share their first pages (a radix-cache hit)
  chunk    a chunk of each prompt's tokens over the tokens already cached
  prompt   one layer of a prompt from its first token: write_kv of every token, forward
  mixed    one scheduler step: a prompt chunk and a batch of decodes, one after the other

Context lengths are part of the case (drawn from its own "lens" seed); the seed of
`prepare` draws values and page placement.
"""
from __future__ import annotations

import math
import random

import torch

from miniserve_amd import PagedAttention, paged_attention
from miniserve_amd.graphs import DecodeLayer, GraphedDecodeRunner

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16,
          "fp8": torch.float8_e4m3fn}
BYTES = {"fp32": 4, "fp16": 2, "bf16": 2, "fp8": 1}
# (query heads, KV heads, head_dim) of the repository's benchmark configurations
SMALL, LLAMA, WIDE7 = (14, 2, 64), (32, 8, 128), (28, 4, 128)


def _case(work, heads, *, q="bf16", kv=None, batch, lo, hi, log=False, q_len=1, layers=1,
          prefix=0, window=0, decodes=0, block=16, lens=1, name=None):
    """A case's plain fields. Contexts (tokens cached before the call's own) lie in
    [lo, hi]; `decodes`: rows of a mixed step's decode batch, over the same range."""
    c = {"work": work, "heads": heads[0], "kv_heads": heads[1], "head_dim": heads[2], "q": q,
         "kv": kv or q, "batch": batch, "lo": lo, "hi": hi, "log": log, "q_len": q_len,
         "layers": layers, "prefix": prefix, "window": window, "decodes": decodes,
         "block": block, "lens": lens}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest calls: four short chats in a small model, in the runner's default
        # fp32, eagerly. Launch and host latency.
        _case("layer", SMALL, q="fp32", batch=4, lo=128, hi=511, name="layer_small_fp32"),
        # A small model's whole decode step at the batch its graph bucket was made for.
        _case("graph", SMALL, batch=32, lo=512, hi=2047, layers=24, name="graph_small_bf16"),
        # A 7B-class model's whole decode step with few, longer contexts.
        _case("graph", WIDE7, batch=16, lo=1024, hi=4095, layers=28, name="graph_wide_bf16"),
        # The headline batch: 64 sequences of ragged length, bandwidth-bound.
        _case("decode", LLAMA, batch=64, lo=1024, hi=8192, log=True, name="decode_64_bf16"),
        # The same batch over an fp8 cache (half the bytes, conversions on the way).
        _case("decode", LLAMA, kv="fp8", batch=64, lo=1024, hi=8192, log=True,
              name="decode_64_fp8"),
        # Sliding-window layers: the context is long, the keys read are few.
        _case("decode", LLAMA, q="fp16", batch=32, lo=2048, hi=16384, log=True, window=1024,
              name="decode_window_fp16"),
        # Long documents behind a shared system prompt: the largest read.
        _case("prefix", LLAMA, batch=8, lo=32768, hi=131072, prefix=512,
              name="prefix_long_bf16"),
        # Chunked prefill: two prompts' 512-token chunks over 4096 cached tokens.
        _case("chunk", WIDE7, batch=2, lo=4096, hi=4096, q_len=512, name="chunk_bf16"),
        # The same chunks over an fp8 cache.
        _case("chunk", WIDE7, q="fp16", kv="fp8", batch=2, lo=4096, hi=4096, q_len=512,
              name="chunk_fp8"),
        # The same chunks in the runner's default fp32.
        _case("chunk", WIDE7, q="fp32", batch=2, lo=4096, hi=4096, q_len=512,
              name="chunk_fp32"),
        # A whole prompt of odd length in the class's default fp16, from the model's
        # transposed projections.
        _case("prompt", LLAMA, q="fp16", batch=1, lo=0, hi=0, q_len=3001, name="prompt_fp16"),
        # A head size other than 64 and 128, one scheduler step: a chunk and its decodes.
        _case("mixed", (24, 8, 96), batch=1, lo=512, hi=2048, q_len=256, decodes=16,
              name="mixed_d96_bf16"),
    ]


def draw(rng):
    def logint(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    work = rng.choice(["layer", "graph", "graph", "decode", "decode", "decode", "prefix",
                       "chunk", "chunk", "chunk", "prompt", "mixed"])
    lens = rng.randrange(1, 1 << 30)
    heads = rng.choice([SMALL, LLAMA, WIDE7])
    if work == "layer":
        hi = logint(64, 1024)
        return _case(work, heads, q=rng.choice(["fp32", "fp32", "bf16", "fp16"]),
                     batch=rng.randint(1, 8), lo=max(1, hi // 4), hi=hi, lens=lens)
    if work == "graph":
        heads = rng.choice([SMALL, WIDE7])
        hi = logint(1024, 4096)
        return _case(work, heads, q=rng.choice(["bf16", "fp16"]),
                     batch=rng.randint(3, 32 if heads == SMALL else 16), lo=hi // 4, hi=hi,
                     layers=rng.randint(8, 24), lens=lens)
    if work == "decode":
        hi = logint(2048, 16384)
        q = rng.choice(["bf16", "fp16"])
        return _case(work, heads, q=q, kv=rng.choice([q, "fp8"]), batch=logint(8, 64),
                     lo=max(64, hi // 8), hi=hi, log=True,
                     window=rng.choice([0, 0, logint(256, 4096)]),
                     block=rng.choice([16, 16, 32]), lens=lens)
    if work == "prefix":
        hi = logint(8192, 65536)
        prefix = logint(64, 512)
        return _case(work, heads, batch=rng.randint(4, 16), lo=max(hi // 4, prefix * 16), hi=hi,
                     prefix=prefix, lens=lens)
    if work == "chunk":
        hi = logint(256, 3584)
        q, kv = rng.choice([("bf16", "bf16"), ("fp16", "fp16"), ("bf16", "fp8"),
                            ("fp16", "fp8"), ("fp32", "fp32")])
        return _case(work, heads, q=q, kv=kv, batch=rng.randint(1, 2), lo=hi // 2, hi=hi,
                     q_len=rng.randint(64, 512), lens=lens)
    if work == "prompt":
        return _case(work, heads, q=rng.choice(["fp16", "bf16"]), batch=rng.randint(1, 2), lo=0,
                     hi=0, q_len=logint(100, 3000), lens=lens)
    kvh = rng.choice([2, 4, 8])
    return _case("mixed", (kvh * rng.choice([1, 2, 3, 4]), kvh, rng.choice([32, 80, 96, 112, 160,
                                                                          192, 256])),
                 q=rng.choice(["bf16", "fp16"]), batch=1, lo=256, hi=logint(512, 2048),
                 q_len=rng.randint(64, 256), decodes=rng.randint(4, 16), lens=lens)


def _contexts(case, n):
    """Tokens cached before the call, per row."""
    r = random.Random(case["lens"])
    lo, hi = case["lo"], case["hi"]
    if not case["log"]:
        return [r.randint(lo, hi) for _ in range(n)]
    return [min(hi, int(math.exp(r.uniform(math.log(lo), math.log(hi + 1))))) for _ in range(n)]


def _batches(case):
    """[(rows, query tokens per row, context lengths with those tokens)] of one pass."""
    n, t = case["batch"], case["q_len"]
    ctx = _contexts(case, n + case["decodes"])
    if case["work"] in ("decode", "prefix"):  # lengths count the decoded token already
        return [(n, 1, ctx)]
    got = [(n, t, [c + t for c in ctx[:n]])]
    if case["decodes"]:
        got.append((case["decodes"], 1, [c + 1 for c in ctx[n:]]))
    return got


def _visible(case, q_len, length):
    """(keys read, query-key pairs) of a row: causal, with the window if there is one."""
    win = case["window"] or length
    pairs = sum(min(length - q_len + i + 1, win) for i in range(q_len))
    return min(length, win + q_len - 1), pairs


def work(case):
    heads, kvh, d = case["heads"], case["kv_heads"], case["head_dim"]
    qb, kvb = BYTES[case["q"]], BYTES[case["kv"]]
    writes = case["work"] in ("layer", "graph", "prompt")
    nbytes = flops = 0
    for n, t, lengths in _batches(case):
        keys = 0
        for length in lengths:
            k, pairs = _visible(case, t, length)
            keys += k
            flops += 4 * heads * d * pairs
        keys -= (n - 1) * case["prefix"] * case["block"]  # shared pages once
        if writes:
            keys -= n * t  # a new token's row comes from k and v, not from the cache
            nbytes += 2 * n * t * kvh * d * (qb + kvb)
        nbytes += 2 * keys * kvh * d * kvb + 2 * n * t * heads * d * qb
        nbytes += 4 * keys // case["block"] + 4 * n
    return {"bytes": nbytes * case["layers"], "flops": flops * case["layers"]}


def tolerance(case):
    # About four times the measured error against 64 bits: up to 5.4e-7 in fp32 (sums over
    # head_dim and 4.6k keys, more over longer contexts), 2.5e-4 to 2.9e-4 with a 16-bit
    # result in fp16 and 1.6e-3 to 2.3e-3 in bf16 (its rounding and the weights').
    return {"fp32": {"rel": 5e-6}, "fp16": {"rel": 1.2e-3}, "bf16": {"rel": 1e-2}}[case["q"]]


def _randn(gen, shape, dtype):
    x = torch.randn(shape, generator=gen, dtype=torch.float32, device="cuda")
    return x.to(DTYPES[dtype])


def _pages(case, gen_cpu):
    """Block tables of every batch of the pass (CPU, int64, unused entries 0) over one
    pool, and the pool's page count."""
    bs, shared = case["block"], case["prefix"]
    counts = [[-(-length // bs) for length in lengths] for _, _, lengths in _batches(case)]
    need = sum(map(sum, counts)) - max(0, case["batch"] - 1) * shared
    pool = math.ceil(1.25 * need) + 1
    perm = torch.randperm(pool, generator=gen_cpu)
    at, tables = shared, []
    for rows in counts:
        table = torch.zeros(len(rows), max(rows), dtype=torch.int64)
        for b, c in enumerate(rows):
            table[b, :shared] = perm[:shared]
            table[b, shared:c] = perm[at:at + c - shared]
            at += c - shared
        tables.append(table)
    return tables, pool


def prepare(case, seed):
    gen = torch.Generator("cuda").manual_seed(seed)
    tables, pool = _pages(case, torch.Generator("cpu").manual_seed(seed))
    H, KVH, D, L = case["heads"], case["kv_heads"], case["head_dim"], case["layers"]
    bs, q, kv = case["block"], case["q"], case["kv"]
    caches = [(_randn(gen, (pool, bs, KVH, D), kv), _randn(gen, (pool, bs, KVH, D), kv))
              for _ in range(L)]
    pa = PagedAttention(H, KVH, D, num_blocks=pool, block_size=bs, dtype=DTYPES[q],
                        kv_dtype=DTYPES[kv], device="cuda", window=case["window"] or None)
    s = {"case": case, "pa": pa, "caches": caches, "batches": []}
    for (n, t, lengths), table in zip(_batches(case), tables):
        b = {"lens": lengths, "table": table}
        if case["work"] == "graph":
            b["q"] = _randn(gen, (L, n, 1, H, D), q)
            b["k"], b["v"] = (_randn(gen, (L, n, 1, KVH, D), q) for _ in range(2))
            b["lists"] = [row[:-(-length // bs)].tolist() for row, length in zip(table, lengths)]
            b["ctx"] = [length - 1 for length in lengths]
        else:
            # Projections after RoPE are [batch, heads, tokens, dim]; the calls take views.
            b["q"] = _randn(gen, (n, H, t, D), q).transpose(1, 2)
            b["k"] = _randn(gen, (n, KVH, t, D), q).transpose(1, 2)
            b["v"] = _randn(gen, (n, t, KVH, D), q)
            b["starts"] = [length - t for length in lengths]
        if case["work"] in ("layer", "prompt"):
            b["table"] = table.cuda()  # int64, as the runner keeps it
        else:
            b["table"] = table.to(device="cuda", dtype=torch.int32)
            b["dev_lens"] = torch.tensor(lengths, dtype=torch.int32, device="cuda")
            if case["work"] != "graph" and t > 1:
                b["q"] = b["q"].contiguous()
        s["batches"].append(b)
    if case["work"] == "graph":
        b = s["batches"][0]
        layers = [DecodeLayer(pa, kc, vc) for kc, vc in caches]
        n = len(b["lens"])
        bucket = 1 << (n - 1).bit_length()
        s["runner"] = GraphedDecodeRunner(layers, table_width=b["table"].shape[1],
                                          buckets=[bucket], dtype=DTYPES[q])
        # the runner's graphs exist before the first step of a serving program
        s["runner"].decode(b["q"], b["k"], b["v"], b["lists"], b["ctx"])
    return s


def run(s):
    case, pa = s["case"], s["pa"]
    kc, vc = s["caches"][0]
    b = s["batches"][0]
    if case["work"] == "graph":
        out = s["runner"].decode(b["q"], b["k"], b["v"], b["lists"], b["ctx"])
        return [out, [list(pair) for pair in s["caches"]]]
    if case["work"] in ("layer", "prompt"):
        pa.write_kv(kc, vc, b["k"], b["v"], b["table"], start=b["starts"])
        return [pa.forward(b["q"], kc, vc, b["table"], b["lens"]), kc, vc]
    if case["work"] == "prefix":
        return paged_attention(b["q"], kc, vc, b["table"], b["dev_lens"],
                               prefix_pages=case["prefix"])
    return [pa.forward(x["q"], kc, vc, x["table"], x["dev_lens"]) for x in s["batches"]]


def _attend64(case, q, kc, vc, table, lengths):
    """Causal attention in 64 bits over the gathered context, row by row."""
    n, t, H, D = q.shape
    KVH, bs = case["kv_heads"], case["block"]
    out = torch.empty((n, t, H, D), dtype=torch.float64, device=q.device)
    for b, length in enumerate(lengths):
        pages = table[b, :-(-length // bs)].to(q.device, torch.int64)
        pos = torch.arange(length, device=q.device).view(1, 1, length)
        at = (length - t + torch.arange(t, device=q.device)).repeat_interleave(H // KVH)
        at = at.view(1, -1, 1)
        keep = pos <= at
        if case["window"]:
            keep = keep & (pos > at - case["window"])

        def rows(cache):  # [KVH, length, D]
            x = cache[pages].flatten(0, 1)[:length].double()
            return x.transpose(0, 1).contiguous()

        qq = q[b].double().view(t, KVH, H // KVH, D).permute(1, 0, 2, 3).reshape(KVH, -1, D)
        s = torch.bmm(qq.contiguous(), rows(kc).transpose(1, 2).contiguous()) / math.sqrt(D)
        s = s.masked_fill_(~keep, -math.inf).softmax(-1)
        o = torch.bmm(s, rows(vc))
        out[b] = o.view(KVH, t, H // KVH, D).permute(1, 0, 2, 3).reshape(t, H, D)
    return out


def exact(case, seed):
    s = prepare(case, seed)
    b = s["batches"][0]
    if case["work"] == "graph":  # prepare's own step has appended the new tokens
        out = torch.stack([_attend64(case, b["q"][i], kc, vc, b["table"], b["lens"])
                           for i, (kc, vc) in enumerate(s["caches"])])
        return [out, [[None, None] for _ in s["caches"]]]
    kc, vc = s["caches"][0]
    if case["work"] in ("layer", "prompt"):
        bs = case["block"]
        for i, start in enumerate(b["starts"]):
            pos = torch.arange(start, start + case["q_len"], device=kc.device)
            page = b["table"][i][pos // bs]
            kc[page, pos % bs] = b["k"][i].to(kc.dtype)
            vc[page, pos % bs] = b["v"][i].to(vc.dtype)
    outs = [_attend64(case, x["q"], kc, vc, x["table"], x["lens"]) for x in s["batches"]]
    if case["work"] in ("layer", "prompt"):
        return [outs[0], None, None]
    return outs[0] if case["work"] == "prefix" else outs
