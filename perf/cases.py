"""The calls whose time this framework is judged by, through its public entry points.

A case is one attention call of speculative decoding: a batch of requests, each
with ``q_len`` draft tokens, over a paged KV cache. The sizes are those of the
benchmark (``bench.py``), the runner's matrix (``matrix.py``) and the random
sweep of the tests, with odd and ragged lengths among them. Fields:

* ``entry``: ``native`` (``paged_mtp_attention``), ``v3`` / ``v5`` (the drop-in
  ``forward_v3`` / ``forward_v5`` with their default ``chunk_keys``), ``xqa``
  (``xqa_batch_decode_with_kv_cache`` with a packed draft mask) or ``wrapper``
  (``BatchDecodeWithPagedKVCacheWrapper``, planned once, run per layer);
* ``batch``, ``q_len``, ``lo``, ``hi``: KV lengths spread evenly from ``lo`` to
  ``hi`` over the batch, dealt to the requests in an order of the seed;
* ``known``: whether the caller passes the longest length (``native``);
* ``hq``, ``hkv``, ``d``, ``page``; ``dtype`` (fp16, bf16), ``kv`` (the query's
  type or e4m3), ``layout`` (separate caches, interleaved NHD or HND).
"""

import math

import torch

from small_q_attention_amd import cuda as sqa, decode_api
from small_q_attention_amd.masks import pack_draft_mask

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "e4m3": torch.float8_e4m3fn}
POOL = 1.25  # pages of the pool over pages in use: a serving engine keeps some free
WORKSPACE = 128 << 20  # the buffer a caller of the FlashInfer-shaped entries hands over


def _case(name, entry, batch, q_len, lo, hi, *, known=True, hq=32, hkv=8, d=128, page=16,
          dtype="fp16", kv=None, layout="separate"):
    return {"name": name, "entry": entry, "batch": batch, "q_len": q_len, "lo": lo, "hi": hi,
            "known": known, "hq": hq, "hkv": hkv, "d": d, "page": page, "dtype": dtype,
            "kv": kv or dtype, "layout": layout}


def listed():
    return [
        # One short conversation, two draft tokens: the smallest call, all latency.
        _case("one_1k_q2", "native", 1, 2, 1024, 1024),
        # One user at 8K of context, four draft tokens: interactive decoding.
        _case("one_8k_q4", "native", 1, 4, 8192, 8192),
        # The same user's program written for the reference: forward_v3 with its
        # default arguments, the longest length given (the runner's call).
        _case("dropin_one_8k_q2", "v3", 1, 2, 8192, 8192),
        # A small batch of such users (the benchmark's cfg2).
        _case("four_8k_q4", "native", 4, 4, 8192, 8192),
        # The drop-in call at the runner's largest batch, eight draft tokens.
        _case("dropin_16x8k_q8", "v5", 16, 8, 8192, 8192),
        # Long contexts at a serving batch: the benchmark's headline (cfg3).
        _case("sixteen_32k_q8", "native", 16, 8, 32768, 32768),
        # Sixteen draft tokens, the most a request carries.
        _case("sixteen_8k_q16", "native", 16, 16, 8192, 8192),
        # A serving batch as it comes: every request another length (as cfg5).
        _case("ragged_16_q8", "native", 16, 8, 1999, 31973),
        # Many short conversations, lengths on the device only.
        _case("ragged_64_short_q4", "native", 64, 4, 131, 2047, known=False),
        # One rank's share of the heads when four GPUs split a layer.
        _case("shard_16x8k_q4", "native", 16, 4, 8192, 8192, hq=8, hkv=2),
        # FP8 cache with a draft tree per request, one interleaved cache.
        _case("tree_e4m3_16_q8", "xqa", 16, 8, 4099, 16381, kv="e4m3", layout="NHD"),
        # bf16 through a planned wrapper, 64-token pages, head-major cache.
        _case("wrapper_bf16_32_q4", "wrapper", 32, 4, 1031, 8191, page=64, dtype="bf16",
              layout="HND"),
    ]


def _lengths(case):
    b, lo, hi = case["batch"], case["lo"], case["hi"]
    return [hi if b == 1 else lo + (hi - lo) * i // (b - 1) for i in range(b)]


def _cost(case):
    """KV bytes, weighted up where few kv heads or many rows make a call dearer."""
    es = 1 if case["kv"] == "e4m3" else 2
    kv = sum(_lengths(case)) * case["hkv"] * case["d"] * 2 * es
    rows = case["q_len"] * case["hq"] // case["hkv"]
    return kv * (4 / min(case["hkv"], 4)) * (2.5 if rows > 32 else 1) * (1.8 if es == 1 else 1)


def draw(rng):
    entry = rng.choice(["native", "native", "v3", "v5", "xqa", "wrapper"])
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    dropin = entry in ("v3", "v5")
    hkv = rng.choice([1, 2, 4, 8, 8, 8])
    group = 4 if dropin else rng.choice([1, 4, 4, 4, 8])
    d = 128 if dropin else rng.choice([64, 128, 128, 128, 128, 256])
    most = (32 if d == 256 else 64) // group
    if entry in ("xqa", "wrapper"):
        q_len = rng.randint(1, min(16, most))
    else:
        q_len = rng.choice([q for q in (2, 4, 8, 16) if q <= most])
    dtype = "fp16" if dropin else rng.choice(["fp16", "fp16", "bf16"])
    kv = "e4m3" if entry in ("xqa", "wrapper") and rng.random() < 0.4 else dtype
    batch, hi = log(1, 64), log(128, 32768)
    lo = hi if rng.random() < 0.4 else max(q_len, hi // rng.choice([2, 4, 16]))
    c = _case("", entry, batch, q_len, min(lo, hi), hi, known=rng.random() < 0.6,
              hq=hkv * group, hkv=hkv, d=d, page=rng.choice([16, 16, 32, 64, 256]), dtype=dtype,
              kv=kv, layout=rng.choice(["NHD", "HND"]) if entry in ("xqa", "wrapper")
              else "separate")
    limit = _cost(_case("", "native", 16, 8, 32768, 32768)) * 0.95
    while _cost(c) > limit and (c["batch"] > 1 or c["hi"] > 128):
        if c["batch"] > 1:
            c["batch"] = max(1, c["batch"] * 3 // 4)
        else:
            c["hi"] //= 2
            c["lo"] = min(c["lo"], c["hi"])
    if c["batch"] == 1:
        c["lo"] = c["hi"]
    del c["name"]
    return c


def _inputs(case, seed):
    """Query, K and V views ``[pages, page, Hkv, D]`` (of one interleaved tensor or of two
    separate ones), the cache as the entry takes it, block tables, lengths, draft trees."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(int(seed))
    gh = torch.Generator().manual_seed(int(seed))
    b, q_len, hkv, d, page = (case[k] for k in ("batch", "q_len", "hkv", "d", "page"))
    lens = torch.tensor(_lengths(case))[torch.randperm(b, generator=gh)]
    used = (lens + page - 1) // page
    pool = int(math.ceil(int(used.sum()) * POOL))
    perm = torch.randperm(pool, generator=gh).to(torch.int32)
    tables = torch.zeros(b, int(used.max()), dtype=torch.int32)
    at = 0
    for i, n in enumerate(used.tolist()):
        tables[i, :n] = perm[at:at + n]
        at += n
    dt, kdt = DTYPES[case["dtype"]], DTYPES[case["kv"]]
    half = dt if kdt is torch.float8_e4m3fn else kdt

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=dev, dtype=half)

    query = normal(b, q_len, case["hq"], d).to(dt)
    if case["layout"] == "separate":
        cache = (normal(pool, page, hkv, d), normal(pool, page, hkv, d))
        k, v = cache
    else:
        shape = (page, hkv) if case["layout"] == "NHD" else (hkv, page)
        cache = normal(pool, 2, *shape, d)
        k, v = cache[:, 0], cache[:, 1]
        if case["layout"] == "HND":
            k, v = k.transpose(1, 2), v.transpose(1, 2)
    # A few keys stand out, as attention sinks and rare tokens do: four times the
    # others at 1% of the slots.
    hit = torch.rand(pool, page, 1, 1, generator=g, device=dev) < 0.01
    k.mul_(torch.where(hit, 4.0, 1.0).to(half))
    if kdt is not half:
        cache = cache.to(kdt)
        k, v = cache[:, 0], cache[:, 1]
        if case["layout"] == "HND":
            k, v = k.transpose(1, 2), v.transpose(1, 2)
    trees = None
    if case["entry"] == "xqa":
        # Each draft token hangs below an earlier one; a row sees its ancestors.
        parent = torch.rand(b, q_len, generator=gh)
        trees = torch.zeros(b, q_len, q_len, dtype=torch.bool)
        for i in range(q_len):
            trees[:, i, i] = True
            if i:
                up = (parent[:, i] * i).long()
                trees[:, i] |= trees[torch.arange(b), up]
        trees = trees.to(dev)
    return query, cache, k, v, tables.to(dev), lens.to(torch.int32).to(dev), trees


def prepare(case, seed):
    query, cache, _, _, tables, lens, trees = _inputs(case, seed)
    s = {"case": case, "entry": case["entry"], "page": case["page"], "query": query,
         "cache": cache, "tables": tables, "lens": lens, "most": case["hi"],
         "q_len": case["q_len"], "scale": case["d"] ** -0.5, "layout": case["layout"]}
    if case["entry"] in ("v3", "v5"):
        (sqa.load_v3 if case["entry"] == "v3" else sqa.load_v5)()
    elif case["entry"] in ("xqa", "wrapper"):
        s["query"] = query.view(-1, case["hq"], case["d"])
        s["workspace"] = torch.zeros(WORKSPACE, dtype=torch.uint8, device="cuda")
    if case["entry"] == "xqa":
        s["mask"] = pack_draft_mask(trees)
    if case["entry"] == "wrapper":
        page = case["page"]
        used = (lens.long() + page - 1) // page
        indptr = torch.zeros(case["batch"] + 1, dtype=torch.int32, device="cuda")
        indptr[1:] = used.cumsum(0)
        indices = tables[torch.arange(tables.shape[1], device="cuda")[None] < used[:, None]]
        w = decode_api.BatchDecodeWithPagedKVCacheWrapper(s["workspace"], case["layout"])
        w.plan(indptr, indices, (lens - (used - 1) * page).to(torch.int32), case["hq"],
               case["hkv"], case["d"], page, q_data_type=DTYPES[case["dtype"]],
               kv_data_type=DTYPES[case["kv"]], q_len_per_req=case["q_len"])
        s["wrapper"] = w
    return s


def run(s):
    entry = s["entry"]
    if entry == "xqa":
        return decode_api.xqa_batch_decode_with_kv_cache(
            s["query"], s["cache"], s["workspace"], s["tables"], s["lens"], s["most"], s["scale"],
            1.0, kv_layout=s["layout"], q_len_per_req=s["q_len"], mask=s["mask"])
    if entry == "wrapper":
        return s["wrapper"].run(s["query"], s["cache"])
    k, v = s["cache"]
    if entry == "v3":
        return sqa.forward_v3(s["query"], k, v, s["tables"], s["lens"], s["page"],
                              max_seq_len=s["most"])
    if entry == "v5":
        return sqa.forward_v5(s["query"], k, v, s["tables"], s["lens"], s["page"],
                              max_seq_len=s["most"])
    return sqa.paged_mtp_attention(s["query"], k, v, s["tables"], s["lens"], s["page"],
                                   max_seq_len=s["most"] if s["case"]["known"] else 0)


def work(case):
    """K and V of every key once, the query, the output, the block tables and lengths."""
    lens = _lengths(case)
    es = 1 if case["kv"] == "e4m3" else 2
    kv = sum(lens) * case["hkv"] * case["d"] * 2 * es
    qo = 2 * case["batch"] * case["q_len"] * case["hq"] * case["d"] * 2
    tables = 4 * sum(-(-n // case["page"]) for n in lens) + 4 * case["batch"]
    q = case["q_len"]
    seen = sum(q * n - q * (q - 1) // 2 for n in lens)  # the draft chain
    return {"bytes": kv + qo + tables, "flops": 4 * case["hq"] * case["d"] * seen}


def tolerance(case):
    # fp16: probabilities, partial rows and outputs carry 11 bits each; bf16
    # outputs 8. Four times the error against 64 bits that the calls show (3e-4
    # and 1.7e-3).
    return {"rel": 1.2e-3, "max": 1e-2} if case["dtype"] == "fp16" else {"rel": 7e-3, "max": 4e-2}


def exact(case, seed):
    query, _, k, v, tables, lens, trees = _inputs(case, seed)
    b, q_len, hq, d = query.shape
    hkv, page = case["hkv"], case["page"]
    group = hq // hkv
    out = torch.zeros(b, q_len, hq, d, dtype=torch.float64, device=query.device)
    for i, n in enumerate(lens.tolist()):
        ids = tables[i, :-(-n // page)].long()
        # [Hkv, keys, D], contiguous, in 64 bits.
        ki = k.view(torch.uint8)[ids].view(k.dtype) if k.element_size() == 1 else k[ids]
        vi = v.view(torch.uint8)[ids].view(v.dtype) if v.element_size() == 1 else v[ids]
        ki, vi = (x.reshape(-1, hkv, d)[:n].to(torch.float64).transpose(0, 1).contiguous()
                  for x in (ki, vi))
        qi = query[i].to(torch.float64).view(q_len, hkv, group, d).permute(1, 0, 2, 3)
        s = qi.reshape(hkv, q_len * group, d) @ ki.transpose(1, 2).contiguous() * d ** -0.5
        seen = torch.ones(q_len, n, dtype=torch.bool, device=query.device)
        chain = torch.ones(q_len, q_len, dtype=torch.bool, device=query.device).tril()
        seen[:, n - q_len:] = chain if trees is None else trees[i]
        s = s.masked_fill(~seen.repeat_interleave(group, 0)[None], float("-inf"))
        o = torch.softmax(s, -1) @ vi
        out[i] = o.view(hkv, q_len, group, d).permute(1, 0, 2, 3).reshape(q_len, hq, d)
    return out.view(b * q_len, hq, d) if case["entry"] in ("xqa", "wrapper") else out
