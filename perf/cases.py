"""The workloads by which this framework's speed is judged, and the ranges they stand for.

Every case goes through the entry points a user's program calls: ``DiffCache`` (prefill, the native
``decode_attention``, the three hooks of the reference's harness, a captured step) and the PQ
baseline (``PQIndex.search``, ``encode``).  A case is a dict of plain values:

  kind      decode   one token through every layer of a cache, eager calls
            graph    the same step captured once in a HIP graph and replayed
            hooks    the reference's three hooks per layer (group mean, scan + select best first,
                     row gather into the assembled buffer)
            prefill  a prompt's keys and values into every layer of a cache
            search   one PQ search of every unit
            encode   PQ codes of new keys
  layers, batch, hq, hkv, hd, ctx, budget, sketch, mode, sink, recent, window   (cache kinds)
  batch, hkv, hd, n, m, n_cand, topk                                            (PQ kinds)
"""
import math

import torch

from diffcache_amd import DiffCache
from diffcache_amd import _hip as hip
from diffcache_amd.pq import PQIndex, encode

DEV = "cuda"


def _cache(name, kind, layers, batch, hq, hkv, hd, ctx, budget, sketch=True, mode="ref_dist", sink=4, recent=64,
           window=128):
    return dict(name=name, kind=kind, layers=layers, batch=batch, hq=hq, hkv=hkv, hd=hd, ctx=ctx, budget=budget,
                sketch=sketch, mode=mode, sink=sink, recent=recent, window=window)


def listed():
    return [
        # a chat turn: one sequence of a few thousand tokens, where launches and host work count
        _cache("chat_4k", "decode", 8, 1, 32, 8, 128, 4096, 512),
        # one sequence of about 32K tokens (benchmark configuration 2, several layers of it)
        _cache("doc_32k", "decode", 4, 1, 32, 8, 128, 32601, 1024),
        # one long document
        _cache("doc_128k", "decode", 4, 1, 32, 8, 128, 131072, 2048),
        # batched serving at 128K (benchmark configuration 3, two of its layers)
        _cache("serve_8x128k", "decode", 2, 8, 32, 8, 128, 131072, 2048),
        # one sequence of a million tokens (benchmark configuration 5, one of its layers)
        _cache("book_1m", "decode", 1, 1, 32, 8, 128, 1048576, 4096),
        # a cache without the sketch (no memory to spare), plain inner-product order, ragged length
        _cache("bf16_4x50k", "decode", 2, 4, 32, 8, 128, 50001, 2048, sketch=False, mode="ip"),
        # wide heads, few of them, odd batch and length
        _cache("wide_3x24k", "decode", 2, 3, 16, 4, 256, 24683, 1024),
        # a serving loop that captured its decode step: small batch, narrow heads, middling length
        _cache("graph_2x16k", "graph", 4, 2, 32, 4, 64, 16391, 1024),
        # the reference's own harness (hooks, best-first rows; its Qwen2.5-7B shapes and buffer sizes)
        _cache("hooks_127k", "hooks", 4, 1, 28, 4, 128, 127284, 1024, sink=128, recent=128, window=512),
        # prompts entering the cache
        _cache("prefill_2x40k", "prefill", 2, 2, 32, 8, 128, 40003, 1024),
        # PQ baseline (benchmark configuration 4)
        dict(name="pq_search_1m", kind="search", batch=1, hkv=8, hd=128, n=1 << 20, m=32, n_cand=4096, topk=1024),
        # PQ baseline: codes of a long prompt's keys (one head)
        dict(name="pq_encode_200k", kind="encode", batch=1, hkv=1, hd=128, n=200003, m=32, n_cand=0, topk=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_MOST = 2 * 64 * 131072 * 128   # key elements of the largest listed decode step


def draw(rng):
    kind = rng.choice(["decode"] * 6 + ["graph", "hooks", "prefill", "prefill", "search", "encode"])
    if kind == "search":
        while True:
            c = dict(kind=kind, batch=rng.choice([1, 1, 2]), hkv=rng.choice([2, 4, 8]), hd=rng.choice([64, 128]),
                     n=_log_int(rng, 1 << 15, 1 << 20), m=rng.choice([16, 32]), n_cand=rng.choice([1024, 2048, 4096]),
                     topk=rng.choice([256, 512, 1024]))
            if c["batch"] * c["hkv"] * c["n"] <= 8 << 20:
                return c
    if kind == "encode":
        return dict(kind=kind, batch=1, hkv=1, hd=rng.choice([64, 128]), n=_log_int(rng, 5000, 200000),
                    m=rng.choice([16, 32]), n_cand=0, topk=0)
    while True:
        hd = rng.choice([64, 128, 128, 128, 256])
        hkv = rng.choice([2, 4, 8])
        group = rng.choice([1, 4, 4, 4, 7, 8])
        batch = _log_int(rng, 1, 16)
        layers = rng.choice([1, 2, 4, 8])
        ctx = _log_int(rng, 2048, 1 << 20)
        if kind == "prefill":
            ctx = _log_int(rng, 2048, 1 << 17)
        budget = rng.choice([256, 512, 1024, 2048, 4096])
        cost = layers * batch * hkv * ctx * hd
        if budget * 4 > ctx or cost > (_MOST // 8 if kind == "prefill" else _MOST):
            continue
        sketch = rng.random() < 0.75
        if cost > _MOST // 2 and not sketch:
            continue
        sink, recent, window = (128, 128, 512) if kind == "hooks" else (4, 64, 128)
        c = _cache("", kind, layers, batch, hkv * group, hkv, hd, ctx, budget, sketch,
                   rng.choice(["ref_dist", "ref_dist", "ip"]), sink, recent, window)
        del c["name"]
        if kind == "prefill" or _fits(c):
            return c


def _room(case):
    """Rows of the store beyond the prompt: the recent window's, and for a captured step, which is laid
    out for a whole generation, a quarter of the prompt."""
    return max(case["window"], case["ctx"] // 4) if case["kind"] == "graph" else case["window"]


def _fits(case):
    """A cache sizes its workspace for the longest region its store can hold; a region of a length that
    would need more than that one (a layout with more blocks per unit) is left out."""
    region = case["ctx"] - case["sink"] - case["recent"]
    rows = case["budget"] + case["sink"] + case["window"] + 1
    need = [hip.layer_workspace_bytes(case["batch"] * case["hkv"], n, case["budget"], case["hq"] // case["hkv"],
                                      case["hd"], rows) for n in (region, region + _room(case))]
    return need[0] <= need[1]


def _prompt(case, g):
    """Keys with per-channel log-normal scales (outlier channels), values ~ N(0, 1)."""
    b, n, h, d = case["batch"], case["ctx"], case["hkv"], case["hd"]
    k = torch.empty((b, n, h, d), device=DEV, dtype=torch.bfloat16).normal_(generator=g)
    k.mul_(torch.exp(torch.randn((1, 1, h, d), generator=g, device=DEV)).to(torch.bfloat16))
    v = torch.empty((b, n, h, d), device=DEV, dtype=torch.bfloat16).normal_(generator=g)
    return k, v


def _queries(case, k, g):
    """Every query head leans towards the mean of 32 random keys of its kv head."""
    b, n, h, d = k.shape
    hq = case["hq"]
    pick = torch.randint(0, n, (b, hq, 32), generator=g, device=DEV)
    bi = torch.arange(b, device=DEV).view(b, 1, 1)
    hi = (torch.arange(hq, device=DEV) // (hq // h)).view(1, hq, 1)
    centre = k[bi, pick, hi].float().mean(dim=2)
    return (0.7 * centre + 0.3 * torch.randn((b, hq, d), generator=g, device=DEV)).to(torch.bfloat16)


def _prepare_cache(case, g):
    layers, b, hq, hkv, hd, ctx = (case[x] for x in ("layers", "batch", "hq", "hkv", "hd", "ctx"))
    cache = DiffCache(num_layers=layers, batch_size=b, max_length=ctx + _room(case), num_kv_heads=hkv, num_q_heads=hq,
                      head_dim=hd, retrieval_budget=case["budget"], nsw_m=16, nsw_ef_cons=200,
                      kvbuf_prefix_len=case["sink"], kvbuf_suffix_len=case["recent"],
                      kvbuf_suffix_maxlen=case["window"], attn_mass_threshold=0.9, k_check_seq=[100, 200, 400, 800],
                      r_sq=[[4.0] * hkv for _ in range(layers)], key_mode=case["mode"], key_sketch=case["sketch"])
    s = dict(case=case, cache=cache)
    if case["kind"] == "prefill":
        s["kv"] = [_prompt(case, g) for _ in range(layers)]
        return s
    s["q"], s["k"], s["v"], s["out"] = [], [], [], []
    # the rows of the store that the step's token goes to
    s["rows"] = [(ks[:, :, ctx], vs[:, :, ctx]) for ks, vs in zip(cache.kstore, cache.vstore)]
    for layer in range(layers):
        k, v = _prompt(case, g)
        cache.prefill_update_kv_cache(k, v, layer)
        s["q"].append(_queries(case, k, g))
        s["k"].append(torch.randn((b, 1, hkv, hd), generator=g, device=DEV).to(torch.bfloat16))
        s["v"].append(torch.randn((b, 1, hkv, hd), generator=g, device=DEV).to(torch.bfloat16))
        s["out"].append(torch.empty((b, hq, hd), device=DEV, dtype=torch.bfloat16))
        del k, v
    if case["kind"] == "graph":
        _step(s)            # workspaces are laid out on the first step
        _take_back(s)
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            _step(s)
    return s


def _prepare_pq(case, g):
    b, h, hd, n, m = (case[x] for x in ("batch", "hkv", "hd", "n", "m"))
    ds = hd // m
    books = torch.randn((h, m, 256, ds), generator=g, device=DEV)
    codes = torch.randint(0, 256, (b * h, n, m), generator=g, device=DEV, dtype=torch.uint8)
    keys = torch.empty((b, h, n, hd), device=DEV, dtype=torch.bfloat16)
    first = (torch.arange(m, device=DEV) * 256).view(1, m)
    for u in range(b * h):     # keys scatter around the points their codes name, as trained codebooks leave them
        near = books[u % h].reshape(m * 256, ds)[codes[u].long() + first].view(n, hd)
        keys[u // h, u % h] = near + 0.3 * torch.randn((n, hd), generator=g, device=DEV)
    if case["kind"] == "encode":
        return dict(case=case, keys=keys[0, 0].contiguous(), books=books[0].contiguous())
    q = torch.randn((b * h, hd), generator=g, device=DEV).to(torch.bfloat16)
    return dict(case=case, q=q, index=PQIndex(keys, books, codes, n_cand=case["n_cand"], topk=case["topk"]))


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    return _prepare_pq(case, g) if case["kind"] in ("search", "encode") else _prepare_cache(case, g)


def _step(s):
    for layer in range(s["case"]["layers"]):
        s["cache"].decode_attention(layer, s["q"][layer], s["k"][layer], s["v"][layer], out=s["out"][layer])


def _take_back(s):
    """The token just decoded is taken back (as a rejected draft token is), so that every pass finds the
    window as the first one did."""
    s["cache"].advance_host_step(-1)
    hip.step_advance(s["cache"].step_state, -1)


def run(s):
    kind = s["case"]["kind"]
    if kind == "search":
        return s["index"].search(s["q"])
    if kind == "encode":
        return encode(s["keys"], s["books"])
    cache = s["cache"]
    if kind == "decode":
        _step(s)
        _take_back(s)
        return s["out"], s["rows"]
    if kind == "graph":
        s["graph"].replay()
        cache.advance_host_step(1)
        _take_back(s)
        return s["out"], s["rows"]
    layers, b0 = s["case"]["layers"], s["case"]["budget"]
    if kind == "hooks":
        for layer in range(layers):
            cache.decode_pre_query_operation(s["q"][layer])
            cache.decode_query_kvcache(layer)
            cache.decode_post_query_operation(layer)
        cache.kvbuf_suffix_len -= 1
        hip.step_advance(cache.step_state, -1)
        return [(cache.kbuf[layer][:, :, :b0], cache.vbuf[layer][:, :, :b0]) for layer in range(layers)]
    for layer in range(layers):
        cache.prefill_update_kv_cache(s["kv"][layer][0], s["kv"][layer][1], layer)
    kept = b0 + cache.kvbuf_prefix_len + cache.kvbuf_suffix_len
    out = [(cache.kstore[layer], cache.vstore[layer], cache.kbuf[layer][:, :, b0:kept], cache.vbuf[layer][:, :, b0:kept])
           for layer in range(layers)]
    if s["case"]["sketch"]:
        out += [(sk.codes, sk.scale, sk.resid) for sk in cache.sketch]
    return out


def work(case):
    kind = case["kind"]
    if kind in ("search", "encode"):
        units, n, hd, m = case["batch"] * case["hkv"], case["n"], case["hd"], case["m"]
        books = case["hkv"] * 256 * hd * 4
        if kind == "encode":    # keys in, codes out, every key against every centroid
            return {"bytes": n * (2 * hd + m) + books, "flops": 2.0 * 256 * n * hd}
        # every code once, the candidates' keys, the tables
        return {"bytes": units * (n * m + case["n_cand"] * hd * 2 + case["topk"] * 4) + books,
                "flops": 1.0 * units * (n * m + 2 * case["n_cand"] * hd + 2 * 256 * hd)}
    layers, b, hq, hkv, hd, ctx = (case[x] for x in ("layers", "batch", "hq", "hkv", "hd", "ctx"))
    units = b * hkv
    if kind == "prefill":       # keys and values in, both into the store, one code byte per key element
        per = 8 + (1 if case["sketch"] else 0)
        return {"bytes": 1.0 * layers * units * ctx * hd * per, "flops": 8.0 * layers * units * ctx * hd}
    region = ctx - case["sink"] - case["recent"]
    k = min(case["budget"], region)
    scan = region * hd * (1 if case["sketch"] else 2)
    score = 2 * region * hd
    if kind == "hooks":         # the scan, and the selected K and V rows copied
        return {"bytes": layers * (units * (scan + 2 * 2 * k * hd * 2) + b * hq * hd * 2), "flops": 1.0 * layers * units * score}
    rows = k + case["sink"] + case["recent"] + 1
    return {"bytes": layers * (units * (scan + 2 * rows * hd * 2) + 2 * b * hq * hd * 2),
            "flops": 1.0 * layers * (units * score + b * hq * 4 * rows * hd)}


def tolerance(case):
    if case["kind"] in ("hooks", "prefill", "search"):
        return "exact"          # ids, and copies of rows; the sketch is defined element by element
    if case["kind"] == "encode":
        # keys as far from one centroid as from another, to fp32 (5e-7 of the codes against 64 bits)
        return {"rel": 0.0, "differ": 2e-6 + 2.0 / (case["n"] * case["m"])}
    return {"rel": 7e-3, "max": 1.6e-2}         # attention rounded to bf16 (1.7e-3 and 3.9e-3 against 64 bits)
