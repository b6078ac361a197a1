"""Performance cases: the model steps and retrieval calls that a deployment of this framework spends its GPU time on.

A chat turn embeds the query (bge), searches the transaction collection, prefills prompts behind cached prefixes and
decodes replies; the layered hybrid decoders serve the same steps through their own mixers.  ``listed()`` holds fixed
cases, ``draw()`` more of the same ranges; ``run()`` makes one call and ``exact()`` is its value in float64, written from
the models' equations in plain torch.  Weights, caches and states come from the seed alone.
"""
from __future__ import annotations

import dataclasses
import math
import random
import zlib

import torch

from financial_chatbot_llm_amd import ops
from financial_chatbot_llm_amd.models.bert import BertEncoder
from financial_chatbot_llm_amd.models.common import AttentionMetadata, KVCache
from financial_chatbot_llm_amd.models.configs import get_model_config, layered_config
from financial_chatbot_llm_amd.models.fanotar import FanotarModel, example_config as fanotar_config
from financial_chatbot_llm_amd.models.gezavik import GezavikModel, example_config as gezavik_config
from financial_chatbot_llm_amd.models.llama import LlamaModel
from financial_chatbot_llm_amd.models.mixtral import MixtralModel
from financial_chatbot_llm_amd.models.sigudra import SigudraModel, example_config as sigudra_config
from financial_chatbot_llm_amd.ops.attention import LEAN_NT_MIN_B, DecodeWorkspace, mark_shared_blocks, prefill_plan

DEV = "cuda"
F64 = torch.float64
PAGE = 64
NOW = 1_760_000_000          # newest transaction date of the synthetic collection
LAYERED = {"gezavik": (GezavikModel, gezavik_config, "aMmAmMaM"), "sigudra": (SigudraModel, sigudra_config, "dGPgDpdG"),
           "fanotar": (FanotarModel, fanotar_config, "AEkKAEkK")}


def listed():
    return [
        # the query of one chat turn: the smallest call of the serving path, all launch latency
        {"name": "embed-one-query", "kind": "embed", "texts": 1, "longest": 18},
        # bulk ingest of transactions: one batch of documents as the ingest loop makes them
        {"name": "embed-ingest-batch", "kind": "embed", "texts": 1024, "longest": 64},
        # the micro-batched searches of concurrent turns: every user's own rows since a date, no limit sent
        {"name": "search-16-users", "kind": "search", "queries": 16, "rows": 1_000_000, "users": 10_000, "limit": 10_000},
        # one user alone: a reply token of a short conversation (all 8B weights for one row)
        {"name": "chat-decode-1", "kind": "chat", "chunks": 0, "new": 0, "cached": 0, "rows": 1, "ctx": 900, "shared": 0},
        # the server under load: one reply token for each of 64 conversations behind one system prompt
        {"name": "chat-decode-64", "kind": "chat", "chunks": 0, "new": 0, "cached": 0, "rows": 64, "ctx": 3900, "shared": 1024},
        # a mixed step: new turns' prompts behind their cached history, beside the rows that decode
        {"name": "chat-prefill-mixed", "kind": "chat", "chunks": 5, "new": 433, "cached": 2600, "rows": 40, "ctx": 3500, "shared": 1024},
        # sparse experts in fp8: one reply token for 48 conversations (4 of Mixtral's 32 equal layers)
        {"name": "moe-decode-48", "kind": "moe", "chunks": 0, "new": 0, "cached": 0, "rows": 48, "ctx": 1200, "shared": 0},
        # hybrid decoders: two whole prompts; 64 rows decoding; ragged prompts of odd lengths; a single row; a prompt's
        # later portion behind its cache; and float32, in which traces are replayed
        {"name": "gezavik-prefill", "kind": "gezavik", "width": 2048, "dtype": "bf16", "chunks": 2, "new": 2048, "cached": 0, "rows": 0, "ctx": 0},
        {"name": "gezavik-decode-64", "kind": "gezavik", "width": 2048, "dtype": "bf16", "chunks": 0, "new": 0, "cached": 0, "rows": 64, "ctx": 1100},
        {"name": "sigudra-prefill-ragged", "kind": "sigudra", "width": 2048, "dtype": "bf16", "chunks": 3, "new": 1223, "cached": 0, "rows": 0, "ctx": 0},
        {"name": "sigudra-fp32-replay", "kind": "sigudra", "width": 1024, "dtype": "fp32", "chunks": 1, "new": 333, "cached": 0, "rows": 5, "ctx": 700},
        {"name": "fanotar-mixed", "kind": "fanotar", "width": 2048, "dtype": "bf16", "chunks": 3, "new": 389, "cached": 1500, "rows": 21, "ctx": 1300},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["embed", "search", "chat", "moe", "gezavik", "gezavik", "sigudra", "sigudra", "fanotar", "fanotar"])
    if kind == "embed":
        return {"kind": kind, "texts": _log(rng, 1, 1024), "longest": rng.randint(6, 64)}
    if kind == "search":
        return {"kind": kind, "queries": _log(rng, 1, 64), "rows": _log(rng, 20_000, 1_000_000), "users": _log(rng, 200, 10_000),
                "limit": _log(rng, 4, 10_000)}
    c = {"kind": kind, "chunks": 0, "new": 0, "cached": 0, "rows": 0, "ctx": 0}
    big = kind in ("chat", "moe")
    mode = rng.choice(["prefill", "decode", "mixed"])
    if mode != "decode":
        c["chunks"] = rng.randint(1, 6)
        c["new"] = max(1, _log(rng, 24, 2048 if big else 4096) // c["chunks"])
        c["cached"] = rng.choice([0, _log(rng, 64, 2600 if big else 1500)])
    if mode != "prefill":
        c["rows"] = _log(rng, 1, 64)
        c["ctx"] = _log(rng, 100, 3900 if big else 1500)
    if big:
        c["shared"] = rng.choice([0, 256, 1024])
        return c
    c["dtype"] = rng.choice(["bf16", "bf16", "bf16", "fp32"])
    c["width"] = 1024 if c["dtype"] == "fp32" else rng.choice([1024, 2048])
    if c["dtype"] == "fp32":       # traces are short
        c["new"] = min(c["new"], 200)
    return c


# ----------------------------------------------------------------------------------------------
# inputs
# ----------------------------------------------------------------------------------------------
def _rand(seed, tag, shape, scale=1.0, dtype=torch.bfloat16, uniform=False):
    g = torch.Generator(device=DEV).manual_seed((seed * 1_000_003 + zlib.crc32(tag.encode())) & 0x7FFFFFFF)
    t = (torch.rand if uniform else torch.randn)(shape, generator=g, device=DEV, dtype=dtype)
    return t if scale == 1.0 else t.mul_(scale)


def _tokens(seed, tag, n, vocab):
    return _rand(seed, tag, (n,), dtype=torch.float32, uniform=True).mul_(vocab).to(torch.int64).clamp_(0, vocab - 1)


def _segments(case):
    """(first position, new tokens) of every chunk and decode row: ragged, the same for every seed."""
    r = random.Random("%(chunks)d %(new)d %(cached)d %(rows)d %(ctx)d" % case)
    segs = []
    for _ in range(case["chunks"]):
        n = max(1, int(case["new"] * r.uniform(0.6, 1.4))) if case["chunks"] > 1 else case["new"]
        segs.append((int(case["cached"] * r.uniform(0.5, 1.5)) if case["cached"] else 0, n))
    for _ in range(case["rows"]):
        segs.append((max(1, int(case["ctx"] * r.uniform(0.4, 1.6))) if case["rows"] > 1 else case["ctx"], 1))
    return segs


def _layout(case, segs):
    """Page table of every segment: the first ``shared`` tokens of those that are long enough lie on common pages."""
    shared = case.get("shared", 0) // PAGE
    pages, top = [], shared
    for start, n in segs:
        need = -(-(start + n) // PAGE)
        common = shared if start >= shared * PAGE else 0
        pages.append(list(range(common)) + list(range(top, top + need - common)))
        top += need - common
    return pages, top


def _batch(case, segs, vocab, seed):
    """Flat ids, positions and cache slots of a step."""
    pages, total = _layout(case, segs)
    pos = torch.cat([torch.arange(s, s + n) for s, n in segs])
    slots = torch.cat([torch.tensor(p)[torch.arange(s, s + n) // PAGE] * PAGE + torch.arange(s, s + n) % PAGE
                       for p, (s, n) in zip(pages, segs)])
    ids = _tokens(seed, "ids", len(pos), vocab)
    cu = torch.tensor([0] + [n for _, n in segs]).cumsum(0)
    return ids, pos, slots, cu, pages, total


def _table(pages):
    bt = torch.zeros((len(pages), max((len(p) for p in pages), default=1)), dtype=torch.int32)
    for i, p in enumerate(pages):
        bt[i, :len(p)] = torch.tensor(p, dtype=torch.int32)
    return bt


def _i32(t):
    return t.to(device=DEV, dtype=torch.int32)


def _big_config(kind):
    c = get_model_config("llama3-8b" if kind == "chat" else "mixtral-8x7b")
    return c if kind == "chat" else dataclasses.replace(c, num_layers=4)


def _big_weight(name, shape, seed):
    """Weights of the usual initialisation: each block's output projections smaller, so that the residual stream leads;
    a router that decides (near-ties between experts are rare in a trained one)."""
    if name.endswith("norm"):
        return _rand(seed, name, shape, 0.1).add_(1.0)
    leaf = name.rsplit(".", 1)[-1]
    return _rand(seed, name, shape, {"embed": 1.0, "o": 0.0025, "down": 0.0025, "w2": 0.001, "router": 0.06}.get(leaf, 0.02))


def _big_kv(cfg, layer, n, seed):
    """Cached keys (rotated) and values of one layer, [slots, kv heads * dim] each."""
    return [_rand(seed, f"{kv}{layer}", (n, cfg.kv_size), 1.3) for kv in "kv"]


def _layer_config(case):
    _, config, pattern = LAYERED[case["kind"]]
    return config(width=case["width"], vocab=32768, pattern=pattern, scale_up=True,
                  **({"heads": case["width"] // 128} if case["kind"] == "gezavik" else {}))


def _layer_value(name, shape, seed, kind):
    """One checkpoint tensor of a layered decoder (bf16), each kind of parameter in its usual range.  Single experts add
    little to the residual stream (a token whose chosen experts nearly tie may go either way): their output is small,
    as are the norms that Sigudra puts on each sublayer's output, and Gezavik's softmax router decides."""
    leaf = name.rsplit(".", 1)[-1]
    f = lambda uniform=False: _rand(seed, name, shape, dtype=torch.float32, uniform=uniform)  # noqa: E731
    if leaf in ("norm", "norm1", "norm2", "norm1b", "norm2b", "out") and len(shape) == 1:
        t = (1.0 + 0.1 * f()) * ({"norm1": 0.25, "norm2": 0.08}.get(leaf, 1.0) if kind == "sigudra" else 1.0)
    elif leaf == "alpha":
        t = 0.4 + 0.4 * f(True)
    elif leaf == "A_log":
        t = torch.log(1.0 + 7.0 * f(True))
    elif leaf == "dt_bias":           # step sizes in [0.01, 0.2] before the softplus
        dt = torch.exp(f(True) * math.log(20.0) + math.log(0.01))
        t = dt + torch.log(-torch.expm1(-dt))
    elif leaf == "lam":
        t = torch.log(torch.expm1(torch.exp(f(True) * math.log(60.0) + math.log(0.01))))
    elif leaf == "D":
        t = 1.0 + 0.2 * f()
    elif leaf == "correction":
        t = 0.05 * f()
    elif name.endswith("a2.b"):
        t = 2.0 + 0.5 * f()
    elif leaf == "b" and (len(shape) == 1 or name.endswith(("ra.b", "ri.b"))):
        t = 0.1 * f()
    elif leaf == "conv":
        t = f() * shape[1] ** -0.5
    elif leaf in ("embed", "bigram", "sink"):
        t = f()
    else:
        t = f() * shape[-1] ** -0.5
        if leaf == "down" and ".e" in name:
            t = 0.15 * t
        elif leaf == "router" and kind == "gezavik":
            t = 3.0 * t
    return t.to(torch.bfloat16)


def _layer_model(case):
    cls = LAYERED[case["kind"]][0]
    return cls(layered_config(_layer_config(case)), device=DEV, dtype=torch.float32 if case["dtype"] == "fp32" else torch.bfloat16)


def _entries(layers):
    """(kind, tensors) of every cache entry of a hybrid cache, pairs taken apart."""
    for e in layers:
        if e[0] == "pair":
            yield from _entries(e[1:])
        elif e[0] == "slots":
            yield "slots", [e[1][k] for k in sorted(e[1])]
        elif e[0] == "state":
            yield "slots", [e[1], e[2]]
        elif e[0] != "none":
            yield "rows", [e[1]]


def _fill(cache, seed):
    """Cached rows and states as an earlier part of the sequences leaves them: rows of unit size, smaller states."""
    i = 0
    for kind, ts in _entries(cache.layers):
        for t in ts:
            t.copy_(_rand(seed, f"cache{i}", tuple(t.shape), 0.8 if kind == "rows" else 0.3, dtype=torch.float32))
            i += 1
    if "last_token" in cache.model:
        cache.model["last_token"].copy_(_tokens(seed, "last", cache.num_slots, 32768))


def _search_inputs(case, seed):
    n, q, d = case["rows"], case["queries"], 768
    corpus = torch.empty((n, d), dtype=torch.bfloat16, device=DEV)
    for a in range(0, n, 1 << 18):
        x = _rand(seed, f"rows{a}", (min(1 << 18, n - a), d), dtype=torch.float32)
        corpus[a:a + x.shape[0]] = torch.nn.functional.normalize(x, dim=-1)
    users = _tokens(seed, "users", n, case["users"]).to(torch.int32)
    dates = NOW - _tokens(seed, "dates", n, 365 * 86400)
    queries = torch.nn.functional.normalize(_rand(seed, "queries", (q, d), dtype=torch.float32), dim=-1).to(torch.bfloat16)
    who = _tokens(seed, "who", q, case["users"]).to(torch.int32)
    since = NOW - 86400 * torch.where(torch.arange(q, device=DEV) % 3 == 0, 365, 30 + 7 * torch.arange(q, device=DEV) % 300)
    return corpus, users, dates, queries, who, since, torch.full((q,), case["limit"], dtype=torch.int32, device=DEV)


def _texts(case, seed):
    """Token ids of every text, [CLS] .. [SEP]."""
    r = random.Random("%d %d" % (case["texts"], case["longest"]))
    lens = [case["longest"]] + [r.randint(min(6, case["longest"]), case["longest"]) for _ in range(case["texts"] - 1)]
    flat = (_tokens(seed, "text", sum(lens), 29_000) + 1000).tolist()
    out = []
    for n in lens:
        out.append([101] + flat[:n - 2] + [102])
        flat = flat[n:]
    return out


def _bert_weight(name, shape, seed):
    t = _rand(seed, name, shape, 0.05 if name.endswith("_emb") else 0.03)
    return t.add_(1.0) if name.endswith("_g") else t


# ----------------------------------------------------------------------------------------------
# preparing and running
# ----------------------------------------------------------------------------------------------
def _forward(s):
    h = s["model"].forward(s["ids"], s["pos"], s["meta"], s["kv"])
    return {"hidden": h, "logits": s["model"].logits(h.index_select(0, s["last"]))}


def _capture(s, restore):
    """The step as one graph, as a serving loop keeps it per batch size; what the trial runs wrote is put back."""
    for _ in range(2):
        _forward(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        s["out"] = _forward(s)
    s["graph"] = g
    restore()
    torch.cuda.synchronize()


@torch.no_grad()
def prepare(case, seed):
    kind = case["kind"]
    if kind == "embed":
        m = BertEncoder(get_model_config("bge-base-en"), DEV)
        m.load_state({n: _bert_weight(n, sh, seed) for n, sh in m.shapes().items()})
        return {"kind": kind, "model": m, "texts": _texts(case, seed)}
    if kind == "search":
        return {"kind": kind, "args": _search_inputs(case, seed), "kmax": case["limit"]}
    segs = _segments(case)
    big = kind in ("chat", "moe")
    cfg = _big_config(kind) if big else None
    ids, pos, slots, cu, pages, total = _batch(case, segs, cfg.vocab_size if big else 32768, seed)
    nc, nd = case["chunks"], case["rows"]
    s = {"kind": kind, "ids": _i32(ids), "pos": _i32(pos), "last": (cu[1:] - 1).to(DEV)}
    tp = int(cu[nc])
    meta = AttentionMetadata(slots=_i32(slots), num_prefill_tokens=tp, num_decode=nd)
    s["meta"] = meta
    if big:
        m = LlamaModel(cfg, device=DEV) if kind == "chat" else MixtralModel(cfg, device=DEV, fp8=True)
        m.load_state({n: _big_weight(n, sh, seed) for n, sh in m.full_shapes().items()})
        if kind == "moe":
            m.quantize_experts()
        kv = KVCache(cfg.num_layers, total, m.hkv, m.D, device=DEV)
        for i in range(cfg.num_layers):
            k, v = _big_kv(cfg, i, total * PAGE, seed)
            for a in range(0, k.shape[0], 1 << 16):
                kk, vv = k[a:a + (1 << 16)], v[a:a + (1 << 16)]
                at = torch.arange(a, a + kk.shape[0], dtype=torch.int32, device=DEV)
                ops.rope_kv_write(torch.cat([kk.new_zeros((kk.shape[0], cfg.q_size)), kk, vv], 1), at, None, at, kv.k(i), kv.v(i),
                                  m.hq, m.hkv, m.D, apply_rope=False)
        ctx = torch.tensor([a + n for a, n in segs], dtype=torch.int32)
        longest = int(ctx.max())
        meta.decode_ws = DecodeWorkspace.create(max(nd, 1), m.hq, m.D, longest, m.device)
        if nc:
            meta.cu_q, meta.ctx_lens_p, meta.block_tables_p = _i32(cu[:nc + 1]), _i32(ctx[:nc]), _i32(_table(pages[:nc]))
            meta.max_q_len = max(n for _, n in segs[:nc])
            work = prefill_plan(cu[:nc + 1].numpy().astype("int32"), ctx[:nc].numpy(), m.hq // m.hkv, m.hkv)
            if work is not None:
                meta.prefill_work = torch.from_numpy(work).to(DEV)
                if work.shape[1] == 6:
                    meta.prefill_lean = (int(work[0, 1]), int(work[0, 2]), int(work[0, 3]))
        if nd:
            bt = _table(pages[nc:]).numpy()
            if nd >= LEAN_NT_MIN_B:       # as the runner marks its decode batches
                mark_shared_blocks(bt, ctx[nc:].numpy())
            meta.ctx_lens_d, meta.block_tables_d = _i32(ctx[nc:]), torch.from_numpy(bt).to(DEV)
    else:
        m = _layer_model(case)
        m.load_state({n: _layer_value(n, sh, seed, kind) for n, sh in m.full_shapes().items()})
        kv = m.make_cache(total, len(segs))
        _fill(kv, seed)
        meta.seg_cu, meta.seg_bt = _i32(cu), _i32(_table(pages))
        meta.seg_state = torch.arange(len(segs), dtype=torch.int32, device=DEV)
        meta.seg_max_len = max(n for _, n in segs)
    s["model"], s["kv"] = m, kv
    if nc == 0:
        _capture(s, (lambda: None) if big else (lambda: _fill(kv, seed)))
    return s


@torch.no_grad()
def run(s):
    if s["kind"] == "embed":
        return {"vectors": s["model"].encode(s["texts"])}
    if s["kind"] == "search":
        ids, scores, counts = ops.filtered_topk(*s["args"], s["kmax"])
        return {"ids": ids, "scores": scores, "counts": counts}
    if "graph" in s:
        s["graph"].replay()
        out = dict(s["out"])
    else:
        out = _forward(s)
    if s["kind"] not in ("chat", "moe"):
        out["cache"] = [t for _, ts in _entries(s["kv"].layers) for t in ts] + list(s["kv"].model.values())
    return out


# ----------------------------------------------------------------------------------------------
# what a pass cannot do without
# ----------------------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "embed":
        c = get_model_config("bge-base-en")
        r = random.Random("%d %d" % (case["texts"], case["longest"]))
        lens = [case["longest"]] + [r.randint(min(6, case["longest"]), case["longest"]) for _ in range(case["texts"] - 1)]
        per = c.num_layers * (4 * c.hidden_size ** 2 + 2 * c.hidden_size * c.intermediate_size)
        return {"bytes": 2 * per + 6 * sum(lens) * c.hidden_size + 4 * case["texts"] * c.hidden_size,
                "flops": 2 * per * sum(lens) + 4 * c.num_layers * c.hidden_size * sum(n * n for n in lens)}
    if kind == "search":
        hits = min(case["queries"] * case["rows"] / case["users"], case["rows"])
        return {"bytes": 12 * case["rows"] + hits * 768 * 2 + 8 * case["queries"] * case["limit"], "flops": 2 * 768 * hits}
    segs = _segments(case)
    T, S = sum(n for _, n in segs), len(segs)
    if kind in ("chat", "moe"):
        c = _big_config(kind)
        pages, total = _layout(case, segs)
        H, F = c.hidden_size, c.intermediate_size
        att = H * (c.q_size + 2 * c.kv_size) + c.q_size * H
        if kind == "chat":
            wb, wf = 2 * (att + 3 * H * F), 2 * (att + 3 * H * F)
        else:                             # fp8 experts: all of them from a few rows on
            e = min(c.num_experts, 2 * T)
            wb, wf = 2 * att + e * 3 * H * F, 2 * (att + 2 * 3 * H * F)
        kvb = 2 * 2 * c.kv_size
        cached = sum(a for a, _ in segs)
        common = case.get("shared", 0) // PAGE * PAGE
        users = sum(1 for a, _ in segs if a >= common)
        cached -= max(users - 1, 0) * common
        scores = sum(n * a + n * (n + 1) // 2 for a, n in segs)
        return {"bytes": c.num_layers * (wb + (cached + T) * kvb) + 2 * c.vocab_size * H + 2 * S * c.vocab_size + 2 * T * H,
                "flops": c.num_layers * (T * wf + 4 * c.q_size * scores) + 2 * S * c.vocab_size * H}
    m, cfg = _layer_model(case), _layer_config(case)
    eb = 4 if case["dtype"] == "fp32" else 2
    W = case["width"]
    nbytes, flops = eb * 32768 * W + eb * S * 32768 + eb * T * W, 2 * S * 32768 * W
    for l, spec in zip(m.layers, cfg["layers"]):
        p = l.prefix + "."
        mlp = spec["mlp"]
        for name, shape in m.full_shapes().items():
            if not name.startswith(p) or len(shape) < 2:
                continue
            size, share, use = math.prod(shape), 1.0, 1.0
            if mlp["kind"] == "moe" and name.startswith(p + "mlp.e"):
                E, top = mlp["router"]["experts"], mlp["router"]["top"]
                share, use = 1.0 - (1.0 - top / E) ** T, top / (E + mlp["router"].get("identity", 0))
            nbytes += eb * size * share
            flops += 2 * T * size * use
        specs = [spec["mixer"]] if "left" not in spec["mixer"] else [spec["mixer"]["left"], spec["mixer"]["right"]]
        for x in specs:
            if "mask" in x:               # attention: the keys in reach, and the new rows
                w = x["mask"]["size"]
                keys = sum(min(a, w) + n for a, n in segs)
                pairs = sum(sum(min(w, a + i + 1) for i in range(n)) for a, n in segs)
                row = x["kv_rank"] + x["rot_dim"] if "kv_rank" in x else x.get("kv_heads", 1) * (x["dim"] + x["vdim"])
                per = x["kv_rank"] * 2 + x["rot_dim"] if "kv_rank" in x else x["dim"] + x["vdim"]
                nbytes += eb * keys * row
                flops += 2 * pairs * x["heads"] * per
            elif "vdim" in x:             # a matrix state per head, updated by every token
                state = x["heads"] * x["vdim"] * x.get("state", x.get("dim"))
                nbytes += 4 * state * sum(2 if a else 1 for a, _ in segs)
                flops += 6 * state * T
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """From the error against float64 that bf16 and fp8 show here: two to four times it, sums in another order included;
    single values of a row whose chosen experts nearly tie may be off by more."""
    kind = case["kind"]
    if kind == "search":       # f32 dot products; rows whose scores nearly tie may change places
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.01}
    if kind == "embed":        # seen: 0.007
        return {"rel": 0.02}
    if kind in ("chat", "moe"):
        return {"rel": 0.03}
    if case["dtype"] == "fp32":     # seen: up to 6e-6
        return {"rel": 3e-5, "differ": 0.01}
    return {"rel": 0.03, "max": 0.99, "differ": 0.01}


# ----------------------------------------------------------------------------------------------
# float64
# ----------------------------------------------------------------------------------------------
def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def _softplus(x):
    return x.clamp(min=0) + torch.log1p(torch.exp(-x.abs()))


def _attend(q, k, v, start, scale, window=None, bias=None, sink=None, causal=True):
    """q [n, H, D] at positions start .., k [m, G, D], v [m, G, P] from position 0."""
    n, H, _ = q.shape
    G = k.shape[1]
    i = torch.arange(start, start + n, device=DEV)[:, None]
    j = torch.arange(k.shape[0], device=DEV)[None]
    hide = (j > i) if causal else torch.zeros_like(j > i)
    if window:
        hide = hide | (i - j >= window)
    out = torch.empty((n, H, v.shape[2]), dtype=F64, device=DEV)
    for g in range(G):
        hs = slice(g * (H // G), (g + 1) * (H // G))
        s = torch.matmul(q[:, hs].transpose(0, 1).contiguous(), k[:, g].T.contiguous()) * scale
        if bias is not None:
            s = s - bias[hs, None, None] * (i - j)
        s = s.masked_fill(hide, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[hs, None, None].expand(-1, n, 1)], -1)
        p = torch.softmax(s, -1)[..., :k.shape[0]]
        out[:, hs] = torch.matmul(p, v[:, g].contiguous()).transpose(0, 1)
    return out


def _rope_half(x, pos, freq):
    a = pos.to(F64)[:, None, None] * freq
    c, s = torch.cos(a), torch.sin(a)
    u, w = x.chunk(2, -1)
    return torch.cat([u * c - w * s, w * c + u * s], -1)


def _exact_big(case, seed):
    kind, cfg = case["kind"], _big_config(case["kind"])
    segs = _segments(case)
    ids, pos, slots, cu, pages, total = _batch(case, segs, cfg.vocab_size, seed)
    pos, slots = pos.to(DEV), slots.to(DEV)
    H, F, D, Hq, G, eps = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim, cfg.num_heads, cfg.num_kv_heads, cfg.norm_eps
    w = lambda n, *shape: _big_weight(n, shape, seed).to(F64)  # noqa: E731
    freq = cfg.rope_theta ** (-torch.arange(0, D, 2, dtype=F64, device=DEV) / D)
    x = _big_weight("embed", (cfg.vocab_size, H), seed)[ids].to(F64)
    for i in range(cfg.num_layers):
        p = f"layers.{i}."
        h = _rms(x, eps) * w(p + "in_norm", H)
        q, k, v = (h @ w(p + "qkv", cfg.q_size + 2 * cfg.kv_size, H).T).split([cfg.q_size, cfg.kv_size, cfg.kv_size], 1)
        q, k = (_rope_half(t.reshape(len(pos), -1, D), pos, freq) for t in (q, k))
        kc, vc = _big_kv(cfg, i, total * PAGE, seed)
        o = []
        for s, (a, n) in enumerate(segs):
            at = (torch.tensor(pages[s], device=DEV)[:, None] * PAGE + torch.arange(PAGE, device=DEV)).reshape(-1)[:a]
            b, e = int(cu[s]), int(cu[s + 1])
            keys = torch.cat([kc[at].to(F64).view(a, G, D), k[b:e]])
            vals = torch.cat([vc[at].to(F64).view(a, G, D), v[b:e].reshape(n, G, D)])
            o.append(_attend(q[b:e], keys, vals, a, D ** -0.5))
        x = x + torch.cat(o).reshape(len(pos), -1) @ w(p + "o", H, cfg.q_size).T
        h = _rms(x, eps) * w(p + "post_norm", H)
        if kind == "chat":
            g, u = (h @ w(p + "gate_up", 2 * F, H).T).chunk(2, 1)
            x = x + (_silu(g) * u) @ w(p + "down", H, F).T
        else:
            E, top = cfg.num_experts, cfg.top_k_experts
            pr, idx = torch.softmax(h @ w(p + "router", E, H).T, -1).topk(top, -1)
            pr = pr / pr.sum(-1, keepdim=True)
            w13, w2 = _big_weight(p + "w13", (E, 2 * F, H), seed), _big_weight(p + "w2", (E, H, F), seed)
            y = torch.zeros_like(x)
            for e in range(E):
                t, c = (idx == e).nonzero(as_tuple=True)
                g, u = (h[t] @ w13[e].to(F64).T).chunk(2, 1)
                y.index_add_(0, t, pr[t, c][:, None] * ((_silu(g) * u) @ w2[e].to(F64).T))
            x = x + y
    h = _rms(x, eps) * w("final_norm", H)
    return {"hidden": h, "logits": h[(cu[1:] - 1).to(DEV)] @ w("lm_head", cfg.vocab_size, H).T}


def _exact_embed(case, seed):
    c = get_model_config("bge-base-en")
    H, F, nh, D = c.hidden_size, c.intermediate_size, c.num_heads, c.head_dim
    w = lambda n, *shape: _bert_weight(n, shape, seed).to(F64)  # noqa: E731
    ln = lambda x, n: ((x - x.mean(-1, keepdim=True)) / torch.sqrt(x.var(-1, unbiased=False, keepdim=True) + c.norm_eps)  # noqa: E731
                       * w(n + "_g", H) + w(n + "_b", H))
    texts = _texts(case, seed)
    L = max(len(t) for t in texts)
    ids = torch.zeros((len(texts), L), dtype=torch.int64)
    for i, t in enumerate(texts):
        ids[i, :len(t)] = torch.tensor(t)
    ids = ids.to(DEV)
    lens = torch.tensor([len(t) for t in texts], device=DEV)
    hide = (torch.arange(L, device=DEV)[None] >= lens[:, None])[:, None, None]
    x = ln(w("word_emb", c.vocab_size, H)[ids] + w("pos_emb", c.max_position, H)[:L] + w("type_emb", c.type_vocab_size, H)[0], "emb_ln")
    for i in range(c.num_layers):
        p = f"layers.{i}."
        q, k, v = (t.reshape(len(texts), L, nh, D).transpose(1, 2).contiguous()
                   for t in (x @ w(p + "qkv", 3 * H, H).T + w(p + "qkv_b", 3 * H)).chunk(3, -1))
        s = torch.matmul(q, k.transpose(2, 3).contiguous()) * D ** -0.5
        o = torch.matmul(torch.softmax(s.masked_fill(hide, -math.inf), -1), v).transpose(1, 2).reshape(len(texts), L, H)
        x = ln(x + o @ w(p + "o", H, H).T + w(p + "o_b", H), p + "ln1")
        h = x @ w(p + "fc1", F, H).T + w(p + "fc1_b", F)
        x = ln(x + 0.5 * h * (1.0 + torch.erf(h / math.sqrt(2.0))) @ w(p + "fc2", H, F).T + w(p + "fc2_b", H), p + "ln2")
    return {"vectors": x[:, 0] / x[:, 0].norm(dim=-1, keepdim=True)}


def _exact_search(case, seed):
    corpus, users, dates, queries, who, since, _ = _search_inputs(case, seed)
    nq, kmax = case["queries"], case["limit"]
    ids = torch.full((nq, kmax), -1, dtype=torch.int32, device=DEV)
    scores, counts = torch.zeros((nq, kmax), dtype=F64, device=DEV), torch.zeros((nq,), dtype=torch.int32, device=DEV)
    for i in range(nq):
        rows = ((users == who[i]) & (dates >= since[i])).nonzero().flatten()
        s, at = torch.sort(corpus[rows].to(F64) @ queries[i].to(F64), descending=True, stable=True)
        k = min(kmax, len(rows))
        ids[i, :k], scores[i, :k], counts[i] = rows[at[:k]].to(torch.int32), s[:k], k
    return {"ids": ids, "scores": scores, "counts": counts}


class _Layered64:
    """One step of a layered decoder in float64 over the cache and states that the sequences bring along."""

    def __init__(self, case, seed):
        self.case, self.cfg, self.seed = case, _layer_config(case), seed
        self.segs = _segments(case)
        self.ids, pos, self.slots, self.cu, self.pages, total = _batch(case, self.segs, 32768, seed)
        self.pos, self.slots = pos.to(DEV), self.slots.to(DEV)
        m = _layer_model(case)
        self.shapes = m.full_shapes()
        cache = m.make_cache(total, len(self.segs))
        _fill(cache, seed)
        # name the entries: a mixer takes its own from the front, in the order of the cache
        self.cache = [t.to(F64) for _, ts in _entries(cache.layers) for t in ts]
        self.kinds = [k for k, ts in _entries(cache.layers) for _ in ts]
        self.last = cache.model.get("last_token")
        self.next, self.eps = 0, self.cfg["norm"]["eps"]

    def w(self, name):
        return _layer_value(name, self.shapes[name], self.seed, self.case["kind"]).to(F64)

    def lin(self, x, name):
        return x @ self.w(name).T

    def entry(self):
        self.next += 1
        return self.next - 1

    def rows(self):
        for s in range(len(self.segs)):
            yield s, self.segs[s][0], int(self.cu[s]), int(self.cu[s + 1])

    def conv(self, x, at, taps, bias=None):
        """Causal convolution behind the last inputs kept in entry ``at`` (zeros at a sequence's start)."""
        K = taps.shape[1]
        y = torch.empty_like(x)
        for s, a, b, e in self.rows():
            full = torch.cat([self.cache[at][s] if a else torch.zeros_like(self.cache[at][s]), x[b:e]])
            y[b:e] = sum(full[j:j + e - b] * taps[:, j] for j in range(K))
            self.cache[at][s] = full[-(K - 1):]
        return y if bias is None else y + bias

    def scan(self, state, step):
        """``step(S, t)`` for every token of a segment; the segments that are equally far run side by side."""
        n = max(int(self.cu[s + 1] - self.cu[s]) for s in range(len(self.segs)))
        fresh = torch.tensor([a == 0 for a, _ in self.segs], device=DEV)
        S = torch.where(fresh.view(-1, *[1] * (state.dim() - 1)), 0.0, state)
        first, lens = self.cu[:-1].to(DEV), (self.cu[1:] - self.cu[:-1])
        order = [(lens > t).nonzero().flatten().to(DEV) for t in range(n)] if n > 1 else [torch.arange(len(self.segs), device=DEV)]
        for t in range(n):
            live = order[t]
            S[live] = step(S[live], first[live] + t)
        state.copy_(S)

    def write(self, at, new):
        self.cache[at][self.slots] = new

    def keys(self, at, s, upto):
        i = (torch.tensor(self.pages[s], device=DEV)[:, None] * PAGE + torch.arange(PAGE, device=DEV)).reshape(-1)[:upto]
        return self.cache[at][i]

    # -- mixers ------------------------------------------------------------------------------------
    def mamba2(self, h, p, m):
        H, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
        inner, T = H * P, len(h)
        conv, at = self.entry(), self.entry()
        z, u, dt = self.lin(h, p + "in").split([inner, inner + 2 * G * N, H], 1)
        u = _silu(self.conv(u, conv, self.w(p + "conv"), self.w(p + "conv.b")))
        x, B, C = u[:, :inner].reshape(T, H, P), u[:, inner:inner + G * N].reshape(T, G, N), u[:, inner + G * N:].reshape(T, G, N)
        B, C = (t.repeat_interleave(H // G, 1) for t in (B, C))
        dt = _softplus(dt + self.w(p + "dt_bias"))
        keep = torch.exp(-torch.exp(self.w(p + "A_log")) * dt)
        y = torch.empty((T, H, P), dtype=F64, device=DEV)

        def step(S, t):                   # S [sequences, H, P, N]
            S = keep[t][..., None, None] * S + (dt[t][..., None] * x[t])[..., None] * B[t][:, :, None]
            y[t] = (S * C[t][:, :, None]).sum(-1)
            return S
        self.scan(self.cache[at], step)
        y = ((y + self.w(p + "D")[:, None] * x).reshape(T, inner) * _silu(z)).reshape(T, m["norm_groups"], -1)
        return self.lin(_rms(y, self.eps).reshape(T, inner) * self.w(p + "norm"), p + "o")

    def latent_attention(self, h, p, m):
        H, dn, dr, dv, R, T = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"], len(h)
        at = self.entry()
        a = self.pos.to(F64)[:, None] * m["rot"]["base"] ** (-torch.arange(0, dr, 2, dtype=F64, device=DEV) / dr)

        def rope(t):                      # adjacent pairs; t [T, heads, dr]
            c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
            return torch.stack([t[..., ::2] * c - t[..., 1::2] * s, t[..., 1::2] * c + t[..., ::2] * s], -1).flatten(-2)
        q = self.lin(_rms(self.lin(h, p + "dq"), self.eps) * self.w(p + "dq.norm"), p + "uq").reshape(T, H, dn + dr)
        c, kr = self.lin(h, p + "dkv").split([R, dr], 1)
        self.write(at, torch.cat([_rms(c, self.eps) * self.w(p + "dkv.norm"), rope(kr[:, None])[:, 0]], 1))
        uk, uv = self.w(p + "uk"), self.w(p + "uv")
        o = torch.empty((T, H, dv), dtype=F64, device=DEV)
        qr = rope(q[..., dn:])
        for s, start, b, e in self.rows():
            lo = max(0, start - m["mask"]["size"])
            rows = self.keys(at, s, start + e - b)[lo:]
            k = torch.cat([(rows[:, :R] @ uk.T).view(-1, H, dn), rows[:, None, R:].expand(-1, H, -1)], -1)
            o[b:e] = _attend(torch.cat([q[b:e, :, :dn], qr[b:e]], -1), k, (rows[:, :R] @ uv.T).view(-1, H, dv), start - lo,
                             m["scale"], m["mask"]["size"])
        return self.lin((o * torch.sigmoid(self.lin(h, p + "g"))[:, :, None]).reshape(T, -1), p + "o")

    def matrix_scan(self, q, k, v, g, at, beta=None):
        y = torch.empty_like(v)

        def step(S, t):                   # S [sequences, H, D, P]
            S = g[t][..., None] * S
            u = v[t]
            if beta is not None:
                u = beta[t][..., None] * (u - (S * k[t][..., None]).sum(-2))
            S = S + k[t][..., None] * u[..., None, :]
            y[t] = (S * q[t][..., None]).sum(-2)
            return S
        self.scan(self.cache[at], step)
        return y

    def channel_delta(self, h, p, m):
        H, G, D, P, T = m["heads"], m["kv_heads"], m["dim"], m["vdim"], len(h)
        at, conv = self.entry(), self.entry()      # entries in name order: S, conv
        u = torch.cat([self.lin(h, p + n) for n in "qkv"], 1)
        u = _silu(self.conv(u, conv, torch.cat([self.w(p + n + ".conv") for n in "qkv"])))
        q, k, v = u.split([G * D, G * D, H * P], 1)
        q, k = (t.reshape(T, G, D) / torch.sqrt((t.reshape(T, G, D) ** 2).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
        q, k = (t.repeat_interleave(H // G, 1) for t in (q * D ** -0.5, k))
        dt = _softplus(self.lin(self.lin(h, p + "a1"), p + "a2") + self.w(p + "dt_bias")).reshape(T, H, D)
        g = torch.exp(-torch.exp(self.w(p + "A_log"))[:, None] * dt)
        o = self.matrix_scan(q, k, v.reshape(T, H, P), g, at, torch.sigmoid(self.lin(h, p + "b")))
        gate = torch.sigmoid(self.lin(self.lin(h, p + "g1"), p + "g2"))
        return self.lin((_rms(o, self.eps) * self.w(p + "norm")).reshape(T, -1) * gate, p + "o")

    def gla(self, h, p, m):
        H, D, P, T = m["heads"], m["dim"], m["vdim"], len(h)
        q, k, v = self.lin(h, p + "q").view(T, H, D) * D ** -0.5, self.lin(h, p + "k").view(T, H, D), self.lin(h, p + "v").view(T, H, P)
        z = self.lin(self.lin(h, p + "a1"), p + "a2") + self.w(p + "a2.b")
        o = self.matrix_scan(q, k, v, (torch.sigmoid(z) ** (1.0 / m["tau"])).view(T, H, D), self.entry())
        return self.lin((_rms(o, self.eps) * self.w(p + "norm")).reshape(T, -1) * _silu(self.lin(h, p + "g")), p + "o")

    def parallel(self, h, p, m):
        left, right, T = m["left"], m["right"], len(h)
        H, G, D, P, l, r = left["heads"], left["kv_heads"], left["dim"], left["vdim"], p + "left.", p + "right."
        at, S, conv = self.entry(), self.entry(), self.entry()
        q = (_rms(self.lin(h, l + "q"), self.eps) * self.w(l + "q.norm")).view(T, H, D)
        k = _rms(self.lin(h, l + "k"), self.eps) * self.w(l + "k.norm")
        self.write(at, torch.cat([k, self.lin(h, l + "v")], 1))
        o = torch.empty((T, H, P), dtype=F64, device=DEV)
        for s, start, b, e in self.rows():
            lo = max(0, start - left["mask"]["size"])
            rows = self.keys(at, s, start + e - b)[lo:]
            o[b:e] = _attend(q[b:e], rows[:, :G * D].reshape(-1, G, D), rows[:, G * D:].reshape(-1, G, P), start - lo,
                             left["scale"], left["mask"]["size"])
        o = self.lin((o * torch.sigmoid(self.lin(h, l + "g"))[:, :, None]).reshape(T, -1), l + "o")
        R, B = right["width"], right["blocks"]
        u = self.conv(self.lin(h, r + "x") + self.w(r + "x.b"), conv, self.w(r + "conv"), self.w(r + "conv.b"))
        ub = u.view(T, B, R // B).transpose(0, 1).contiguous()
        gate = lambda n: torch.sigmoid(torch.matmul(ub, self.w(r + n).transpose(1, 2).contiguous()).transpose(0, 1)  # noqa: E731
                                       + self.w(r + n + ".b")).reshape(T, R)
        a = torch.exp(-8.0 * gate("ra") * _softplus(self.w(r + "lam")))
        put = torch.sqrt(1.0 - a * a) * gate("ri") * u
        y = torch.empty_like(u)

        def step(st, t):
            y[t] = a[t] * st + put[t]
            return y[t]
        self.scan(self.cache[S], step)
        y = self.lin(y * _gelu(self.lin(h, r + "y") + self.w(r + "y.b")), r + "o")
        return 0.5 * (_rms(o, self.eps) * self.w(l + "out") + _rms(y, self.eps) * self.w(r + "out"))

    def conv_attention(self, h, p, m, shared):
        H, G, D, P, T = m["heads"], m["kv_heads"], m["dim"], m["vdim"], len(h)
        own = m.get("kv_from") is None
        at = self.entry() if own else shared[m["kv_from"]]
        conv, names = self.entry(), "qkv" if own else "q"
        u = self.conv(torch.cat([self.lin(h, p + n) for n in names], 1), conv, torch.cat([self.w(p + n + ".conv") for n in names]))
        q = _rms(u[:, :H * D].reshape(T, H, D), self.eps) * self.w(p + "q.norm")
        q = q * (1.0 + m["q_temp"]["coef"] * torch.log((self.pos + 1) // m["q_temp"]["every"] + 1.0))[:, None, None]
        if own:
            k = _rms(u[:, H * D:(H + G) * D].reshape(T, G, D), self.eps) * self.w(p + "k.norm")
            self.write(at, torch.cat([k.reshape(T, -1), u[:, (H + G) * D:]], 1))
        slope = 2.0 ** (-8.0 * torch.arange(1, H + 1, dtype=F64, device=DEV) / H)
        o = torch.empty((T, H, P), dtype=F64, device=DEV)
        for s, start, b, e in self.rows():
            lo = max(0, start - m["mask"]["size"])
            rows = self.keys(at, s, start + e - b)[lo:]
            o[b:e] = _attend(q[b:e], rows[:, :G * D].reshape(-1, G, D), rows[:, G * D:].reshape(-1, G, P), start - lo,
                             m["scale"], m["mask"]["size"], slope, self.w(p + "sink"))
        return self.lin(o.reshape(T, -1) * torch.sigmoid(self.lin(h, p + "g")), p + "o"), at

    # -- feed-forwards -----------------------------------------------------------------------------
    def unit(self, h, p, limit):
        g, u = self.lin(h, p + "gate"), self.lin(h, p + "up")
        if limit is None:                 # plain SiLU expert
            return self.lin(_silu(g) * u, p + "down")
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        return self.lin(g * torch.sigmoid(1.702 * g) * (u + 1.0), p + "down")

    def feed(self, h, p, mlp):
        kind = self.case["kind"]
        if mlp["kind"] == "dense":
            if kind == "gezavik":
                return self.lin(torch.relu(self.lin(h, p + "up")) ** 2, p + "down")
            if kind == "sigudra":
                return self.lin(_gelu(self.lin(h, p + "gate")) * self.lin(h, p + "up"), p + "down")
            return self.unit(h, p, mlp["limit"])
        r = mlp["router"]
        z = self.lin(h, p + "router")
        if kind == "gezavik":
            s = torch.softmax(z, -1)
        else:
            s = torch.sigmoid(z)
        idx = (s if kind == "sigudra" else s + self.w(p + "correction")).topk(r["top"], -1).indices
        wt = s.gather(1, idx)
        if kind == "fanotar":
            wt = wt / (wt.sum(-1, keepdim=True) + 1e-20) * r["scale"]
        y = torch.zeros_like(h)
        for e in range(r["experts"] + r.get("identity", 0)):
            t, c = (idx == e).nonzero(as_tuple=True)
            a = wt[t, c][:, None]
            if e >= r["experts"]:         # identity expert
                o = a * h[t]
            elif kind == "sigudra":       # the score multiplies the expert's input
                o = self.unit(a * h[t], f"{p}e{e}.", None)
            else:
                o = a * self.unit(h[t], f"{p}e{e}.", mlp["expert"]["limit"])
            y.index_add_(0, t, o)
        return y + self.unit(h, p + "shared.", mlp["shared"]["limit"]) if mlp.get("shared") else y

    # -- whole models ------------------------------------------------------------------------------
    def ln(self, x, name):
        return (x - x.mean(-1, keepdim=True)) / torch.sqrt(x.var(-1, unbiased=False, keepdim=True) + self.eps) * self.w(name)

    def dyn(self, x, name):
        return torch.tanh(self.w(name + ".alpha") * x) * self.w(name) + self.w(name + ".b")

    def step(self):
        kind, ids, layers = self.case["kind"], self.ids, self.cfg["layers"]
        x = self.w("embed")[ids]
        if kind == "gezavik":
            for i, L in enumerate(layers):
                h = _rms(x, self.eps) * self.w(f"l{i}.norm1")
                x = x + self.cfg["residual_mult"] * (getattr(self, L["type"])(h, f"l{i}.mix.", L["mixer"]) + self.feed(h, f"l{i}.mlp.", L["mlp"]))
            h = _rms(x, self.eps) * self.w("final.norm")
        elif kind == "sigudra":
            b = self.cfg["embedding"]["bigram"]
            prev = torch.cat([ids.new_zeros(1), ids[:-1]])
            prev[self.cu[:-1].to(DEV)] = self.last.to(ids.dtype)
            pair = (prev * b["mul_prev"] + ids * b["mul_cur"]) % b["buckets"]
            x = x + self.w("bigram")[torch.where(self.pos == 0, b["buckets"], pair)]
            for i, L in enumerate(layers):
                x = x + self.ln(getattr(self, L["type"])(x, f"l{i}.mix.", L["mixer"]), f"l{i}.norm1")
                x = x + self.ln(self.feed(x, f"l{i}.mlp.", L["mlp"]), f"l{i}.norm2")
            h = self.ln(x, "final.norm")
        else:
            x, shared = self.dyn(x * self.cfg["embedding"]["scale"], "embed.norm"), {}
            for i, L in enumerate(layers):
                y, shared[i] = self.conv_attention(self.dyn(x, f"l{i}.norm1"), f"l{i}.mix.", L["mixer"], shared)
                x = x + self.dyn(y, f"l{i}.norm1b")
                x = x + self.dyn(self.feed(self.dyn(x, f"l{i}.norm2"), f"l{i}.mlp.", L["mlp"]), f"l{i}.norm2b")
            h = self.dyn(x, "final.norm")
        end = (self.cu[1:] - 1).to(DEV)
        return {"hidden": h, "logits": self.lin(h[end], "head"), "cache": self.cache + ([ids[end]] if self.last is not None else [])}


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "embed":
        return _exact_embed(case, seed)
    if kind == "search":
        return _exact_search(case, seed)
    return _exact_big(case, seed) if kind in ("chat", "moe") else _Layered64(case, seed).step()
