"""Workloads of the sparse decode library, each one call (or one short serving
burst) through the package's public entry points.

A case is a dict of plain values:

  kind      what is called (KINDS below)
  batch     requests in the step
  lo, hi    context lengths in tokens; the lengths are spread over [lo, hi]
  heads, dim, page, k   the pool's shape and the pages kept per request
  steps     (serve) decode steps per burst

Keys and values come from the library's own device generator
(DevicePagePool.prefill_synthetic, PageTable.admit_synthetic: an integer hash
onto k/1000 in [-1, 1]), so that pools of tens of GB are filled in
milliseconds; queries and decode tokens are N(0, 1).  A request's pages lie
scattered over the pool, as a pool that has served for a while hands them out.
"""
from __future__ import annotations

import importlib
import math
import random

import numpy as np
import torch

dsd = importlib.import_module("15-618_dynamic_sparse_decode_amd")

KINDS = {
    "step": "SparseContext.run_batch_device: queries and page lists in HBM",
    "host": "SparseContext.run_batch, outputs and ids back to host memory",
    "scored": "SparseContext.run_batch in debug mode: exact scores of every page too",
    "dense": "dense_run_batch_device: attention over every page",
    "serve": "PageTable admission, table steps with appends, release",
}


def _case(name, kind, batch, lo, hi, heads=32, dim=128, page=16, k=8, steps=0):
    return {"name": name, "kind": kind, "batch": batch, "lo": lo, "hi": hi, "heads": heads,
            "dim": dim, "page": page, "k": k, "steps": steps}


def listed():
    return [
        # One user's request at a short context: the smallest call, all latency.
        _case("one_request_1k", "step", 1, 1024, 1024),
        # The benchmark's step: a ragged batch of short contexts.
        _case("batch16_ragged", "step", 16, 512, 2048),
        # Long contexts at a full batch: the largest sparse step.
        _case("batch32_32k", "step", 32, 32768, 32768, k=64),
        # Large pages and a large share of them kept.
        _case("batch64_page64", "step", 64, 4096, 16384, page=64, k=32),
        # A few very long documents: thousands of pages per request.
        _case("batch4_128k", "step", 4, 65536, 131072, k=64),
        # Grouped-query models keep few KV heads: E = 8 x 128.
        _case("batch32_8heads", "step", 32, 1024, 8192, heads=8, k=16),
        # A busy server's batch: more requests than one launch holds heads for.
        _case("batch128_ragged", "step", 128, 512, 4096),
        # The dense baseline the sparse step is compared with, short contexts.
        _case("dense16_ragged", "dense", 16, 512, 2048),
        # The dense baseline for one long document.
        _case("dense1_32k", "dense", 1, 32768, 32768),
        # The benchmark's step for callers whose queries live on the host.
        _case("host16_ragged", "host", 16, 512, 2048),
        # The same with every page's score returned (accuracy runs).
        _case("scored16_ragged", "scored", 16, 512, 2048),
        # Serving: admit a full batch, decode a while with appends, release.
        _case("serve32", "serve", 32, 1024, 4096, steps=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["short", "long", "pages", "very_long", "heads", "heads", "busy",
                       "dense", "dense_long", "host", "scored", "serve"])

    def spread(least, most):
        a, b = _log_int(rng, least, most), _log_int(rng, least, most)
        return min(a, b), max(a, b)

    if what == "short":
        lo, hi = spread(200, 4000)
        return _case("", "step", _log_int(rng, 1, 64), lo, hi, k=rng.choice([4, 8, 8, 16]))
    if what == "long":
        lo, hi = spread(5000, 32768)
        return _case("", "step", _log_int(rng, 1, 32), lo, hi, k=rng.choice([8, 32, 64]))
    if what == "pages":
        lo, hi = spread(2000, 16384)
        return _case("", "step", _log_int(rng, 4, 64), lo, hi, page=rng.choice([32, 64]),
                     k=rng.choice([8, 16, 32]))
    if what == "very_long":
        lo, hi = spread(40000, 131072)
        return _case("", "step", _log_int(rng, 1, 8), lo, hi, k=rng.choice([16, 64, 128]))
    if what == "heads":
        lo, hi = spread(500, 12000)
        heads, dim = rng.choice([(8, 128), (16, 128), (4, 128), (64, 128), (40, 128), (32, 64),
                                 (16, 64), (8, 64), (12, 64), (32, 80), (8, 96)])
        return _case("", "step", _log_int(rng, 1, 32), lo, hi, heads=heads, dim=dim,
                     page=rng.choice([16, 16, 32]), k=rng.choice([8, 16, 32]))
    if what == "busy":
        lo, hi = spread(200, 4000)
        return _case("", "step", _log_int(rng, 65, 256), lo, hi, k=rng.choice([4, 8, 16]))
    if what == "dense":
        lo, hi = spread(200, 4000)
        heads, dim = rng.choice([(32, 128), (32, 128), (8, 128), (32, 64)])
        return _case("", "dense", _log_int(rng, 4, 20), lo, hi, heads=heads, dim=dim)
    if what == "dense_long":
        lo, hi = spread(8000, 40000)
        return _case("", "dense", rng.randint(1, 2), lo, hi, heads=rng.choice([8, 32]))
    if what in ("host", "scored"):
        lo, hi = spread(200, 4000)
        return _case("", what, _log_int(rng, 1, 32), lo, hi, k=rng.choice([8, 16]))
    lo, hi = spread(500, 4096)
    return _case("", "serve", _log_int(rng, 4, 32), lo, hi, steps=rng.randint(4, 16))


# ---- the shape of a case -------------------------------------------------------

def _lengths(case):
    """The context lengths: the case's own, whatever the seed of its values."""
    rng = random.Random("%(batch)d %(lo)d %(hi)d" % case)
    got = [rng.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]
    got[0] = case["hi"]
    return got


def _pages(case, tokens):
    return -(-tokens // case["page"])


def _request_id(seed, r):
    return (seed * 7919 + r * 104729 + 1) % (1 << 30)


def _page_lists(case, seed):
    """(CSR offsets, page ids): every page of the pool once, in a random order."""
    counts = [_pages(case, c) for c in _lengths(case)]
    offsets = np.zeros(len(counts) + 1, np.int32)
    offsets[1:] = np.cumsum(counts)
    return offsets, np.random.RandomState(seed % (1 << 31)).permutation(
        int(offsets[-1])).astype(np.int32)


def _normal(seed, salt, *shape):
    """N(0, 1) float32 on the GPU, from the seed alone."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed * 16 + salt)
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32)


_STREAM = None


def _stream():
    """The one stream this program runs its steps on."""
    global _STREAM
    if _STREAM is None:
        _STREAM = torch.cuda.Stream()
    return _STREAM.cuda_stream


# ---- prepare and run -------------------------------------------------------------

def _filled_pool(case, seed, offsets, ids):
    pool = dsd.DevicePagePool(case["heads"], case["dim"], case["page"], len(ids))
    for r, tokens in enumerate(_lengths(case)):
        mine = ids[offsets[r]:offsets[r + 1]]
        counts = np.full(len(mine), case["page"], np.int32)
        counts[-1] = tokens - (len(mine) - 1) * case["page"]
        pool.prefill_synthetic(mine, counts, _request_id(seed, r))
    return pool


def prepare(case, seed):
    E, B, k = case["heads"] * case["dim"], case["batch"], case["k"]
    if case["kind"] == "serve":
        lengths, steps = _lengths(case), case["steps"]
        most = [_pages(case, c + steps) for c in lengths]
        pool = dsd.DevicePagePool(case["heads"], case["dim"], case["page"], sum(most))
        table = dsd.PageTable(pool, B, max(most))
        ctx = dsd.SparseContext(pool, k, B, sum(most), B * k)
        rows = [_normal(seed, salt, steps, B, E).cpu().numpy() for salt in (1, 2, 3)]
        return {"case": case, "ctx": ctx, "table": table, "lengths": lengths,
                "requests": [_request_id(seed, r) for r in range(B)],
                "slots": np.arange(B, dtype=np.int32), "upload": np.ones(B, np.uint8),
                "queries": rows[0], "keys": rows[1], "values": rows[2]}
    offsets, ids = _page_lists(case, seed)
    pool = _filled_pool(case, seed, offsets, ids)
    queries = _normal(seed, 1, B, E)
    state = {"case": case, "pool": pool, "total": len(ids),
             "most": int(np.diff(offsets).max())}
    if case["kind"] != "dense":
        state["ctx"] = dsd.SparseContext(pool, k, B, len(ids), B * k)
    if case["kind"] in ("host", "scored"):
        state.update(queries=queries.cpu().numpy(), offsets=offsets, ids=ids)
        return state
    state.update(queries=queries, offsets=torch.from_numpy(offsets).cuda(),
                 ids=torch.from_numpy(ids).cuda(), outputs=torch.zeros_like(queries),
                 selected=torch.full((B, k), -1, dtype=torch.int32, device="cuda"),
                 counts=torch.zeros(B, dtype=torch.int32, device="cuda"))
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        state["ctx"].run_batch_device(
            case["batch"], state["total"], state["most"], state["queries"].data_ptr(),
            state["offsets"].data_ptr(), state["ids"].data_ptr(), state["outputs"].data_ptr(), 0,
            state["selected"].data_ptr(), state["counts"].data_ptr(), _stream())
        return {"outputs": state["outputs"], "selected": state["selected"],
                "counts": state["counts"]}
    if kind == "dense":
        dsd.dense_run_batch_device(
            state["pool"], case["batch"], state["queries"].data_ptr(),
            state["offsets"].data_ptr(), state["ids"].data_ptr(), state["outputs"].data_ptr(),
            _stream())
        return {"outputs": state["outputs"]}
    if kind in ("host", "scored"):
        got = state["ctx"].run_batch(
            state["queries"], state["offsets"], state["ids"],
            output_mode=dsd.OUTPUT_DEBUG if kind == "scored" else dsd.OUTPUT_OUTPUTS,
            timing_mode=dsd.TIMING_NONE, want_ids=True)
        out = {"outputs": got["outputs"], "selected": np.concatenate(got["selected"])}
        if kind == "scored":
            out["scores"] = got["scores"]
        return out
    table, ctx, slots = state["table"], state["ctx"], state["slots"]
    for slot, (tokens, request) in enumerate(zip(state["lengths"], state["requests"])):
        table.admit_synthetic(slot, tokens, request)
    outputs = []
    for t in range(case["steps"]):
        outputs.append(ctx.run_table(table, slots, queries=state["queries"][t])["outputs"])
        if t + 1 < case["steps"]:
            table.append(slots, state["upload"], keys=state["keys"][t],
                         values=state["values"][t])
    table.release(slots)
    return {"outputs": outputs}


# ---- what a pass cannot do without -------------------------------------------------

def _step_work(case, lengths):
    E = case["heads"] * case["dim"]
    kept = sum(min(c, case["k"] * case["page"]) for c in lengths)
    pages = sum(_pages(case, c) for c in lengths)
    # summaries, ids; queries, outputs, selected ids; selected K and V
    moved = pages * (4 * E + 4) + len(lengths) * (8 * E + 4 * case["k"]) + kept * 8 * E
    return moved, 2 * pages * E + 4 * kept * E


def work(case):
    E, lengths = case["heads"] * case["dim"], _lengths(case)
    if case["kind"] == "dense":
        tokens = sum(lengths)
        pages = sum(_pages(case, c) for c in lengths)
        return {"bytes": tokens * 8 * E + pages * 4 + case["batch"] * 8 * E,
                "flops": 4 * tokens * E}
    if case["kind"] == "serve":
        # the prompts' K and V and their summaries written once; each step's
        # reads; each appended token's rows read and written
        moved = sum(c * 8 * E + _pages(case, c) * 4 * E for c in lengths)
        flops = 0
        for t in range(case["steps"]):
            b, f = _step_work(case, [c + t for c in lengths])
            moved, flops = moved + b, flops + f
        moved += (case["steps"] - 1) * case["batch"] * 4 * 4 * E
        return {"bytes": moved, "flops": flops}
    moved, flops = _step_work(case, lengths)
    if case["kind"] == "scored":
        moved += 4 * sum(_pages(case, c) for c in lengths)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    # Ids are whole numbers and the same.  Outputs are 32-bit softmax sums and
    # scores 32-bit chains: measured 1e-7 to 6e-7 from 64 bits.
    return {"rel": 2e-6, "max": 2e-5}


# ---- the same in plain torch and 64 bits -------------------------------------------

_M32 = 0xFFFFFFFF
_GRID = torch.from_numpy(((np.arange(2001) - 1000).astype(np.float32) / np.float32(1000)))


def _mix(x, v, salt):
    return x ^ ((v + salt + (x << 6) + (x >> 2)) & _M32)


def _prompt(case, request, pages, which):
    """Rows [page][token][E] of prompt pages `pages` (a tensor): keys (which
    = 1) or values (2) of the device generator."""
    E = case["heads"] * case["dim"]
    x = torch.tensor(0x9E3779B9, dtype=torch.int64, device="cuda")
    x = _mix(x, request, 0x85EBCA6B)
    x = _mix(x, pages.view(-1, 1, 1), 0xC2B2AE35)
    x = _mix(x, torch.arange(case["page"], device="cuda").view(1, -1, 1), 0x27D4EB2F)
    x = _mix(x, torch.arange(E, device="cuda").view(1, 1, -1), 0x165667B1)
    x = _mix(x, which, 0xD3A2646C)
    x = x ^ (x >> 16)
    x = (x * 0x7FEB352D) & _M32
    x = x ^ (x >> 15)
    x = (x * 0x846CA68B) & _M32
    x = x ^ (x >> 16)
    return _GRID.cuda()[x % 2001]


def _summaries(case, request, tokens):
    """fp32 page means: tokens added in order, then times fl(1 / count)."""
    n = _pages(case, tokens)
    E = case["heads"] * case["dim"]
    step = max(1, (1 << 24) // (case["page"] * E))
    parts = []
    for p0 in range(0, n, step):
        pages = torch.arange(p0, min(n, p0 + step), device="cuda")
        keys = _prompt(case, request, pages, 1)
        counts = torch.full((len(pages),), case["page"], device="cuda")
        if p0 + step >= n:
            counts[-1] = tokens - (n - 1) * case["page"]
        acc = torch.zeros(len(pages), E, device="cuda")
        for t in range(case["page"]):
            acc = torch.where((t < counts).view(-1, 1), acc + keys[:, t], acc)
        inv = torch.from_numpy(np.float32(1) / counts.cpu().numpy().astype(np.float32)).cuda()
        parts.append(acc * inv.view(-1, 1))
    return torch.cat(parts)


def _scale(case):
    return np.float32(1) / np.sqrt(np.float32(case["dim"]))


def _select(case, queries, summaries, ids):
    """Per request, the positions the rule keeps in its page list: fp32
    products added one after the other, the best scores first, the smaller
    page id first among equals.  summaries, ids: one entry per request."""
    products = torch.cat([q.view(1, -1) * s for q, s in zip(queries, summaries)]).t().contiguous()
    acc = torch.zeros(products.shape[1], device="cuda")
    for row in products:
        acc += row
    scores = np.split(acc.cpu().numpy() * _scale(case), np.cumsum([len(i) for i in ids])[:-1])
    return [np.lexsort((i, -s))[:case["k"]] for i, s in zip(ids, scores)]


def _attend(case, query, keys, values):
    """softmax(q K^T * scale) V per head in 64 bits; keys, values [tokens][E]."""
    H, D = case["heads"], case["dim"]
    out = torch.empty(H, D, dtype=torch.float64, device="cuda")
    for h0 in range(0, H, 8):
        q = query.view(H, D)[h0:h0 + 8].double()
        k = keys.view(-1, H, D)[:, h0:h0 + 8].double()
        v = values.view(-1, H, D)[:, h0:h0 + 8].double()
        p = torch.softmax((k * q).sum(-1) * float(_scale(case)), dim=0)
        out[h0:h0 + 8] = (p.unsqueeze(-1) * v).sum(0)
    return out.view(-1)


def _rows(case, request, pages, tokens, which):
    """K or V rows of prompt pages `pages` (a list, in order), valid tokens only."""
    at = torch.as_tensor(np.asarray(pages, np.int64), device="cuda")
    step = max(1, (1 << 24) // (case["page"] * case["heads"] * case["dim"]))
    rows = torch.cat([_prompt(case, request, at[i:i + step], which)
                      for i in range(0, len(at), step)])
    t = at.view(-1, 1) * case["page"] + torch.arange(case["page"], device="cuda")
    return rows[t < tokens]


def exact(case, seed):
    lengths, B = _lengths(case), case["batch"]
    E = case["heads"] * case["dim"]
    if case["kind"] == "serve":
        return _exact_serve(case, seed)
    offsets, ids = _page_lists(case, seed)
    queries = _normal(seed, 1, B, E)
    requests = [_request_id(seed, r) for r in range(B)]
    if case["kind"] == "dense":
        kept = [np.arange(_pages(case, c)) for c in lengths]
    else:
        summaries = [_summaries(case, q, c) for q, c in zip(requests, lengths)]
        kept = _select(case, queries, summaries, np.split(ids, offsets[1:-1]))
    outputs = torch.empty(B, E, dtype=torch.float64, device="cuda")
    for r, (request, tokens) in enumerate(zip(requests, lengths)):
        keys, values = (_rows(case, request, kept[r], tokens, w) for w in (1, 2))
        outputs[r] = _attend(case, queries[r], keys, values)
    out = {"outputs": outputs}
    if case["kind"] != "dense":
        out["selected"] = None
    if case["kind"] == "step":
        out["counts"] = None
    if case["kind"] == "scored":
        out["scores"] = torch.cat([s.double() @ q.double() for s, q in zip(summaries, queries)])
        out["scores"] *= float(_scale(case))
    return out


def _exact_serve(case, seed):
    B, steps = case["batch"], case["steps"]
    E, ps = case["heads"] * case["dim"], case["page"]
    prompts = _lengths(case)
    queries, new_keys, new_values = (_normal(seed, salt, steps, B, E) for salt in (1, 2, 3))
    requests = [_request_id(seed, r) for r in range(B)]
    summaries = []
    for request, tokens in zip(requests, prompts):
        s = torch.zeros(_pages(case, tokens + steps), E, device="cuda")
        s[:_pages(case, tokens)] = _summaries(case, request, tokens)
        summaries.append(s)
    outputs = torch.empty(steps, B, E, dtype=torch.float64, device="cuda")
    for t in range(steps):
        live = [_pages(case, c + t) for c in prompts]
        kept = _select(case, queries[t], [s[:n] for s, n in zip(summaries, live)],
                       [np.arange(n) for n in live])
        for r, (request, prompt) in enumerate(zip(requests, prompts)):
            sides = []
            for which, new in ((1, new_keys), (2, new_values)):
                mine = [p for p in kept[r] if p * ps < prompt]
                rows = [_rows(case, request, mine, prompt, which)] if mine else []
                rows += [new[i, r].view(1, E) for i in range(t) if (prompt + i) // ps in kept[r]]
                sides.append(torch.cat(rows))
            outputs[t, r] = _attend(case, queries[t, r], *sides)
            # the running mean, each operation rounded to 32 bits
            page, old = (prompt + t) // ps, (prompt + t) % ps
            total = summaries[r][page] * float(old) + new_keys[t, r]
            summaries[r][page] = (total.double() / (old + 1)).float()
    return {"outputs": list(outputs)}
