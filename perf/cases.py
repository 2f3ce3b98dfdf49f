"""The work this framework is measured on: calls of its public entry points at the sizes its configurations, tests and
benchmark use, from a training batch's rows to counts over 1e9 corpus tokens.

  listed()               the named cases
  draw(rng)              one more case of the same ranges
  prepare(case, seed)    the inputs and the handle a program holds before the call, on the GPU, from the seed alone
  run(state)             one pass through the entry points, and its outputs
  work(case)             the bytes a pass cannot do without (each input read once, each output written once)
  tolerance(case)        how far another correct implementation's outputs may be off
  exact(case, seed)      run's outputs by plain torch in 64-bit integers (None where that takes too long)

Streams are documents of geometric length (mean 1024) ending with the end-of-text token, body tokens Zipf(1.1) over
permuted ids, and a share of the documents holding a copied span: of the corpus itself, or, for the query streams, of
the corpus they are held out from."""

import math
import os
import sys
from types import SimpleNamespace

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "n-gram-hinted-lm_amd"))

BOS = 50256
DOC = 1025  # mean document: 1024 body tokens and the end-of-text token
M = 1 << 20

RECORD_LEVELS = "2,3,4,5,6,10,20"  # the count record's levels; its rows come from 6, 10 and 20
VAL_LEVELS = "2,3,4,5,6,8,10,12,16,20"  # the validation statistics' levels


def listed():
    return [
        # a training step's rows: one micro-batch of 64 x 1024 positions cut out of a build's rows
        {"name": "batch_rows_64k", "kind": "batch_rows", "corpus": 4 * M, "queries": 4 * 65536, "n": 65536},
        # the count mixture's features of eight 65536-position fit blocks at seven levels
        {"name": "features_512k", "kind": "features", "n": 8 * 65536, "levels": 7},
        # a small query-filtered count: bigrams and trigrams of four 1M-token shards, top-1
        {"name": "counts_4m", "kind": "counts", "corpus": 4 * M, "shards": 4, "queries": 256 << 10, "levels": "2,3",
         "topk": 1, "copies": 0.10, "span": 256},
        # the record's build on part of its corpus: its seven levels, its rows, no top lists
        {"name": "counts_record_64m", "kind": "counts", "corpus": 64_000_000, "shards": 8, "queries": M + 4 * 65536,
         "levels": RECORD_LEVELS, "topk": 0, "copies": 0.05, "span": 1024},
        # one GPU's share of the record at full size: 1e9 tokens, n = 2..8, 16M positions, top-4
        {"name": "counts_1b", "kind": "counts", "corpus": 1_000_000_000, "shards": 10, "queries": 16_000_000,
         "levels": "2,3,4,5,6,7,8", "topk": 4, "copies": 0.05, "span": 1024},
        # the validation statistics (ten levels, counts of the target only among the top 1024, three variants' rows) of
        # the whole validation stream against one training shard
        {"name": "val_stats_100m", "kind": "val_stats", "corpus": 100_000_000, "shards": 1, "queries": 10_485_760,
         "copies": 0.05, "span": 1024},
        # corpus-wide tables of a small corpus, built and asked for the counts of a validation slice
        {"name": "table_4m", "kind": "table", "corpus": 4 * M, "shards": 4, "queries": 256 << 10, "levels": "1,2,3",
         "topk": 0, "copies": 0.10, "span": 256},
        # corpus-wide tables of one shard, built and asked for the top-4 continuations of 8M positions
        {"name": "table_100m", "kind": "table", "corpus": 100_000_000, "shards": 1, "queries": 8_000_000,
         "levels": "2,3,4", "topk": 4, "copies": 0.10, "span": 256},
        # the longest suffix match of a small validation stream, every position
        {"name": "longest_4m", "kind": "longest", "corpus": 4 * M, "shards": 4, "queries": 256 << 10, "every": 1,
         "cap": 32, "copies": 0.10, "span": 256},
        # the longest suffix match at scale: every fourth position of a 64M-token held-out stream against 1e9 tokens
        {"name": "longest_1b", "kind": "longest", "corpus": 1_000_000_000, "shards": 10, "queries": 64_000_000,
         "every": 4, "cap": 64, "copies": 0.15, "span": 2048},
        # a run's online rows from an empty state: 16 steps of 2^19 fresh tokens, hint and count rows of every step
        {"name": "online_16x512k", "kind": "online", "steps": 16, "step": 1 << 19, "levels": "2,3,4,5,6",
         "copies": 0.10, "span": 256},
        # the online counts of every position of two small training shards (a document sees the documents before it)
        {"name": "train_counts_256k", "kind": "train_counts", "corpus": 256 << 10, "shards": 2, "levels": "2,3,4",
         "copies": 0.10, "span": 256},
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi], odd half the time."""
    v = int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    return min(hi, v | 1) if rng.random() < 0.5 else v


def draw(rng):
    kind = rng.choice(["counts", "counts", "counts", "val_stats", "table", "table", "longest", "longest", "online",
                       "train_counts", "batch_rows", "features"])
    copies, span = round(rng.uniform(0.02, 0.15), 3), rng.choice([256, 1024, 2048])
    if kind == "features":
        return {"kind": kind, "n": _log(rng, 4096, 2 * M), "levels": rng.choice([2, 3, 7, 10])}
    if kind == "batch_rows":
        n = _log(rng, 1024, 256 << 10)
        return {"kind": kind, "corpus": _log(rng, M, 16 * M), "queries": n + _log(rng, 1, 65536), "n": n}
    if kind == "train_counts":
        return {"kind": kind, "corpus": _log(rng, 32 << 10, 512 << 10), "shards": rng.randint(1, 4),
                "levels": rng.choice(["2", "2,3,4", "2,3,4,5,6", "1,2,3"]), "copies": copies, "span": 256}
    if kind == "online":
        return {"kind": kind, "steps": rng.randint(2, 16), "step": _log(rng, 1 << 14, 1 << 19),
                "levels": rng.choice(["2,3,4,5,6", "2,3", "6,10,20", RECORD_LEVELS]), "copies": copies, "span": 256}
    if kind == "table":
        corpus = _log(rng, M, 100_000_000)
        return {"kind": kind, "corpus": corpus, "shards": rng.randint(1, 5),
                "queries": _log(rng, 65536, max(131072, corpus // 12)), "topk": rng.choice([0, 1, 4, 8]),
                "levels": rng.choice(["2,3,4", "1,2,3", "2,3", "3,6", "2"]), "copies": copies, "span": span}
    if kind == "longest":
        corpus = _log(rng, M, 1_000_000_000)
        return {"kind": kind, "corpus": corpus, "shards": rng.randint(1, 10),
                "queries": _log(rng, 65536, max(131072, corpus // 16)), "every": rng.choice([1, 4]),
                "cap": rng.choice([20, 32, 64]), "copies": copies, "span": span}
    if kind == "val_stats":
        corpus = _log(rng, M, 200_000_000)
        return {"kind": kind, "corpus": corpus, "shards": rng.randint(1, 4),
                "queries": _log(rng, 65536, max(131072, corpus // 16)), "copies": copies, "span": span}
    corpus = _log(rng, M, 1_000_000_000)
    return {"kind": kind, "corpus": corpus, "shards": rng.randint(1, 10),
            "queries": _log(rng, 65536, max(131072, corpus // 64)), "topk": rng.choice([0, 1, 2, 4, 8]),
            "levels": rng.choice(["2,3", "2,3,4,5,6,7,8", RECORD_LEVELS, "3,4,6", "6,10,20"]), "copies": copies,
            "span": span}


# ------------------------------------------------------------------------------------------------------------------
# Inputs
# ------------------------------------------------------------------------------------------------------------------

def _law(device):
    """The Zipf(1.1) law over ranks 1..50256 and the ranks' token ids: one law, as a language is one."""
    w = np.arange(1, BOS + 1, dtype=np.float64) ** -1.1
    cdf = np.cumsum(w) / w.sum()
    perm = np.random.Generator(np.random.PCG64(7)).permutation(BOS).astype(np.uint16)
    return torch.from_numpy(cdf).to(device), torch.from_numpy(perm.view(np.int16)).to(device)


def _stream(n, gen, rate, span, source=None):
    """n tokens (int16 holding uint16): documents of Zipf draws, `rate` of them with a span of up to `span` tokens copied
    from the stream itself or from `source`."""
    dev = gen.device
    cdf, perm = _law(dev)
    out = torch.empty(n, dtype=torch.int16, device=dev)
    for a in range(0, n, 64 * M):
        b = min(n, a + 64 * M)
        u = torch.rand(b - a, dtype=torch.float64, device=dev, generator=gen)
        out[a:b] = perm[torch.searchsorted(cdf, u, right=True).clamp_max_(BOS - 1)]
        out[a:b][torch.rand(b - a, device=dev, generator=gen) < 1.0 / DOC] = BOS - 65536
    src = out if source is None else source
    m = int(rate * n / DOC)
    if m:
        cell = n // m  # each copy lands in a stretch of its own, so the stream does not depend on the order they land in
        length = torch.randint(16, span + 1, (m,), device=dev, generator=gen).clamp_max_(min(cell, src.numel()) // 2)
        u, v = (torch.rand((2, m), dtype=torch.float64, device=dev, generator=gen))
        dst = torch.arange(m, device=dev) * cell + (u * (cell - length)).long()
        at = (v * (src.numel() - length)).long()
        pure = src.clone() if source is None else src
        within = torch.arange(int(length.sum()), device=dev) - torch.repeat_interleave(length.cumsum(0) - length, length)
        out[torch.repeat_interleave(dst, length) + within] = pure[torch.repeat_interleave(at, length) + within]
    return out


def _avail(x):
    """Per position the tokens of its document up to and including it (int32): a segment starts at 0 and at every BOS."""
    idx = torch.arange(x.numel(), device=x.device)
    start = x == BOS - 65536
    start[0] = True
    return (idx - torch.cummax(torch.where(start, idx, torch.zeros_like(idx)), 0).values + 1).to(torch.int32)


def _bounds(n, shards):
    """The shards' bounds in the stream: equal shards, the last one taking the rest."""
    return [i * (n // shards) for i in range(shards)] + [n]


def _inputs(case, seed):
    """The corpus laid out for the device (and without gaps, `flat`), and the query stream against it."""
    from ngram_amd import data

    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rate, span = case.get("copies", 0.10), case.get("span", 256)
    flat = _stream(case["corpus"], gen, rate, span)
    bounds = _bounds(case["corpus"], case.get("shards", 1))
    sizes = [b - a for a, b in zip(bounds, bounds[1:])]
    starts, length = data.pack_layout(sizes)
    tok = torch.full((length,), -1, dtype=torch.int16, device="cuda")
    for a, n, at in zip(bounds, sizes, starts):
        tok[at : at + n] = flat[a : a + n]
    q = _stream(case["queries"] + 1, gen, rate, span, flat)
    return SimpleNamespace(case=case, flat=flat, bounds=bounds, sizes=sizes, starts=starts, tok=tok, x=q[:-1].clone(),
                           tgt=q[1:].clone(), avail=_avail(q[:-1]))


def _levels(case):
    return [int(k) for k in case["levels"].split(",")]


def _tallies(case, seed):
    """Counts of the shapes a build gives (int32 [3, levels, n]): heavy-tailed totals, most contexts with few tokens."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    shape = (case["levels"], case["n"])
    tot = torch.exp2(torch.rand(shape, dtype=torch.float64, device="cuda", generator=gen) * 33 - 4).long()
    dist = torch.minimum((tot.double() ** torch.rand(shape, dtype=torch.float64, device="cuda", generator=gen)).long(),
                         torch.tensor(65535, device="cuda"))
    cnt = (tot * torch.rand(shape, dtype=torch.float64, device="cuda", generator=gen)).long()
    return torch.stack([tot, dist, cnt]).clamp_max_((1 << 31) - 1).to(torch.int32)


def prepare(case, seed):
    from ngram_amd.counts import CountBuild

    kind = case["kind"]
    if kind == "features":
        return SimpleNamespace(case=case, counts=_tallies(case, seed))
    if kind in ("online", "train_counts"):
        n = case["corpus"] if kind == "train_counts" else case["steps"] * case["step"]
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        tokens = _stream(n, gen, case["copies"], case["span"]).cpu().numpy().view(np.uint16)
        if kind == "train_counts":
            b = _bounds(n, case["shards"])
            return SimpleNamespace(case=case, shards=[tokens[lo:hi].copy() for lo, hi in zip(b, b[1:])])
        spans = np.array([(s * case["step"], (s + 1) * case["step"], s) for s in range(case["steps"])], np.int64)
        return SimpleNamespace(case=case, tokens=tokens, spans=spans)
    st = _inputs(case, seed)
    del st.flat
    if kind in ("counts", "batch_rows"):
        levels = _levels(case) if kind == "counts" else (6, 10, 20)
        st.build = CountBuild.from_device(st.tok, st.sizes, st.starts, levels=levels, level_shards={},
                                          topk=case.get("topk", 0))
        if kind == "batch_rows":  # the build is behind the training steps that cut their rows out of it
            st.build.counts(st.x, st.tgt, st.avail)
    if kind == "longest":
        st.query = None
        if case["every"] > 1:
            st.query = torch.zeros(case["queries"], dtype=torch.bool, device="cuda")
            st.query[case["every"] - 1 :: case["every"]] = True
    return st


# ------------------------------------------------------------------------------------------------------------------
# One pass
# ------------------------------------------------------------------------------------------------------------------

def run(st):
    case = st.case
    kind = case["kind"]
    if kind == "batch_rows":
        return st.build.batch_rows(case["queries"] - case["n"], case["n"], 4 * case["n"])
    if kind == "features":
        from ngram_amd import exact_match

        return exact_match.features(st.counts)
    if kind == "counts":
        b = st.build
        out = {"counts": b.counts(st.x, st.tgt, st.avail)}
        if case["topk"]:
            out["top_tok"], out["top_cnt"] = b.top_tok, b.top_cnt
        if {6, 10, 20} <= set(b.levels):
            out["cells"], out["entries"] = b.row_cells, b.row_entries
        return out
    if kind == "val_stats":
        from ngram_amd import gpu_val_stats

        r = gpu_val_stats.build_stats(st.tok, st.sizes, st.starts, st.x, st.tgt, st.avail)
        return {"counts": r["counts"], "rows": r["rows"]}
    if kind == "table":
        from ngram_amd.count_table import CountTable

        t = CountTable.from_device(st.tok, st.sizes, st.starts, _levels(case))
        t.build()
        return t.query_device(st.x, st.tgt, st.avail, topk=case["topk"])
    if kind == "longest":
        from ngram_amd.longest import longest_match

        length, nxt, cnt, _ = longest_match(st.tok, st.x, st.avail, case["cap"], query=st.query)
        return {"length": length, "next": nxt, "count": cnt}
    if kind == "train_counts":
        from ngram_amd import exact_match

        tot, dist, cnt = exact_match.train_counts(st.shards, _levels(case))
        return {"tot": tot.view(np.int32), "dist": dist.view(np.int16), "cnt": cnt.view(np.int32)}
    from ngram_amd.online import OnlineRows

    levels = _levels(case)
    rows = OnlineRows(st.tokens, [0, len(st.tokens)], st.spans)
    rows.prepare(levels, [2, 3, 4, 5, 6, 10, 20], 8, levels)
    rows.advance_device(case["steps"])
    o = rows.state["outs"]
    return {k: o[k] for k in ("cell", "next", "weights", "tot", "dist", "cnt")}


def work(case):
    kind = case["kind"]
    if kind == "features":
        per = case["n"] * case["levels"]
        return {"bytes": 12 * per + 28 * per, "flops": 2 * per}
    if kind == "batch_rows":
        return {"bytes": 36 * case["n"] + 4 * case["n"] * 9, "flops": 0}
    if kind == "online":
        n, nl = case["steps"] * case["step"], len(_levels(case))
        return {"bytes": 2 * n + n * (34 + 10 * nl), "flops": 0}
    if kind == "train_counts":
        return {"bytes": case["corpus"] * (2 + 10 * len(_levels(case))), "flops": 0}
    T, N = case["corpus"], case["queries"]
    b = 2 * T + 8 * N
    if kind == "longest":
        return {"bytes": b + 10 * N, "flops": 0}
    if kind == "val_stats":
        return {"bytes": b + N * (10 * 12 + 3 * 36), "flops": 0}
    levels = _levels(case)
    b += N * len(levels) * (12 + 6 * case["topk"])
    if kind == "counts" and {6, 10, 20} <= set(levels):
        b += 36 * N
    return {"bytes": b, "flops": 0}


def tolerance(case):
    # whole numbers, and floats that are whole numbers below 2^24 or round the way float32 does: the same bits
    return "exact"


# ------------------------------------------------------------------------------------------------------------------
# The same outputs by plain torch in 64-bit integers
# ------------------------------------------------------------------------------------------------------------------

EXACT_TOKENS = 110_000_000


class _Ladder:
    """The query contexts' ids, and where they occur in the corpus, level by level: a k-context's id is the rank of (the
    id of its first k - 1 tokens, its last token) among the queries'."""

    def __init__(self, st):
        self.c = st.flat.long() & 0xFFFF
        self.q = st.x.long() & 0xFFFF
        self.tgt = st.tgt.long() & 0xFFFF
        self.q_avail = st.avail
        idx = torch.arange(self.c.numel(), device=self.c.device)
        b = torch.tensor(st.bounds, device=self.c.device)
        part = torch.bucketize(idx, b[1:], right=True)
        self.c_avail = idx - b[part] + 1
        self.has_next = idx + 1 < b[part + 1]
        self.nxt = torch.cat([self.c[1:], self.c[:1]])
        self.k = 0
        self.c_id, self.q_id = torch.zeros_like(self.c), torch.zeros_like(self.q)

    def step(self):
        """One level deeper; the occurrences' pair keys (context id << 16 | next) and how often each occurs."""
        self.k += 1

        def key(i, t, ok):
            before = torch.cat([i[:1], i[:-1]]) if self.k > 1 else torch.zeros_like(i)
            return torch.where(ok & (before >= 0), (before << 16) | t, torch.full_like(t, -1))

        qk = key(self.q_id, self.q, self.q_avail >= self.k)
        u = torch.unique(qk)
        u = u[u >= 0]
        ck = key(self.c_id, self.c, self.c_avail >= self.k)

        def rank(v):
            if not u.numel():
                return torch.full_like(v, -1)
            r = torch.searchsorted(u, v).clamp_max(u.numel() - 1)
            return torch.where((u[r] == v) & (v >= 0), r, torch.full_like(r, -1))

        self.q_id, self.c_id, self.contexts = rank(qk), rank(ck), int(u.numel())
        hit = (self.c_id >= 0) & self.has_next
        return torch.unique((self.c_id[hit] << 16) | self.nxt[hit], return_counts=True)

    def level(self, topk, top_rule=None):
        """tot, dist, cnt [N] and the top lists [N, topk] of the level stepped to."""
        pairs, n = self.step()
        C, N, dev = max(1, self.contexts), self.q.numel(), self.q.device
        ctx = pairs >> 16
        tot = torch.zeros(C, dtype=torch.int64, device=dev).scatter_add_(0, ctx, n)
        dist = torch.bincount(ctx, minlength=C)
        # rank of each pair within its context: count descending, then token ascending (the pairs ascend already)
        order = torch.sort(n, descending=True, stable=True).indices
        order = order[torch.sort(ctx[order], stable=True).indices]
        first = dist.cumsum(0) - dist
        rank = torch.empty_like(order)
        rank[order] = torch.arange(order.numel(), device=dev) - first[ctx[order]]
        ok = self.q_id >= 0
        at = self.q_id.clamp_min(0)
        want = (at << 16) | self.tgt
        cnt = torch.zeros(N, dtype=torch.int64, device=dev)
        tok, top = (torch.zeros((N, topk), dtype=torch.int64, device=dev) for _ in range(2))
        if pairs.numel():
            j = torch.searchsorted(pairs, want).clamp_max(pairs.numel() - 1)
            found = ok & (pairs[j] == want)
            if top_rule is not None:
                found &= rank[j] < top_rule
            cnt = torch.where(found, n[j], cnt)
            for r in range(topk):
                has = ok & (dist[at] > r)
                p = order[(first[at] + r).clamp_max(order.numel() - 1)]
                tok[:, r] = torch.where(has, pairs[p] & 0xFFFF, tok[:, r])
                top[:, r] = torch.where(has, n[p], top[:, r])
        zero = torch.zeros_like(cnt)
        return torch.where(ok, tot[at], zero), torch.where(ok, dist[at], zero).clamp_max(65535), cnt, tok, top


def _exact_counts(st, levels, topk, top_rule=None):
    lad, out = _Ladder(st), []
    for k in range(1, max(levels) + 1):
        if k in levels:
            out.append(lad.level(topk, top_rule))
        else:
            lad.step()
    res = {"counts": torch.stack([torch.stack([o[j] for o in out]) for j in range(3)])}
    if topk:
        res["top_tok"] = _i16(torch.stack([o[3] for o in out]))
        res["top_cnt"] = torch.stack([o[4] for o in out])
    return res


def _i16(t):
    """uint16 values as the int16 of the same bits."""
    return torch.where(t >= 1 << 15, t - 65536, t).to(torch.int16)


def exact(case, seed):
    kind = case["kind"]
    if kind == "features":
        c = _tallies(case, seed).long()
        L, nb = case["levels"], 25
        lvl = torch.arange(L, device=c.device)[:, None]
        bins = torch.floor(torch.log2(c[0].clamp_min(1).float())).long().clamp(0, nb - 1) + nb * lvl
        flag = (c[1] == 1).long() + 2 * lvl + nb * L
        return (*[v.double().t().contiguous() for v in (c[0], c[1], torch.minimum(c[2], c[0]))],
                bins.t().contiguous(), flag.t().contiguous())
    if kind in ("batch_rows", "online", "train_counts") or case["corpus"] > EXACT_TOKENS:
        return None
    st = _inputs(case, seed)
    if kind == "val_stats":
        return {**_exact_counts(st, [int(k) for k in VAL_LEVELS.split(",")], 0, 1024), "rows": None}
    if kind == "table":
        return _exact_counts(st, _levels(case), case["topk"], 1024)
    if kind == "counts":
        res = _exact_counts(st, _levels(case), case["topk"])
        return {**res, "cells": None, "entries": None} if {6, 10, 20} <= set(_levels(case)) else res
    lad = _Ladder(st)
    length, nxt, cnt = (torch.zeros_like(lad.q) for _ in range(3))
    asked = torch.ones_like(lad.q, dtype=torch.bool)
    if case["every"] > 1:
        asked[:] = False
        asked[case["every"] - 1 :: case["every"]] = True
    for k in range(1, case["cap"] + 1):
        tot, _, _, tok, top = lad.level(1)
        on = asked & (tot > 0)
        length = torch.where(on, k, length)
        nxt, cnt = torch.where(on, tok[:, 0], nxt), torch.where(on, top[:, 0], cnt)
    return {"length": length, "next": _i16(nxt), "count": cnt}
