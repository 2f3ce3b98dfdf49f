"""Longest exact suffix match of query positions against a training corpus on one MI355X (configuration c5; the
match-length notion of exact_match/src/kgram.rs kgram_stats :38-56, 237-278, taken up to k = 64 by
src/retrieval_blog_post/kgram.py :16, 84-108): per query position i the largest k <= cap whose k-context
x[i-k+1..i] is valid (within its segment) and occurred in the corpus (k tokens within one shard followed by a token
of that shard), that context's most frequent next token (count descending, then token ascending) and its count; 0, 0,
0 if not even the 1-context occurred.

Two phases, both on libngram_amd.so. Existence, k = 1, 2, ...: the query contexts of the positions still matching
(a query index per level over the list of positions still matching), the corpus positions whose (k-1)-context
matched (a hit bitmap while dense, then a position list) probed for their k-context (ng_scan_exist: a bitmap, a
per-context hit bit and each hit position's context id, no counting), until no position matches; once the lists
shrink slowly, the remaining levels run as one stream of launches with device-side counts (ng_lm_levels: no host sync
per level). A match is monotone in k (kgram.rs:12-15), so each position's length is its last matching level. Then
counting, only for each position's final context: a bitmap level's hit positions whose stored context id is final emit
their (context, next) events (ng_scan_ids_emit: no second query index or probe); the list levels' final contexts share
one table, their key holding their length, which their listed positions are probed against (ng_lm_index,
ng_lm_lists_emit). The events of one level, or of a small corpus's levels together, are partitioned and counted in LDS
(partcount.py: no global atomics, so the hot pairs of short contexts cost no serialized chains), each context's top
entry made from its pairs and gathered to its positions (ng_lm_top1).

Surfaces: `longest_match(...)` on GPU tensors, and `LongestMatch.create(files, tokens, threads, cpus)` /
`build() -> dict` in cache_ladder's shape (cache_ladder/src/lib.rs:1-8, cache_ladder.pyi)."""

from __future__ import annotations

import ctypes
import os
import time
from types import SimpleNamespace

import numpy as np
import torch


from .data import BOS, HEADER_BYTES, shard_tokens
from .data import pack_layout as layout
from .lib import Lib, i32, u64
from .partcount import (W_MAX, count32, count_events, emit_region, first_digit, key_mbits, pack_events, pbits32_max,
                        runs_fit, summarize, w_bits)
from .qindex import LOAD as QLOAD, TAIL as QTAIL, QueryIndex


_RATIO: dict[int, float] = {}  # distinct pairs per counted event at each level, from the last count (sizes partitions)
# levels (and "lists", the list levels together) whose 32-bit count overflowed by itself: counted by the 64-bit path
_WIDE: set = set()
# each existence level's query contexts per listed position in the last call: sizes the next call's query index for
# its own number of positions
_CONTEXTS: dict[int, float] = {}


def longest_match(tok: torch.Tensor, x: torch.Tensor, avail: torch.Tensor, cap: int = 64, elib: Lib | None = None,
                  lib: Lib | None = None, timing: dict | None = None, query: torch.Tensor | None = None):
    """Per query position (x int16 [N] inputs, avail int32 [N] tokens since the segment start): (length int32,
    next int16 (uint16 bits), count int32 (uint32 bits)) of its longest match <= cap, and per level
    (k, eligible, matched) over the existence phase. `tok`: the corpus laid out with SENT gaps (layout()).
    `query` (bool [N], optional): only these positions are queried (their contexts still read x before them); the
    others get 0, 0, 0."""
    if not 1 <= cap <= 64:
        raise ValueError("cap must be in [1, 64]")
    EVENTS[0] = 0
    elib = elib or Lib()
    lib = lib or Lib()
    dev = x.device
    N, L = x.numel(), tok.numel()
    nwords = L // 32
    # scan blocks: as many as the device takes, but at least 8192 positions each (a block's hits are a segment of the
    # count's first pass, whose cost per segment a small corpus would otherwise pay thousands of times)
    grid = max(1, min(torch.cuda.get_device_properties(dev).multi_processor_count * SCAN_BLOCKS_PER_CU, -(-L // 8192)))
    t0 = time.perf_counter()
    length = elib.zeros(N, torch.int32, dev)
    # the queried positions, as a list; each level keeps the ones still matching (the lists shrink fast). meta holds what
    # the host reads: the positions by min(avail, cap), then per level the positions kept for the next one, those matched,
    # the corpus positions hit, and the query index's counters (row 0: the queried positions)
    meta = elib.zeros(cap + 1 + 6 * (cap + 2), torch.int64, dev)
    hist, rows = meta[: cap + 1], meta[cap + 1 :].view(cap + 2, 6)
    act = torch.empty(max(N, 1), dtype=torch.int32, device=dev)
    mask = None
    if query is not None:
        # torch combines the two: it refuses a mask in host memory, which the kernel would read through its address, and
        # one of another shape
        mask = torch.ne((avail >= 1) & query, 0).expand(N).view(torch.uint8)
    elib("ng_lm_select", avail, mask, N, i32(cap), act, rows[0], hist)
    # each level's hit set (the corpus positions whose k-context is a query context of the level): a bitmap while
    # dense, then, once sparse, a list of positions, which the next level scans instead of every bitmap word
    levels: list[tuple] = []
    ladder = []
    flags = elib.zeros(2, torch.int32, dev)
    # the prefix rule for the bitmap scans (a device flag, no host sync): with every position queried, a position
    # still active at level k has its predecessor active at level k - 1 (its shorter context occurs wherever the
    # longer one does), so where avail is segment-shaped a level's context also has its prefix among the level before's
    # and a corpus position is probed only where the level before hit it and the position before it. A query mask can
    # leave a predecessor out, so it turns the rule off.
    pre = None
    if query is None:
        pre = torch.empty(1, dtype=torch.int32, device=dev)
        elib("ng_avail_closed", avail, N, pre)
    elig: list = []
    deep = None  # the list levels' first level and its active positions
    n_act = N  # level 1's is read with its results; later levels' are exact
    for k in range(1, cap + 1):
        if n_act == 0:
            break
        prev = levels[-1] if levels else None
        sparse = prev is not None and (prev[0] == "list" or prev[2] * LIST_DIV < L)
        if sparse and deep is None:
            deep = (k, act, n_act)
        if sparse and DEVICE_LEVELS:
            # the sparse levels' lists shrink slowly from here on: the remaining levels run without a host sync
            cand = prev[1] if prev[0] == "list" else _bits_list(elib, prev[1], prev[2])
            for k2, hl, nh, matched in _exist_device(elib, tok, L, x, avail, act[:n_act], k, cap, cand, length, flags,
                                                     grid):
                levels.append(("list", hl, nh))
                ladder.append((k2, elig[k2], matched))
            break
        row = rows[k]
        nxt_act = torch.empty(max(n_act, 1), dtype=torch.int32, device=dev)
        if k == 1:
            # level 1: a 1-context's id is its token, so no query table (ng_scan_tok1 holds the query tokens' set)
            ctx_of = torch.empty(max(N, 1), dtype=torch.int32, device=dev)
            member = elib.zeros(2048, torch.int32, dev)
            elib("ng_lm_tok1", x, act, rows[0], N, ctx_of, member)
            hit = elib.zeros(2048, torch.int32, dev)
            bm = torch.empty(nwords, dtype=torch.int32, device=dev)
            # no stored ids: a hit's context id is the token before it, which the counting scan reads itself
            elib("ng_scan_tok1", tok, L, member, bm, hit, None, i32(TOK1_GRID))
            level = ["bm", bm, 0, None, act, ctx_of, 65536]
            lib("popcount", bm, nwords, row[2:])
            elib("ng_act_next", act, rows[0], N, ctx_of, hit, avail, i32(1), length, nxt_act, row, row[1:])
            host = meta.cpu().tolist()
            n_act = host[cap + 1]
            elig = [sum(host[j : cap + 1]) for j in range(cap + 1)]
            if n_act == 0:
                break
        elif sparse:
            host = _exist_list(elib, tok, L, x, avail, act, n_act, k, prev, length, flags, grid, row, nxt_act)
            level = ["list", host.pop(), 0]
        else:
            per = _CONTEXTS.get(k)
            expect = None if per is None else int(per * n_act) + 1
            for checked in (False, True):
                # sized from the last call's contexts, its counters read with the level's results; an index that proves
                # too small for this call's contexts is built again, sized and checked as it is built
                vi = QueryIndex(elib, x, avail, k, act[:n_act], compact=True, expect=expect,
                                defer=not checked and expect is not None, counters=row[3:6])
                hit = elib.zeros((vi.ids + 31) // 32, torch.int32, dev)  # a bit per context id
                bm = torch.empty(nwords, dtype=torch.int32, device=dev)
                ids = torch.empty(L, dtype=torch.int32, device=dev)  # each hit position's context id, for the counting
                mode = 0 if prev[2] * 2 > L else 2  # a lane per position while the gate is dense
                elib("ng_scan_exist", tok, L, i32(k), prev[1], bm, vi.table, u64(vi.cap), vi.rep, x, hit, ids, flags,
                     i32(grid), i32(mode), pre)
                lib("popcount", bm, nwords, row[2:])
                elib("ng_act_next", act, rows[k - 1] if k > 1 else rows[0], n_act, vi.ctx_of, hit, avail, i32(k), length,
                     nxt_act, row, row[1:])
                host = rows[k].cpu().tolist()
                if vi.n is not None:
                    break
                if host[5]:
                    raise RuntimeError(f"k={k}: {host[5]} query positions collide with another context's key")
                vi.n = host[3]
                if not host[4] and vi.n <= 2 * QLOAD * vi.cap:
                    break
                elib.fill(row, 0)
            _CONTEXTS[k] = vi.n / max(1, n_act)
            level = ["bm", bm, 0, ids, act, vi.ctx_of, vi.ids]
            del vi, hit
        r = host[-6:] if k > 1 else host[cap + 1 + 6 * k : cap + 1 + 6 * k + 6]
        level[2] = r[2]
        if level[0] == "bm":
            level.append(n_act)
        else:
            level[1] = level[1][: r[2]]
        levels.append(tuple(level))
        ladder.append((k, elig[k], r[1]))
        act, n_act = nxt_act, r[0]
    if timing is not None:
        torch.cuda.synchronize()
        timing["exist"] = timing.get("exist", 0.0) + time.perf_counter() - t0
        t0 = time.perf_counter()
    nxt = elib.fill(torch.empty(N, dtype=torch.int16, device=dev), 0)
    cnt = elib.zeros(N, torch.int32, dev)
    _count(elib, lib, tok, L, x, avail, levels, ladder, deep, length, flags, grid, nxt, cnt)
    if timing is not None:
        torch.cuda.synchronize()
        timing["count"] = timing.get("count", 0.0) + time.perf_counter() - t0
        timing["events"] = float(EVENTS[0])
    return length, nxt, cnt, ladder


def _exist_list(elib: Lib, tok, L: int, x, avail, act, n_act: int, k: int, prev: tuple, length, flags, grid: int, row,
                nxt_act) -> list:
    """One list level of the existence phase with host reads (the device levels' counterpart): the level's row of meta,
    its hit list last."""
    vi = QueryIndex(elib, x, avail, k, act[:n_act], compact=True)
    _CONTEXTS[k] = vi.n / max(1, n_act)
    hit = elib.zeros((vi.ids + 31) // 32, torch.int32, x.device)
    cand = prev[1] if prev[0] == "list" else _bits_list(elib, prev[1], prev[2])
    hl, nh = _scan_list(elib, tok, L, k, vi, x, cand, hit, 1, flags, grid)
    n_dev = torch.tensor([n_act], dtype=torch.int64, device=x.device)
    elib("ng_act_next", act, n_dev, n_act, vi.ctx_of, hit, avail, i32(k), length, nxt_act, row, row[1:])
    row[2:3].fill_(nh)
    return row.cpu().tolist() + [hl]


def _count(elib: Lib, lib: Lib, tok, L: int, x, avail, levels: list, ladder: list, deep, length, flags, grid: int, nxt,
           cnt) -> None:
    """The counting phase: each position's final context (of its length k) counted, its top entry to nxt / cnt. Levels are
    counted together, their context ids offset, while the ids fit the 32-bit count and the scan regions GROUP_EVENTS: a
    small corpus's levels cost one count's launches, not one each."""
    matched = [m for _, _, m in ladder] + [0]
    final = [matched[j] - matched[j + 1] for j in range(len(ladder))]  # positions whose match ends at level j + 1
    lists = [k for k in range(1, len(levels) + 1) if levels[k - 1][0] == "list" and final[k - 1]]
    R = emit_region(L, grid)
    group: list = []
    used = cap_ev = 0
    for k in [k for k in range(1, len(levels) + 1) if levels[k - 1][0] == "bm" and final[k - 1]] + (["lists"] if lists
                                                                                                    else []):
        if k == "lists":
            ids, ev = int(deep[2] / QLOAD) + 1024 + QTAIL, sum(levels[j - 1][2] for j in lists)
        else:
            ids, ev = levels[k - 1][6], grid * R
        ids = (ids + 31) // 32 * 32  # each level's final bits start at a word
        # by the 64-bit count, alone: a level that needs it, and list levels of more positions than one of its batches takes
        # (room for all of them at once is 8 bytes each several times over, and the 32-bit count's offsets end at 2^32)
        if k in _WIDE or w_bits(ids)[1] > W_MAX or (k == "lists" and ev > BATCH_EVENTS):
            _count_wide(elib, lib, tok, L, x, avail, [k], lists, levels, length, flags, grid, nxt, cnt)
            continue
        if group and (w_bits(used + ids)[1] > W_MAX or cap_ev + ev > GROUP_EVENTS):
            _count_group(elib, lib, tok, L, x, avail, group, lists, levels, deep, length, flags, grid, nxt, cnt)
            group, used, cap_ev = [], 0, 0
        group.append((k, used, ids))
        used += ids
        cap_ev += ev
    if group:
        _count_group(elib, lib, tok, L, x, avail, group, lists, levels, deep, length, flags, grid, nxt, cnt)


def _count_group(elib: Lib, lib: Lib, tok, L: int, x, avail, group: list, lists: list, levels: list, deep, length, flags,
                 grid: int, nxt, cnt) -> None:
    """The levels of `group` ((k, first id, ids), or ("lists", ...): the list levels with final positions) in one 32-bit
    count. A bitmap level's final contexts are marked in a bit set and its stored ids emit their events; the list levels'
    final contexts go into one table, which their listed positions are probed against (ng_lm_index, ng_lm_lists_emit)."""
    dev = x.device
    N = x.numel()
    n_ids = sum(ids for _, _, ids in group)
    _, W = w_bits(n_ids)
    d1 = first_digit(W)
    # events keyed by context range only for a level by itself: several levels' id ranges hold far from equal events, and
    # the partitions of the densest would overflow
    mbits = key_mbits(W) if len(group) == 1 and runs_fit(n_ids, 1) else W
    bms = [g for g in group if g[0] != "lists"]
    total = sum(levels[k - 1][2] for k in lists) if len(bms) < len(group) else 0
    R = emit_region(L, grid) if bms else 0
    gl = 0
    if total or len(bms) < len(group):
        gl = max(1, min(grid, -(-total // 1024)))
        if R:
            gl = max(gl, -(-total // R))
        R = max(R, -(-max(total, 1) // (gl * 256)) * 256)
    nseg = len(bms) * grid + gl
    regions = torch.empty(nseg * R, dtype=torch.int64, device=dev)
    ev_count = torch.empty(nseg, dtype=torch.int32, device=dev)
    dhist = torch.empty((1 << d1) * nseg, dtype=torch.int32, device=dev)
    fid = elib.full_ones(N, torch.int32, dev)
    bits = elib.zeros(n_ids // 32, torch.int32, dev)
    elib.fill(flags, 0)
    for j, (k, base, ids) in enumerate(bms):
        _, bm, _, stored, act, ctx_of, _, n_act = levels[k - 1]
        elib("ng_lm_final", act, n_act, ctx_of, length, i32(k), i32(base), fid, bits[base // 32 :])
        elib("ng_scan_ids_emit_at", tok, L, bm, stored, bits[base // 32 :], regions[j * grid * R :], u64(R),
             ev_count[j * grid :], flags, i32(grid), dhist[j * grid :], nseg, i32(W), i32(d1), i32(mbits),
             u64(base << 16))
    counters = None
    if gl:
        _, base, _ = group[-1]
        k0, act0, n0 = deep
        qcap = int(n0 / QLOAD) + 1024
        slots = qcap + QTAIL
        table = elib.full_ones(slots, torch.int64, dev)
        rep = torch.empty(slots, dtype=torch.int32, device=dev)
        counters = elib.zeros((65, 3), torch.int64, dev)
        elib("ng_lm_index", x, act0, n0, length, i32(k0), table, u64(qcap), u64(slots), rep, i32(base), fid, counters)
        rows = (ctypes.c_int64 * (3 * len(lists)))(*[v for k in lists for v in (levels[k - 1][1].data_ptr(),
                                                                               levels[k - 1][2], k)])
        at = len(bms) * grid
        elib("ng_lm_lists_emit", tok, rows, i32(len(lists)), table, u64(qcap), rep, x, length, regions[at * R :], u64(R),
             ev_count[at:], flags, i32(gl), dhist[at:], nseg, i32(W), i32(d1), i32(mbits), u64(base << 16))
    key = tuple(k for k, _, _ in group)
    min_pbits = 0
    seg = (regions, R, ev_count, dhist, nseg, flags)
    while True:
        c = count32(elib, seg, n_ids, 1, None, None, _RATIO.get(key, 1.0), min_pbits=min_pbits, mbits=mbits)
        got = torch.cat([c.stat[:3], flags[:1].to(torch.int64)] + ([counters.view(-1)] if gl else [])).tolist()
        n_ev, n_u, fl, sfl = got[:4]
        if sfl & 4:
            raise RuntimeError(f"levels {key}: an emit region overflowed")
        if fl & 4:
            raise RuntimeError(f"levels {key}: a total does not fit uint32")
        over = False
        for k in lists if gl else ():
            _, o, coll = got[4 + 3 * k : 7 + 3 * k]
            if coll:
                raise RuntimeError(f"k={k}: {coll} query positions collide with another context's key")
            over |= o != 0
        if over:  # an insert found no slot: the list levels by themselves, their indexes checked as they are built
            del regions, seg, c, dhist
            _count_wide(elib, lib, tok, L, x, avail, ["lists"], lists, levels, length, flags, grid, nxt, cnt)
            bms_left = [g for g in group if g[0] != "lists"]
            if bms_left:
                _count_group(elib, lib, tok, L, x, avail, bms_left, lists, levels, deep, length, flags, grid, nxt, cnt)
            return
        if fl & 1 and not fl & 2 and c.pbits < pbits32_max(n_ids):  # a partition overfull: counted with a bit more
            min_pbits = c.pbits + 1
            continue
        break
    if fl & 3:  # its escape table overflowed, or no more partition bits
        del regions, seg, c, dhist
        if len(group) > 1:  # one level's doing, or only all of them together: each by itself
            for k, _, ids in group:
                _count_group(elib, lib, tok, L, x, avail, [(k, 0, ids)], lists, levels, deep, length, flags, grid, nxt, cnt)
            return
        k = group[0][0]  # this level takes the 64-bit count from now on
        _WIDE.add(k)
        _count_wide(elib, lib, tok, L, x, avail, [k], lists, levels, length, flags, grid, nxt, cnt)
        return
    _RATIO[key] = n_u / max(1, n_ev)
    EVENTS[0] += n_ev
    elib("ng_lm_top1", fid, N, n_ids, c.rec, c.dist, nxt, cnt)


def _count_wide(elib: Lib, lib: Lib, tok, L: int, x, avail, ks: list, lists: list, levels: list, length, flags, grid: int,
                nxt, cnt) -> None:
    """Levels by the 64-bit count: a bitmap level from its stored ids, the list levels with an index each, checked, in
    batches."""
    for k in ks:
        if k != "lists":
            level = levels[k - 1]
            n_act = level[7]
            _count_ids(elib, lib, tok, L, (*level[:4], level[4][:n_act], level[5][:n_act], level[6]), k, length, flags,
                       grid, nxt, cnt)
            continue
        batch, ev = [], 0
        for j in lists:
            fpos = torch.nonzero(length == j).squeeze(1).to(torch.int32)
            batch.append((j, fpos, QueryIndex(elib, x, avail, j, fpos, compact=True)))
            ev += levels[j - 1][2]
            if ev >= BATCH_EVENTS or j == lists[-1]:
                _count_batch(elib, lib, tok, L, x, avail, batch, levels, flags, grid, nxt, cnt)
                batch, ev = [], 0


SCAN_BLOCKS_PER_CU = 32  # scan blocks per compute unit
TOK1_GRID = 2048  # level 1's scan blocks (each ORs its hit words into the level's once)
EVENTS = [0]  # (context, next) events the last longest_match counted (its counting phase), for its timing dict
DEVICE_LEVELS = True  # the existence phase's levels after the second list level run without host syncs
LONG_FIRST = 8  # the device levels try level cap first when at least this many levels lie between
# Levels are counted together until their scan regions hold this many events. At limits of 0 / 2^26 / 2^28 / 2^30: 4M tokens
# 4.59 / 2.43 / 2.42 / 2.42 ms a call, 16M 9.17 / 6.85 / 6.59 / 6.59, 64M 15.8 / 15.8 / 13.8 / 13.5, 256M 31.7 / 31.8 / 31.8 /
# 32.1, 1e9 115.4 at each; but a group's regions are held at once, and 64M tokens peak at 4.5 / 4.5 / 7.8 / 17.1 GiB.
GROUP_EVENTS = 1 << 26
BATCH_EVENTS = 1 << 28  # list levels counted together by the 64-bit count until their listed positions reach this
LIST_DIV = 64  # a level's hits go to a position list once fewer than L / LIST_DIV (8 B each against L / 8 bitmap bytes)


def _exist_device(elib: Lib, tok, L: int, x, avail, act, k0: int, cap: int, cand, length, flags, grid: int):
    """Levels k0..cap of the existence phase launched by one call with no host sync (ng_lm_levels), every buffer sized by
    level k0's active positions (act, all with avail >= k0) and candidates (cand: the corpus positions that matched
    k0 - 1), which bound every later level's. One sync at the end reads each level's sizes; the levels are those whose
    active list was not empty, as the host loop's. Returns [(k, hit list, its length, matched positions)].

    With LONG_FIRST or more levels to go, level `cap` is tried first (the cap round): a position whose cap-token
    context occurs matches every level below it too (a context's suffixes occur wherever it does), so it is done at
    length cap, and the levels in between are walked by the others only. Their hit lists then hold only those
    positions' contexts' occurrences, and level cap's is the round's. The long copies of a corpus make most of the
    deep levels' positions such ones: they would otherwise be probed, and their occurrences listed, at every level."""
    dev = x.device
    n0, nc0 = int(act.numel()), int(cand.numel())
    qcap = int(n0 / QLOAD) + 1024
    slots = qcap + QTAIL
    table = elib.full_ones(slots, torch.int64, dev)
    rep = torch.empty(slots, dtype=torch.int32, device=dev)
    lvl = elib.fill(torch.empty((slots + 7) // 8 * 8, dtype=torch.uint8, device=dev), 0)
    ctx_of, act_a, act_b = (torch.empty(max(n0, 1), dtype=torch.int32, device=dev) for _ in range(3))
    nlev = cap - k0 + 1
    first = cap - k0 >= LONG_FIRST
    hl = torch.empty((nlev, max(nc0, 1)), dtype=torch.int64, device=dev)
    meta = elib.zeros((nlev + 1, 6), torch.int64, dev)
    elib("ng_lm_levels", tok, x, avail, i32(k0), i32(cap), i32(int(first)), act, n0, act_a, act_b, cand, nc0, table,
         u64(qcap), u64(slots), rep, ctx_of, lvl, hl, length, meta, flags, i32(grid))
    host = meta.cpu().tolist()
    if any(r[4] for r in host[:nlev]):
        raise RuntimeError(f"levels {k0}..{cap}: a query index was too small for its contexts")
    if any(r[5] for r in host[:nlev]):
        raise RuntimeError(f"levels {k0}..{cap}: query positions collide with another context's key")
    going, done = (host[-1][0], host[-1][1]) if first else (n0, 0)  # done: the positions done at length cap
    res = []
    active = going
    for j, k in enumerate(range(k0, cap + 1)):
        kept, matched, nh = host[j][:3]
        if first and k == cap:  # its trial took place first: the others that reached it did not match
            matched = 0
        if active + done == 0:
            break
        res.append((k, hl[j, :nh], nh, matched + done))
        active = kept
    return res


def _count_ids(elib: Lib, lib: Lib, tok, L: int, level: tuple, k: int, length, flags, grid: int, nxt, cnt) -> None:
    """The counting phase of a bitmap level from what its existence scan kept: the hit bitmap, each hit position's
    context id (None at level 1 by token: the token before the position), and the level's active positions with their
    context ids. The final contexts (those of the positions
    whose match ends at k) are marked in a bit set; the hit positions of final contexts emit their (context, next)
    events (ng_scan_ids_emit), which are partitioned, counted and summarized per context (top entry), then gathered
    to the final positions."""
    _, bm, nh, ids, act, ctx_of, n_ids = level
    dev = bm.device
    fin = length[act.long()] == k
    fids = ctx_of[fin]
    fpos = act[fin].long()
    m = fids.numel()
    if m == 0:
        return
    final = torch.zeros((n_ids + 31) // 32, dtype=torch.int32, device=dev)
    elib("ng_mark_bits", fids, m, final)
    R = emit_region(L, grid)
    regions = torch.empty(grid * R, dtype=torch.int64, device=dev)
    ev_count = torch.empty(grid, dtype=torch.int32, device=dev)
    dhist = torch.empty(256 * grid, dtype=torch.int32, device=dev)
    flags.zero_()
    elib("ng_scan_ids_emit", tok, L, bm, ids, final, regions, u64(R), ev_count, flags, i32(grid), dhist, grid, i32(0),
         i32(0), i32(0))
    try:  # the scan's flags read with the event total
        c = count_events(elib, lib, None, 0, n_ids, _RATIO.get(k, 1.0),
                         seg=(regions, R, ev_count, dhist, grid, flags), presort="ctx")
    except RuntimeError as e:
        raise RuntimeError(f"k={k}: {e}") from None
    del regions
    _RATIO[k] = c.U / max(1, c.n_ev)
    EVENTS[0] += c.n_ev
    o_tok = torch.zeros(m, dtype=torch.int16, device=dev)
    o_cnt = torch.zeros(m, dtype=torch.int32, device=dev)
    if c.cb:
        sm = summarize(elib, lib, c, n_ids, 1)
        o = [torch.empty(m, dtype=torch.int32, device=dev) for _ in range(3)]
        elib("ng_pos_summary", fids, m, 0, n_ids, None, sm.rec, sm.dist, None, None, i32(1), i32(1), i32(0), o[0], o[1],
             o[2], o_tok, o_cnt, None, None)
    else:  # unpacked pairs: sorted by key, per-context top entry by selection
        _top1_unpacked(elib, lib, SimpleNamespace(ctx_of=fids, ids=n_ids), c, None, o_tok, o_cnt)
    nxt[fpos] = o_tok
    cnt[fpos] = o_cnt


def _bits_list(elib: Lib, bm: torch.Tensor, n: int) -> torch.Tensor:
    """The set positions of a bitmap (n of them) as a u64 list."""
    out = torch.empty(max(n, 1), dtype=torch.int64, device=bm.device)
    total = torch.zeros(1, dtype=torch.int64, device=bm.device)
    elib.cub("ng_bits_list", bm, bm.numel(), out, total, None)
    return out[:n]


def _scan_list(elib: Lib, tok, L: int, k: int, vi, x, cand: torch.Tensor, hit, what: int, flags, grid: int):
    """A level scan of listed corpus positions: hits flagged per context (hit may be None) and emitted as positions
    (what 1) or mixed pair keys (what 0), packed: (list, n)."""
    n = cand.numel()
    g = max(1, min(grid, -(-n // 256)))  # a round of 256 entries per block: as many blocks as fill the GPU
    R = -(-max(n, 1) // (g * 256)) * 256  # a list scan's block emits at most 256 per round
    regions = torch.empty(g * R, dtype=torch.int64, device=cand.device)
    ev_count = torch.empty(g, dtype=torch.int32, device=cand.device)
    elib("ng_scan_sink", tok, L, i32(k), None, None, cand, n, vi.table, u64(vi.cap), vi.rep, x, hit, i32(what),
         regions, u64(R), ev_count, flags, i32(g), i32(0), u64(0))
    out, m = pack_events(elib, regions, R, ev_count, g)
    return out[:m] if what else out, m


def _count_batch(elib: Lib, lib: Lib, tok, L: int, x, avail, batch: list, levels: list, flags, grid: int, nxt,
                 cnt) -> None:
    """The counting phase of several list levels at once: level k's context ids offset by the ids before it in the
    batch, so one partitioned count, one summary and one gather serve them all (per level only its query index and
    its scan: few launches and no host sync per level)."""
    dev = x.device
    bases, n_ids = [], 0
    for _, _, vi in batch:
        bases.append(n_ids)
        n_ids += vi.ids
    cap_ev = sum(levels[k - 1][2] for k, _, _ in batch)  # each listed position emits at most one event
    ev = torch.empty(max(cap_ev, 1), dtype=torch.int64, device=dev)
    at = torch.zeros(1, dtype=torch.int64, device=dev)  # the events packed so far (device side)
    flags.zero_()
    for (k, _, vi), b in zip(batch, bases):
        _, hs, nh = levels[k - 1]
        g = max(1, min(grid, -(-nh // 256)))
        R = -(-max(nh, 1) // (g * 256)) * 256
        regions = torch.empty(g * R, dtype=torch.int64, device=dev)
        ev_count = torch.empty(g, dtype=torch.int32, device=dev)
        elib("ng_scan_sink", tok, L, i32(k), None, None, hs, nh, vi.table, u64(vi.cap), vi.rep, x, None, i32(0),
             regions, u64(R), ev_count, flags, i32(g), i32(0), u64(b << 16))
        offs = torch.empty(g + 1, dtype=torch.int64, device=dev)
        elib("ng_seg_offsets", ev_count, g, offs)
        offs += at
        elib("ng_seg_gather", regions, None, u64(R), None, ev_count, g, offs, ev, None)
        at = offs[g : g + 1].clone()
        del regions, ev_count
    n_ev, fl = torch.cat([at, flags[:1].to(torch.int64)]).tolist()  # one copy
    if fl & 4:
        raise RuntimeError(f"levels {batch[0][0]}..{batch[-1][0]}: an emit region overflowed")
    key = ("batch", batch[0][0])
    c = count_events(elib, lib, ev, n_ev, n_ids, _RATIO.get(key, 1.0), presort="ctx")
    del ev
    _RATIO[key] = c.U / max(1, n_ev)
    EVENTS[0] += n_ev
    if not c.cb:
        raise RuntimeError(f"levels {batch[0][0]}..{batch[-1][0]}: more large counts than the escape table holds")
    sm = summarize(elib, lib, c, n_ids, 1)
    fpos = torch.cat([f for _, f, _ in batch]).long()
    ctx_of = torch.cat([torch.where(vi.ctx_of >= 0, vi.ctx_of + b, -1) for (_, _, vi), b in zip(batch, bases)])
    m = fpos.numel()
    o_tok = torch.zeros(m, dtype=torch.int16, device=dev)
    o_cnt = torch.zeros(m, dtype=torch.int32, device=dev)
    o_tot = torch.empty(m, dtype=torch.int32, device=dev)
    o_dist = torch.empty(m, dtype=torch.int32, device=dev)
    o_tc = torch.empty(m, dtype=torch.int32, device=dev)
    elib("ng_pos_summary", ctx_of, m, 0, n_ids, None, sm.rec, sm.dist, None, None, i32(1), i32(1), i32(0), o_tot, o_dist,
         o_tc, o_tok, o_cnt, None, None)
    nxt[fpos] = o_tok
    cnt[fpos] = o_cnt


def _top1_unpacked(elib: Lib, lib: Lib, vi, c, x, o_tok, o_cnt) -> None:
    """The final contexts' top entries from unpacked (pair key, count) pairs (compact ctx_of, m entries)."""
    dev = o_tok.device
    m = vi.ctx_of.numel()
    ctx_bits = max(1, (max(vi.ids, 2) - 1).bit_length())
    uk = torch.empty(c.U, dtype=torch.int64, device=dev)
    agg = torch.empty(c.U, dtype=torch.int32, device=dev)
    if c.U:
        lib.cub("sort_pairs", c.pairs, uk, c.counts, agg, c.U, i32(0), i32(16 + ctx_bits))
    start = torch.zeros(vi.ids, dtype=torch.int64, device=dev)
    end = torch.zeros(vi.ids, dtype=torch.int64, device=dev)
    tot = torch.zeros(vi.ids, dtype=torch.int64, device=dev)
    top_tok = torch.zeros(vi.ids, dtype=torch.int16, device=dev)
    top_cnt = torch.zeros(vi.ids, dtype=torch.int32, device=dev)
    lib("seg_bounds", uk, c.U, start, end)
    elib("ng_ctx_topk", uk, agg, start, end, vi.ids, i32(1), tot, top_tok, top_cnt)
    o = [torch.zeros(m, dtype=torch.int32, device=dev) for _ in range(3)]
    tgt = torch.zeros(m, dtype=torch.int16, device=dev)
    elib("ng_pos_gather", vi.ctx_of, m, 0, vi.ids, tgt, uk, agg, start, end, tot, top_tok, top_cnt, None, None, None,
         u64(0), None, i32(1), i32(1), i32(0), o[0], o[1], o[2], o_tok, o_cnt, None)


def _segments(x: torch.Tensor, lib: Lib) -> torch.Tensor:
    n = x.numel()
    idx = torch.arange(n, device=x.device)
    start = (x.to(torch.int32) & 0xFFFF) == BOS
    start[:1] = True
    seg = torch.empty_like(idx)
    if n:
        lib.cub("inclusive_max", torch.where(start, idx, torch.zeros_like(idx)), seg, n)
    return (idx - seg + 1).to(torch.int32)


class LongestMatch:
    """The longest match as a ladder rung (cache_ladder's interface, cache_ladder/src/lib.rs:1-8): create(files,
    tokens, threads, cpus) reads the training shards and the query stream (`tokens`: the inputs, then the last one's
    next token) before the clock; build() runs the match on the clock and returns its timings (seconds) and sizes;
    afterwards `length`, `next` (uint16) and `count` (uint32) hold the per-position results (numpy)."""

    def __init__(self):
        raise TypeError("use LongestMatch.create(files, tokens, threads, cpus)")

    @staticmethod
    def create(files: list, tokens, threads: int = 1, cpus: list[int] = (), cap: int = 64) -> "LongestMatch":
        self = object.__new__(LongestMatch)
        arrays = []
        for f in files:
            if isinstance(f, (str, bytes, os.PathLike)):
                n = shard_tokens(f)
                arrays.append(np.fromfile(f, dtype="<u2", count=n, offset=HEADER_BYTES))
            else:
                arrays.append(np.ascontiguousarray(f, dtype=np.uint16))
        q = np.ascontiguousarray(tokens, dtype=np.uint16)
        if not arrays or len(q) < 2 or int(q.max()) > BOS or any(len(a) and int(a.max()) > BOS for a in arrays):
            raise ValueError("need training shards and 2+ valid query tokens")
        sizes = [len(a) for a in arrays]
        starts, L = layout(sizes)
        dev = torch.device("cuda", torch.cuda.current_device())
        self.tok = torch.full((L,), -1, dtype=torch.int16, device=dev)
        for a, st in zip(arrays, starts):
            if len(a):
                self.tok[st : st + len(a)].copy_(torch.from_numpy(a.view(np.int16)))
        self.x = torch.from_numpy(q[:-1].view(np.int16).copy()).to(dev)
        self.cap = cap
        self.elib = self.lib = Lib()
        self.avail = _segments(self.x, self.lib)
        self.tokens = int(sum(sizes))
        torch.cuda.synchronize()
        return self

    def build(self) -> dict:
        timing: dict = {}
        t0 = time.perf_counter()
        length, nxt, cnt, ladder = longest_match(self.tok, self.x, self.avail, self.cap, self.elib, self.lib, timing)
        torch.cuda.synchronize()
        timing["total"] = time.perf_counter() - t0
        self.length = length.cpu().numpy().view(np.uint32)
        self.next = nxt.cpu().numpy().view(np.uint16)
        self.count = cnt.cpu().numpy().view(np.uint32)
        self.ladder = ladder
        timing["levels"] = float(len(ladder))
        return timing
