"""Online causal rows under the step rule on one MI355X, behind exact_match's OnlineRows surface
(exact_match/exact_match.pyi :120-171; exact_match/src/online.rs): a run's training stream (`tokens` in parts
`bounds`), when each position is trained (`spans` [m, 3]: (lo, hi, step), inputs [lo, hi) of `step`, hi its last
target), and per step the hint rows (train_hints.rs's: the deepest of `levels` whose context has a counted
occurrence; its cell, `entries` next tokens and weights) and count rows (train_counts.rs's: tot, dist, cnt of the own
next token) of the queries trained in that step. An occurrence (k tokens within a part and the token after them)
counts for a step-s query iff all its k + 1 tokens were trained before s (alpha = 1 + max tau <= s, online.rs:11-13);
a query's k-context must lie in its segment (segments start at each part's start and at every BOS).

`advance(step_hi, ...)` is the incremental path (online.rs :333): the GPU state (per level a context table with
totals, distinct counts and exact top-`entries` lists, and a split pair table) persists between calls; a step inserts
its newly available occurrences, then answers its queries (libngram_amd.so: ng_online_insert_levels, sort_pairs,
reduce_by_key, ng_online_top, ng_online_query_levels, ng_online_rows). `hints` / `counts` answer a step range from a fresh
state (counts alone need none: every step at once, online_counts.hip); with rule="segment" (the reference's
exactness-test rule) they answer every position from its segment's start, a step per segment."""

from __future__ import annotations

import ctypes

import numpy as np
import torch

from .lib import Lib, i32, u64


MAX_LAUNCH_LEVELS = 8  # levels per fused insert / query launch (ng_online_insert_levels, ng_online_query_levels)
REC_TOP, REC_CNT = 16, 2  # u32 words of a context's record with and without top entries (online.hip OREC_*)


def _ptr(t: torch.Tensor, at: int = 0) -> int:
    """The device address of element `at` of t."""
    return t.data_ptr() + at * t.element_size()


def _i64_array(rows) -> ctypes.Array:
    """Level rows of ints as one host int64 array (values of 2^63 and above wrap, as a u64 argument would)."""
    flat = [v - (1 << 64) if v >= 1 << 63 else v for row in rows for v in row]
    return (ctypes.c_int64 * len(flat))(*flat)

NONE = 0xFFFFFFFF
LOAD = 0.5
MAX_LEVEL = 64  # tokens of the longest context the kernels take


def loader_plan(ntok, nproc: int, BT: int, accum: int, steps: int) -> np.ndarray:
    """A training run's plan under llm.c's sequential loader (old_records/r001_llmc_c/llmc/hint_stats.cuh
    loader_plan :395-409): every rank's micro-batches, [m, 5] int64 rows (step, micro, rank, shard, offset), rank r's
    b-th micro-batch the inputs [offset, offset + BT) of its shard; a rank moves to the next shard once a shard's
    (ntok - 1) // (nproc * BT) samples are used. ValueError if the plan runs past the shards."""
    if nproc < 1 or BT < 1 or accum < 1 or steps < 0:
        raise ValueError(f"bad plan: nproc {nproc}, BT {BT}, accum {accum}, steps {steps}")
    plan = []
    for r in range(nproc):
        shard = sample = 0
        for b in range(steps * accum):
            if sample >= (int(ntok[shard]) - 1) // (nproc * BT):
                shard, sample = shard + 1, 0
                if shard >= len(ntok):
                    raise ValueError(f"the training plan runs past the {len(ntok)} shards")
            plan.append((b // accum, b % accum, r, shard, sample * nproc * BT + r * BT))
            sample += 1
    return np.array(plan, np.int64).reshape(-1, 5)


def plan_stream(ntok, plan: np.ndarray, BT: int) -> list[int]:
    """The training stream's parts for a plan (hint_stats.cuh train_plan :666-676): each shard the plan reads, up to
    its last trained target (shard 0 whole)."""
    nshards = int(plan[:, 3].max()) + 1 if len(plan) else 1
    sizes = [0] * nshards
    for _, _, _, shard, off in plan:
        sizes[shard] = max(sizes[shard], int(off) + BT + 1)
    sizes[0] = max(sizes[0], int(ntok[0]))
    return sizes


def plan_spans(plan: np.ndarray, sizes: list[int], BT: int) -> np.ndarray:
    """OnlineRows spans [m, 3] (lo, hi, step) of a plan over the stream of `sizes` parts: every micro-batch's inputs
    [lo, lo + BT) trained in its step, lo + BT its last target (hint_stats.cuh tr_spans_k :411-420)."""
    starts = np.concatenate([[0], np.cumsum(sizes)[:-1]]).astype(np.int64)
    lo = starts[plan[:, 3]] + plan[:, 4]
    return np.stack([lo, lo + BT, plan[:, 0]], axis=1).astype(np.int64)


def plan_rows(plan: np.ndarray, sizes: list[int], BT: int, accum: int, rank: int) -> np.ndarray:
    """The stream position of each of rank `rank`'s training rows, in training order: row (step * accum + micro) * BT
    + i is input i of that micro-batch (hint_stats.cuh's row_of :411-420). Gather a stream-sized output with it."""
    starts = np.concatenate([[0], np.cumsum(sizes)[:-1]]).astype(np.int64)
    mine = plan[plan[:, 2] == rank]
    rows = np.full(int(plan[:, 0].max() + 1) * accum * BT if len(plan) else 0, -1, np.int64)
    for step, micro, _, shard, off in mine:
        r0 = (int(step) * accum + int(micro)) * BT
        rows[r0 : r0 + BT] = starts[shard] + off + np.arange(BT)
    return rows


# A list's bounds are looked up for every step, one copy for all lists, where the steps are close together: fewer than this
# many, and at most two per span (and 1024) of which one is used. Elsewhere the steps in use are listed, each list read by
# itself. Looked up / listed, construction and prepare at four levels: 65536 positions, 1000 spans with steps below 1000
# 0.84 / 1.00 ms, below 4000 0.99 / 0.90, below 64000 4.9 / 0.9; 2^20 positions, 65536 spans 5.7 / 6.0.
STEP_TABLE = 1 << 20
# A stream of at least FEW_MIN positions of which fewer than one in FEW_SHARE are trained has its trained positions picked
# out before they are sorted, so that sorts, tables and kept lists are as long as they are, not as the stream is.
# Of 2^26 positions, all sorted / the trained ones: half trained, order 4.6 / 6.1 ms and counts of three levels 57 / 46; a
# quarter 4.6 / 4.9 and 42 / 24; 1 in 64 4.6 / 3.7 and 31 / 5.9, the prepared state 1552 / 544 MiB.
FEW_MIN, FEW_SHARE = 1 << 20, 4


class _Steps:
    """A list ordered by step, as its bounds: `steps` (ascending, int64) and where each of them begins; entries of a
    step that is not among them: none."""

    def __init__(self, steps: np.ndarray, begins: np.ndarray, total: int):
        self.steps = steps
        self.begins = np.append(begins, total)

    def before(self, s: int) -> int:
        """The entries of the steps before s."""
        return int(self.begins[np.searchsorted(self.steps, s, side="left")])

    def sizes(self) -> np.ndarray:
        return np.diff(self.begins)


class OnlineRows:
    """A run's training stream and when each of its positions is trained, for its online hint and count rows under
    the step rule, on the GPU (ValueError on bad tokens, bounds or spans, as online.rs new :118-181)."""

    def __init__(self, tokens, bounds: list[int], spans, threads: int = 1, cpus: list[int] = ()):
        tok = np.ascontiguousarray(tokens, dtype=np.uint16)
        n = len(tok)
        if n == 0 or n >= 1 << 30:
            raise ValueError(f"{n} tokens: need 1 to 2^30")
        bounds = [int(b) for b in bounds]
        if len(bounds) < 2 or bounds[0] != 0 or bounds[-1] != n or any(a >= b for a, b in zip(bounds, bounds[1:])):
            raise ValueError("bounds must ascend strictly from 0 to the token count")
        sp = np.asarray(spans, dtype=np.int64)
        if sp.ndim != 2 or sp.shape[1] != 3:
            raise ValueError("spans must be [m, 3]: (lo, hi, step)")
        if len(sp) and ((sp[:, 0] < 0).any() or (sp[:, 0] > sp[:, 1]).any() or (sp[:, 1] > n).any()
                        or (sp[:, 2] < 0).any() or (sp[:, 2] >= NONE).any()):
            raise ValueError("bad span")
        self.n = n
        self.bounds = bounds
        self.lib = Lib()
        dev = torch.device("cuda", torch.cuda.current_device())
        self.dev = dev
        self.tok = torch.from_numpy(tok.view(np.int16) if tok.flags.writeable else tok.view(np.int16).copy()).to(dev)
        # the first step training each position (as an input or a target; as an input), its segment and whether its next
        # token lies in its part, on the device (uint32 bits, NONE where no step does)
        self.bounds_dev = torch.tensor(bounds, dtype=torch.int64, device=dev)
        np_ = len(bounds) - 1
        offs = np.concatenate([[0], np.cumsum(sp[:, 1] - sp[:, 0])]).astype(np.int64)
        at = torch.from_numpy(np.concatenate([sp.reshape(-1), offs])).to(dev)
        self.tau = torch.empty(n, dtype=torch.int32, device=dev)
        self.tau_in = torch.empty(n, dtype=torch.int32, device=dev)
        self.lib("ng_online_tau", at, at[sp.size :], len(sp), int(offs[-1]), self.bounds_dev, np_, n, self.tau,
                 self.tau_in)
        self.max_step = int(sp[:, 2].max()) if len(sp) else -1
        self.max_steps = len(sp)  # at most this many steps are in use
        # at most how many positions have a step: of spans in order without overlap, theirs and each one's last target; else
        # counted once it is asked for (about 70 us)
        self._trained = min(n, int(offs[-1]) + len(sp)) if (sp[1:, 0] >= sp[:-1, 1]).all() else None
        seg = torch.empty(n, dtype=torch.int64, device=dev)
        self.has_next = torch.empty(n, dtype=torch.uint8, device=dev)
        self.lib("ng_online_layout", self.tok, n, self.bounds_dev, np_, seg, self.has_next)
        self.lib.cub("inclusive_max", seg, seg, n)
        self.avail = torch.empty(n, dtype=torch.int32, device=dev)
        self.lib("ng_online_avail", seg, n, self.avail)
        self._done = 0
        self.config = None
        self.state = None
        # a step's merge: "buckets" (ng_online_merge: no sort of the step's events, where its packed words hold the
        # step's occurrences) or "sorted" (sort_pairs + reduce_by_key + ng_online_top); both give the same state
        self.merge = "buckets"

    def __len__(self) -> int:
        return self.n

    @property
    def done(self) -> int:
        return self._done

    def prefault(self) -> None:
        torch.cuda.synchronize(self.dev)

    # -----------------------------------------------------------------------------------------------------------
    def _check_config(self, levels, buckets, entries, count_levels):
        levels, buckets, count_levels = list(levels), list(buckets), list(count_levels)
        if levels or entries:
            if entries < 1 or entries > 8 or not buckets or len(buckets) > 127 or buckets[0] < 1 or any(
                    a >= b for a, b in zip(buckets, buckets[1:])):
                raise ValueError(f"need 1 <= entries <= 8 and buckets ascending from 1: {entries}, {buckets}")
            if any(k not in buckets for k in levels) or any(a >= b for a, b in zip(levels, levels[1:])):
                raise ValueError(f"levels must ascend and be of {buckets}: {levels}")
        if any(k < 1 for k in count_levels):
            raise ValueError(f"levels must be >= 1: {count_levels}")
        return tuple(levels), tuple(buckets), int(entries), tuple(count_levels)

    def prepare(self, levels, buckets, entries, count_levels) -> None:
        """Before the clock: advance()'s GPU state for this configuration, and per level the occurrences ordered by the
        step they become available in (online.rs :320-331)."""
        cfg = self._check_config(levels, buckets, entries, count_levels)
        if self.config is not None:
            if self.config != cfg:
                raise ValueError("advance()'s configuration is fixed by its first call")
            return
        self.config = cfg
        self.state = self._new_state(cfg)

    def _new_state(self, cfg, taus=None) -> dict:
        """advance()'s state; taus: (tau, tau_in, the last step) in place of the spans' (the rule "segment"'s)."""
        levels, buckets, entries, count_levels = cfg
        dev = self.dev
        tau, tau_in, last = taus if taus is not None else (self.tau, self.tau_in, self.max_step)
        E = max(1, entries)
        st = {"levels": {}, "E": E}
        # queries: the positions trained as inputs, by step; and per level its occurrences (ending at g: tokens g-k+1..g
        # and next g+1 within g's part) by the step they count from, alpha = 1 + max tau over them
        ks = sorted(set(levels) | set(count_levels))
        orders = self._by_step([(tau_in, 0)] + [(tau, k) for k in ks], last + 1, taus is not None)
        st["q_pos"], st["q_step"] = orders[0]
        for k, (occ, alpha) in zip(ks, orders[1:]):
            m = int(occ.numel())
            cap = max(1 << 16, int(m / LOAD) + 1)
            # the pair table: 16-byte slots (key, count); a record per context: total, distinct count and, where the
            # level keeps hint rows, its top entries (REC_TOP u32 words: one 64-byte line), else REC_CNT words
            pt = torch.full((cap, 2), -1, dtype=torch.int64, device=dev)
            pt[:, 1] = 0
            rw = REC_TOP if k in levels else REC_CNT
            st["levels"][k] = {
                "occ": occ, "alpha": alpha,
                "ck": torch.full((cap,), -1, dtype=torch.int64, device=dev), "ccap": cap,
                "pt": pt, "pcap": cap, "rec": torch.zeros(cap * rw, dtype=torch.int32, device=dev), "rw": rw,
                "flags": torch.zeros(2, dtype=torch.int32, device=dev),
                "ctx_bits": max(1, (cap - 1).bit_length()),
            }
        # a step's events of every level go through one merge (ng_online_merge, or the sorted one), each level's pair
        # keys tagged with its index above the widest level's pair-key bits (ng_online_insert's tag, the merge's desc)
        st["tshift"] = 16 + max(lv["ctx_bits"] for lv in st["levels"].values())
        st["tag_bits"] = max(1, (len(st["levels"]) - 1).bit_length())
        if st["tshift"] + st["tag_bits"] > 64:
            raise ValueError("the online tables are too large for one step's tagged pair keys")
        desc = []
        for k, lv in st["levels"].items():
            desc += [lv["pt"].data_ptr(), lv["pcap"], lv["rec"].data_ptr(), int(lv["rw"] == REC_TOP),
                     lv["flags"].data_ptr()]
        st["top_desc"] = torch.tensor(desc, dtype=torch.int64, device=dev)
        most = max(1, self._most(lv["alpha"] for lv in st["levels"].values()))
        st["ev"] = torch.empty(most, dtype=torch.int64, device=dev)
        st["merge_temp"] = None
        if self.merge == "buckets":
            size = ctypes.c_size_t(0)
            try:
                self.lib("ng_online_merge", None, ctypes.c_void_p(ctypes.addressof(size)), None, most, None,
                         i32(len(st["levels"])), i32(st["tshift"]), i32(E))
            except RuntimeError:  # -1: the step is too large for the packed words; the sorted merge runs instead
                size = None
            if size is not None:
                st["merge_size"] = size
                st["merge_temp"] = torch.empty(max(1, size.value), dtype=torch.uint8, device=dev)
        if st["merge_temp"] is None:  # the sorted merge's buffers
            st["ev_sorted"] = torch.empty(most, dtype=torch.int64, device=dev)
            st["uk"] = torch.empty(most, dtype=torch.int64, device=dev)
            st["agg"] = torch.empty(most, dtype=torch.int32, device=dev)
            st["nruns"] = torch.zeros(1, dtype=torch.int64, device=dev)
            st["score"] = torch.empty(most, dtype=torch.int64, device=dev)
        nq = self._most([st["q_step"]])
        st["qslot"] = {k: torch.empty(max(1, nq), dtype=torch.int32, device=dev) for k in levels}
        st["hinted"] = torch.zeros(1, dtype=torch.int32, device=dev)
        st["done"] = 0
        if levels:  # ng_online_rows' per-level descriptors (deepest first): the same buffers every step
            desc = []
            for k in sorted(levels, reverse=True):
                lv = st["levels"][k]
                desc += [st["qslot"][k].data_ptr(), lv["rec"].data_ptr(), buckets.index(k)]
            st["rows_desc"] = torch.tensor(desc, dtype=torch.int64, device=dev)
        return st

    def _few(self, every: bool) -> bool:
        """Whether few of the stream's positions have a step (every: all of them do, the rule "segment")."""
        if every or self.n < FEW_MIN:
            return False
        if self._trained is None:
            self._trained = int((self.tau != -1).sum().item())
        return self._trained * FEW_SHARE < self.n

    def _by_step(self, lists: list, last: int, every: bool = False) -> list:
        """Per (tau, k) of `lists` the positions with a step, ordered by it and within a step by position (int32), and
        the steps' bounds (ng_online_order's steps, at most `last`; a stable sort by them). every: every position has a
        step, and every step is in use (the rule "segment")."""
        n, dev = self.n, self.dev
        bits = max(1, (last + 1).bit_length())
        none = (1 << bits) - 1  # above every step: the positions without one sort behind the others
        table = last < STEP_TABLE and (every or last <= 2 * self.max_steps + 1024)
        steps = torch.arange(last + 2, device=dev) if table else None
        few = self._few(every)
        key = torch.empty(n, dtype=torch.int64, device=dev)
        val = torch.empty(n, dtype=torch.int32, device=dev)
        key2 = None if few else torch.empty(n, dtype=torch.int64, device=dev)
        out, bounds = [], []
        for tau, k in lists:
            self.lib("ng_online_order", tau, n, self.bounds_dev, len(self.bounds) - 1, i32(k), u64(none), key, val)
            m, key1, val1 = n, key, val
            if few:
                val1 = torch.nonzero(key != none).squeeze(1)
                m, key1, val1 = val1.numel(), key[val1], val1.to(torch.int32)
                key2 = torch.empty(m, dtype=torch.int64, device=dev)
            order = torch.empty(m, dtype=torch.int32, device=dev)
            if m:
                self.lib.cub("sort_pairs", key1, key2, val1, order, m, i32(0), i32(bits))
            out.append(order)
            if table:
                bounds.append(torch.searchsorted(key2, steps))
            else:
                u, c = torch.unique_consecutive(key2, return_counts=True)
                u, c = u.cpu().numpy(), c.cpu().numpy()
                begins = np.cumsum(c) - c
                at = int(np.searchsorted(u, none))
                bounds.append(_Steps(u[:at], begins[:at], int(begins[at]) if at < len(u) else m))
        if table:
            host = torch.stack(bounds).cpu().numpy()  # one read for every list
            bounds = [_Steps(np.arange(last + 1), h[:-1], int(h[-1])) for h in host]
        return [(order[: int(b.begins[-1])], b) for order, b in zip(out, bounds)]

    @staticmethod
    def _most(lists) -> int:
        """The most entries one step has in all of `lists` together."""
        lists = list(lists)
        steps = np.unique(np.concatenate([b.steps for b in lists])) if lists else np.zeros(0, np.int64)
        total = np.zeros(len(steps), np.int64)
        for b in lists:
            total[np.searchsorted(steps, b.steps)] += b.sizes()
        return int(total.max()) if len(total) else 0

    def _range(self, steps: _Steps, lo: int, hi: int) -> tuple[int, int]:
        return steps.before(lo), steps.before(hi)

    def _step(self, st: dict, s: int, outs: dict, queries: bool = True) -> None:
        """Step s: its newly available occurrences inserted at every level, then (queries) its queries answered."""
        lib = self.lib
        levels, buckets, entries, count_levels = outs["cfg"]
        E = st["E"]
        m = 0
        ins = []
        for t, (k, lv) in enumerate(st["levels"].items()):
            a, b = self._range(lv["alpha"], s, s + 1)
            if b == a:
                continue
            # the pair counts and the contexts' records are updated per distinct pair and per context by the step's
            # merge, not per occurrence: no global atomic per occurrence, no chains of same-address atomics on hot
            # contexts
            ins.append((_ptr(lv["occ"], a), b - a, k, _ptr(lv["ck"]), lv["ccap"], _ptr(lv["pt"]), lv["pcap"],
                        _ptr(st["ev"], m), _ptr(lv["flags"]), t << st["tshift"]))
            m += b - a
        for j in range(0, len(ins), MAX_LAUNCH_LEVELS):  # every level's inserts in one launch
            part = ins[j : j + MAX_LAUNCH_LEVELS]
            lib("ng_online_insert_levels", self.tok, i32(len(part)), _i64_array(part), i32(0))
        if m and st["merge_temp"] is not None:
            lib("ng_online_merge", st["merge_temp"], ctypes.c_void_p(ctypes.addressof(st["merge_size"])), st["ev"], m,
                st["top_desc"], i32(len(st["levels"])), i32(st["tshift"]), i32(E))
        elif m:
            lib.cub("sort_pairs", st["ev"], st["ev_sorted"], None, None, m, i32(0), i32(st["tshift"] + st["tag_bits"]))
            lib.cub("reduce_by_key", st["ev_sorted"], st["uk"], None, st["agg"], st["nruns"], m)  # run lengths
            lib("ng_online_top", st["uk"], st["nruns"], m, st["agg"], st["top_desc"], i32(len(st["levels"])),
                i32(st["tshift"]), st["score"], i32(E), i32(1))
        qa, qb = self._range(st["q_step"], s, s + 1)
        mq = qb - qa
        if mq == 0 or not queries:
            return
        qpos = st["q_pos"][qa:qb]
        qry = []
        nc = len(count_levels)
        for k in list(count_levels) + [k for k in levels if k not in count_levels]:
            lv = st["levels"][k]
            ci = count_levels.index(k) if k in count_levels else -1
            qry.append((k, _ptr(lv["ck"]), lv["ccap"], _ptr(lv["pt"]), lv["pcap"], _ptr(lv["rec"]), lv["rw"],
                        _ptr(st["qslot"][k]) if k in levels else 0,
                        _ptr(outs["tot"]) if ci >= 0 else 0, _ptr(outs["dist"]) if ci >= 0 else 0,
                        _ptr(outs["cnt"]) if ci >= 0 else 0, nc if ci >= 0 else 1, max(ci, 0)))
        for j in range(0, len(qry), MAX_LAUNCH_LEVELS):  # every level's queries in one launch
            part = qry[j : j + MAX_LAUNCH_LEVELS]
            lib("ng_online_query_levels", self.tok, self.avail, self.has_next, qpos, mq, i32(len(part)),
                _i64_array(part))
        if levels:
            lib("ng_online_rows", qpos, mq, i32(len(levels)), st["rows_desc"], i32(E), i32(outs["slots"]), outs["cell"],
                outs["next"], outs["weights"], outs["level"], st["hinted"])

    def _device_outputs(self, cfg, slots: int = 1, with_level: bool = False) -> dict:
        """Stream-sized outputs: hint rows in `slots` slots per position (cell [n, slots], next / weights [n, slots,
        entries], with_level the slots' bucket indices, -1 where empty) and count rows [n, len(count_levels)]."""
        levels, buckets, entries, count_levels = cfg
        n, dev = self.n, self.dev
        E = max(1, entries)
        return {"cfg": cfg, "slots": slots,
                "cell": torch.zeros((n, slots) if slots > 1 else n, dtype=torch.int16, device=dev),
                "next": torch.zeros((n, slots, E) if slots > 1 else (n, E), dtype=torch.int16, device=dev),
                "weights": torch.zeros((n, slots, E) if slots > 1 else (n, E), dtype=torch.int16, device=dev),
                "level": torch.full((n, slots), -1, dtype=torch.int8, device=dev) if with_level else None,
                "tot": torch.zeros((n, max(1, len(count_levels))), dtype=torch.int32, device=dev),
                "dist": torch.zeros((n, max(1, len(count_levels))), dtype=torch.int16, device=dev),
                "cnt": torch.zeros((n, max(1, len(count_levels))), dtype=torch.int32, device=dev)}

    def _check_flags(self, st) -> None:
        for k, lv in st["levels"].items():
            f = int(lv["flags"][0].item())
            if f & 4:
                raise RuntimeError(f"k={k}: a step's merge bucket needed more hash splits than the merge takes")
            if f:
                raise RuntimeError(f"k={k}: a table of the online state overflowed")

    @staticmethod
    def _copy_rows(outs: dict, rows: torch.Tensor, cell, nxt, weights, tot, dist, cnt) -> None:
        """The rows of `rows` (positions) from the device outputs into the caller's host arrays."""
        r = rows.long()
        rn = r.cpu().numpy()
        if cell is not None:
            cell[rn] = outs["cell"][r].cpu().numpy()
            nxt[rn] = outs["next"][r].cpu().numpy().view(np.uint16)
            weights[rn] = outs["weights"][r].cpu().numpy().view(np.uint16)
        if tot is not None:
            nc = tot.shape[1]
            tot[rn] = outs["tot"][r, :nc].cpu().numpy().view(np.uint32)
            dist[rn] = outs["dist"][r, :nc].cpu().numpy().view(np.uint16)
            cnt[rn] = outs["cnt"][r, :nc].cpu().numpy().view(np.uint32)

    def advance(self, step_hi: int, levels, buckets, entries: int, count_levels, cell=None, next=None, weights=None,
                tot=None, dist=None, cnt=None) -> int:
        """The rows of the queries trained in steps [done, step_hi) (what hints + counts write, rule "step"), with the
        counted occurrences kept between calls; returns the queries hinted (online.rs :333)."""
        self.prepare(levels, buckets, entries, count_levels)
        st = self.state
        if step_hi < self._done or step_hi >= 1 << 30:
            raise ValueError(f"bad step range [{self._done}, {step_hi})")
        if "outs" not in st:
            st["outs"] = self._device_outputs(self.config)
        outs = st["outs"]
        st["hinted"].zero_()
        for s in range(self._done, step_hi):
            self._step(st, s, outs)
        self._check_flags(st)
        qa, qb = self._range(st["q_step"], self._done, step_hi)
        if cell is not None or tot is not None:
            self._copy_rows(outs, st["q_pos"][qa:qb], cell, next, weights, tot, dist, cnt)
        self._done = step_hi
        return int(st["hinted"].item())

    def advance_device(self, step_hi: int) -> None:
        """advance() to step_hi with the prepared configuration, leaving the rows in GPU memory (self.state["outs"]),
        without synchronizing."""
        st = self.state
        if "outs" not in st:
            st["outs"] = self._device_outputs(self.config)
        outs = st["outs"]
        for s in range(self._done, step_hi):
            self._step(st, s, outs)
        self._done = step_hi

    def _rule(self, rule: str, step_lo: int, step_hi: int) -> tuple:
        """(tau, tau_in, the last step), or None for the spans', and the step range of a rule."""
        taus = None
        if rule == "segment":
            seg = (torch.cumsum(self.avail == 1, 0) - 1).to(torch.int32)  # a segment starts where avail is 1
            last = int(seg[-1].item())
            taus = (seg, seg, last)
            step_lo, step_hi = 0, last + 1
        elif rule != "step":
            raise ValueError(f"rule must be 'step' or 'segment': {rule}")
        if step_lo > step_hi or step_hi >= 1 << 30:
            raise ValueError(f"bad step range [{step_lo}, {step_hi})")
        return taus, step_lo, step_hi

    def _range_counts(self, count_levels, step_lo, step_hi, rule):
        """The count rows of the queries of [step_lo, step_hi) (outputs and positions as _range_rows'), every step at once:
        per level its occurrences in step order, inserted once, sorted by pair and by context, and each query a few
        searches (ng_online_occ_insert / _index / _query). The same counts as a fresh state advanced step by step,
        without its launches and merges per step."""
        taus, step_lo, step_hi = self._rule(rule, step_lo, step_hi)
        cfg = self._check_config((), (1,), 0, count_levels)
        if not cfg[3]:
            raise ValueError("need count levels")
        tau, tau_in, last = taus if taus is not None else (self.tau, self.tau_in, self.max_step)
        n, dev, lib = self.n, self.dev, self.lib
        outs = self._device_outputs(cfg)
        if rule == "segment":  # every position is a query
            qpos, mq = None, n
            rows = torch.arange(n, dtype=torch.int32, device=dev)
        else:
            order, steps = self._by_step([(tau_in, 0)], last + 1)[0]
            qa, qb = self._range(steps, step_lo, step_hi)
            rows = qpos = order[qa:qb]
            mq = qb - qa
        if mq == 0:
            return outs, rows
        nc = len(count_levels)
        if max(count_levels) > MAX_LEVEL:
            raise RuntimeError(f"k={max(count_levels)}: a context has at most {MAX_LEVEL} tokens")
        bits = max(1, (last + 2).bit_length())
        none = (1 << bits) - 1
        few = self._few(rule == "segment")
        most = max(1, self._trained) if few else n  # a level's occurrences end at trained positions
        cap = max(1 << 16, int(most / LOAD) + 1)
        cbits = cap.bit_length()
        u64s = [torch.empty(most, dtype=torch.int64, device=dev) for _ in range(4)]
        u32s = [torch.empty(most, dtype=torch.int32, device=dev) for _ in range(4)]
        # the steps of the whole stream, of which the occurrences are picked out where they are few
        order = (torch.empty(n, dtype=torch.int64, device=dev), torch.empty(n, dtype=torch.int32, device=dev)) \
            if few else (u64s[0], u32s[0])
        ck = torch.empty(cap, dtype=torch.int64, device=dev)
        bounds = torch.empty((cap, 2), dtype=torch.int32, device=dev)
        first = torch.empty(most, dtype=torch.uint8, device=dev)
        pre = torch.empty(most + 1, dtype=torch.int32, device=dev)
        flags = torch.zeros((len(set(count_levels)), 2), dtype=torch.int32, device=dev)
        ks = sorted(set(count_levels))
        for k, flag in zip(ks, flags):
            (key, ka, kb, akey), (val, va, vb, occ) = u64s, u32s
            lib("ng_online_order", tau, n, self.bounds_dev, len(self.bounds) - 1, i32(k), u64(none), *order)
            m, step_of, at = n, *order
            if few:
                at = torch.nonzero(step_of != none).squeeze(1)
                m, step_of, at = at.numel(), step_of[at], at.to(torch.int32)
            if m == 0:
                continue
            lib.cub("sort_pairs", step_of, akey, at, occ, m, i32(0), i32(bits))
            lib.fill(ck, -1)
            lib("ng_online_occ_insert", self.tok, occ, akey, u64(none), m, i32(k), ck, u64(cap), i32(cbits), key, val,
                flag)
            lib.cub("sort_pairs", key, ka, val, va, m, i32(0), i32(16 + cbits))
            lib.cub("sort_pairs", key, kb, val, vb, m, i32(16), i32(16 + cbits))
            lib.cub("ng_online_occ_index", ka, va, kb, vb, m, i32(cbits), first, pre, bounds)
            lib("ng_online_occ_query", self.tok, self.avail, self.has_next, qpos, mq, tau_in, akey, m, i32(k), ck,
                u64(cap), bounds, vb, pre, ka, va, outs["tot"], outs["dist"], outs["cnt"], i32(nc),
                i32(count_levels.index(k)))
        for k, f in zip(ks, flags[:, 0].cpu().tolist()):
            if f:
                raise RuntimeError(f"k={k}: a table of the online state overflowed")
        return outs, rows

    def _range_rows(self, levels, buckets, entries, count_levels, step_lo, step_hi, rule, slots: int = 1,
                    with_level: bool = False):
        """A fresh state advanced over steps [0, step_hi), the queries of [step_lo, step_hi) answered. The rule
        "segment" (online.rs:14-17: every position a query at its segment's start, an occurrence counted iff its next
        token lies before that start) is the step rule with one step per segment in stream order: tau = tau_in = the
        position's segment index makes an occurrence's alpha 1 + the segment of its next token, so it counts for a
        query exactly when that segment lies before the query's; every step then runs as advance()'s do."""
        taus, step_lo, step_hi = self._rule(rule, step_lo, step_hi)
        cfg = self._check_config(levels, buckets, entries, count_levels)
        st = self._new_state(cfg, taus)
        outs = self._device_outputs(cfg, slots, with_level)
        for s in range(0, step_hi):  # earlier steps only insert their occurrences
            self._step(st, s, outs, queries=s >= step_lo)
        self._check_flags(st)
        qa, qb = self._range(st["q_step"], step_lo, step_hi)
        return st, outs, st["q_pos"][qa:qb]

    def segment_rows(self, levels, buckets, entries: int, slots: int = 1):
        """Every position's hint under the rule "segment" in `slots` slots, deepest levels first (train_hints.rs's
        rows of the stream: cell int16, next and weights uint16 [.., entries], level int8, -1 for an empty slot;
        [n] / [n, entries] with one slot, else [n, slots] / [n, slots, entries])."""
        st, outs, _ = self._range_rows(levels, buckets, entries, (), 0, 0, "segment", slots, True)
        lvl = outs["level"]
        return (outs["cell"].cpu().numpy(), outs["next"].cpu().numpy().view(np.uint16),
                outs["weights"].cpu().numpy().view(np.uint16), (lvl[:, 0] if slots == 1 else lvl).cpu().numpy())

    def segment_counts(self, levels):
        """Every position's count rows under the rule "segment" (train_counts.rs's): tot uint32, dist uint16, cnt
        uint32 [n, len(levels)]."""
        outs, _ = self._range_counts(list(levels), 0, 0, "segment")
        return (outs["tot"].cpu().numpy().view(np.uint32), outs["dist"].cpu().numpy().view(np.uint16),
                outs["cnt"].cpu().numpy().view(np.uint32))

    def hints(self, levels, buckets, entries, step_lo, step_hi, cell, next, weights, rule: str = "step") -> int:
        """The hint rows of the queries trained in steps [step_lo, step_hi), written into the stream-sized cell [n],
        next / weights [n, entries]; returns the queries hinted (online.rs :190)."""
        if entries < 1:
            raise ValueError("need entries >= 1")
        if len(cell) != self.n or next.shape != (self.n, entries) or weights.shape != (self.n, entries):
            raise ValueError(f"outputs must be [{self.n}] and [{self.n}, {entries}]")
        st, outs, rows = self._range_rows(levels, buckets, entries, (), step_lo, step_hi, rule)
        self._copy_rows(outs, rows, cell, next, weights, None, None, None)
        return int(st["hinted"].item())

    def counts(self, levels, step_lo, step_hi, tot, dist, cnt, rule: str = "step") -> None:
        """The count rows of the queries trained in steps [step_lo, step_hi) at each level, written into the
        stream-sized tot / dist / cnt [n, L] (online.rs :259)."""
        nl = len(levels)
        if not nl or min(levels) < 1:
            raise ValueError(f"levels must be >= 1: {levels}")
        if tot.shape != (self.n, nl) or dist.shape != (self.n, nl) or cnt.shape != (self.n, nl):
            raise ValueError(f"outputs must be [{self.n}, {nl}]")
        outs, rows = self._range_counts(list(levels), step_lo, step_hi, rule)
        self._copy_rows(outs, rows, None, None, None, tot, dist, cnt)
