"""GPU: the longest match's deep levels (ng_lm_levels) on candidate lists that a block walks in many rounds, against a
restatement with Python sets: with a grid of 1 to 7 blocks a block takes up to twenty rounds of 1024 positions and gives
out its staged hits several times; lists around a round and around the stage, mostly hits and mostly misses, with and
without level cap tried first."""

import numpy as np
import pytest
import torch

from ngram_amd.lib import Lib, i32, u64

pytestmark = pytest.mark.gpu

K0, CAP = 2, 6
SENT = 0xFFFF


def _restated(tok, x, avail, act, cand, first):
    """(hit positions per level, lengths, [kept, matched] per level, the trial's [going on, matched]) of levels
    K0..CAP."""
    text, query = tok.astype(">u2").tobytes(), x.astype(">u2").tobytes()

    def scan(k, act, cand):
        ctx = {i: query[2 * (i - k + 1) : 2 * (i + 1)] for i in act if avail[i] >= k}
        wanted = set(ctx.values())
        hits = [p for p in cand if p >= k and tok[p] != SENT and text[2 * (p - k) : 2 * p] in wanted]
        seen = {text[2 * (p - k) : 2 * p] for p in hits}
        return hits, [i for i in act if ctx.get(i) in seen]

    length = np.zeros(len(x), np.int32)
    hits, rows, trial = {}, {}, None
    if first:
        hits[CAP], matched = scan(CAP, act, cand)
        length[matched] = CAP
        act = sorted(set(act) - set(matched))
        trial = (len(act), len(matched))
    for k in range(K0, CAP if first else CAP + 1):
        cand, matched = scan(k, act, cand)
        length[matched] = k
        hits[k] = cand
        act = [i for i in matched if avail[i] >= k + 1]
        rows[k] = (len(act), len(matched))
    return hits, length, rows, trial


@pytest.mark.parametrize("n_cand", [1, 1023, 1025, 4097, 20_000])
@pytest.mark.parametrize("grid", [1, 2, 7])
@pytest.mark.parametrize("n_query", [3, 2500])  # of 3^6 contexts: mostly misses, mostly hits
@pytest.mark.parametrize("first", [0, 1])
def test_deep_levels_with_many_rounds_a_block(gpu, n_cand, grid, n_query, first):
    rng = np.random.default_rng(n_cand + 31 * grid + n_query)
    L = 32 * 1000
    tok = rng.integers(0, 3, L).astype(np.uint16)
    tok[rng.random(L) < 0.002] = SENT
    x = rng.integers(0, 3, n_query + CAP).astype(np.uint16)
    avail = np.minimum(np.arange(len(x)) + 1, 40).astype(np.int32)
    avail[rng.random(len(x)) < 0.1] = K0  # some end before the cap
    avail[:K0] = 1
    act = np.flatnonzero(avail >= K0).astype(np.int32)
    cand = np.sort(rng.choice(np.arange(L), n_cand, replace=False)).astype(np.int64)
    hits, length, rows, trial = _restated(tok, x, avail, act.tolist(), cand.tolist(), first)

    lib, dev = Lib(), torch.device("cuda")
    put = lambda a: torch.from_numpy(a).to(dev)  # noqa: E731
    n0, nlev = len(act), CAP - K0 + 1
    qcap = 2 * n0 + 1024
    slots = qcap + 1024
    table = lib.full_ones(slots, torch.int64, dev)
    rep = torch.empty(slots, dtype=torch.int32, device=dev)
    lvl = torch.zeros(slots, dtype=torch.uint8, device=dev)
    act_a, act_b, ctx_of = (torch.empty(n0, dtype=torch.int32, device=dev) for _ in range(3))
    hl = torch.full((nlev, n_cand), -1, dtype=torch.int64, device=dev)
    got_len = torch.zeros(len(x), dtype=torch.int32, device=dev)
    meta = torch.zeros((nlev + 1, 6), dtype=torch.int64, device=dev)
    flags = torch.zeros(2, dtype=torch.int32, device=dev)
    lib("ng_lm_levels", put(tok.view(np.int16)), put(x.view(np.int16)), put(avail), i32(K0), i32(CAP), i32(first),
        put(act), n0, act_a, act_b, put(cand), n_cand, table, u64(qcap), u64(slots), rep, ctx_of, lvl, hl, got_len, meta,
        flags, i32(grid))
    m, lists = meta.cpu().numpy(), hl.cpu().numpy()
    assert np.array_equal(got_len.cpu().numpy(), length)
    assert (m[:nlev, 4:] == 0).all() and not flags.any() and bool((table == -1).all())
    for k in range(K0, CAP + 1):
        n = int(m[k - K0, 2])
        assert sorted(lists[k - K0, :n].tolist()) == sorted(hits[k]), f"k={k}"
        assert (lists[k - K0, n:] == -1).all()
        if k in rows:
            assert tuple(m[k - K0, :2]) == rows[k], f"k={k}"
    if first:
        assert tuple(m[nlev, :2]) == trial
    if n_query == 2500 and n_cand == 20_000 and grid == 1:
        assert len(hits[K0 if not first else CAP]) > 4 * 4096  # several flushes of the stage


@pytest.mark.parametrize("k", [3, 6])
@pytest.mark.parametrize("n_dev", [0, 1, 700, 1900])
def test_one_level_by_device_side_counts(gpu, k, n_dev):
    """ng_query_index_dev, ng_scan_list_dev and ng_act_split over the first n_dev entries of their lists (their number
    on the device): the contexts' hit bits, the hit positions, and the entries without a hit, against Python sets."""
    rng = np.random.default_rng(10 * k + n_dev)
    L, N, g = 32 * 200, 2000, 3
    tok = rng.integers(0, 4, L).astype(np.uint16)
    x = rng.integers(0, 4, N).astype(np.uint16)
    avail = np.minimum(np.arange(N) + 1, rng.integers(1, 20, N)).astype(np.int32)
    act = rng.permutation(N).astype(np.int32)[:1900]
    cand = np.sort(rng.choice(L, 1900, replace=False)).astype(np.int64)
    text, query = tok.astype(">u2").tobytes(), x.astype(">u2").tobytes()
    ctx = {int(i): query[2 * (i - k + 1) : 2 * (i + 1)] for i in act[:n_dev] if avail[i] >= k}
    hits = [int(p) for p in cand[:n_dev] if p >= k and text[2 * (p - k) : 2 * p] in set(ctx.values())]
    seen = {text[2 * (p - k) : 2 * p] for p in hits}
    done = {i for i, c in ctx.items() if c in seen}

    lib, dev = Lib(), torch.device("cuda")
    put = lambda a: torch.from_numpy(a).to(dev)  # noqa: E731
    slots, qcap = 8192, 7168
    d_tok, d_x, d_act, d_cand = put(tok.view(np.int16)), put(x.view(np.int16)), put(act), put(cand)
    d_n = torch.tensor([n_dev], dtype=torch.int64, device=dev)
    table = torch.empty(slots, dtype=torch.int64, device=dev)
    rep, hit = torch.empty(slots, dtype=torch.int32, device=dev), torch.zeros(slots // 32, dtype=torch.int32, device=dev)
    ctx_of, out = (torch.full((1900,), -7, dtype=torch.int32, device=dev) for _ in range(2))
    length, flags = torch.zeros(N, dtype=torch.int32, device=dev), torch.zeros(2, dtype=torch.int32, device=dev)
    counters, n_out, matched = (torch.zeros(3, dtype=torch.int64, device=dev) for _ in range(3))
    lib("ng_query_index_dev", d_x, put(avail), d_act, d_n, 1900, i32(k), table, u64(qcap), u64(slots), rep, ctx_of,
        counters)
    R = 768  # 3 blocks, 256 positions a round
    ev, ev_count = torch.empty(g * R, dtype=torch.int64, device=dev), torch.zeros(g, dtype=torch.int32, device=dev)
    lib("ng_scan_list_dev", d_tok, i32(k), d_cand, d_n, 1900, table, u64(qcap), rep, d_x, hit, i32(1), ev, u64(R), ev_count,
        flags, i32(g), u64(0))
    lib("ng_act_split", d_act, d_n, 1900, ctx_of, hit, i32(k), length, out, n_out, matched)
    assert not counters[1:].any() and not flags.any()
    assert (ctx_of[n_dev:] == -7).all()
    got = np.concatenate([ev[b * R : b * R + int(c)].cpu().numpy() for b, c in enumerate(ev_count.tolist())])
    assert sorted(got.tolist()) == hits
    assert set(np.flatnonzero(length.cpu().numpy())) == done and int(matched[0]) == len(done)
    left = out[: int(n_out[0])].tolist()
    assert sorted(left) == sorted(set(act[:n_dev].tolist()) - done)
