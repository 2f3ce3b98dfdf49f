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
