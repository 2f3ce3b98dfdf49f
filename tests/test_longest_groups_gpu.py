"""GPU: the longest match on small streams against the oracle: few and many tokens (dense levels that turn sparse at
once, or never), positions left out by a mask, sizes around a block of the list kernels, levels counted together, one by
one and by the 64-bit count, index sizes learnt from another stream, and deep levels with and without the round at the
cap."""

import numpy as np
import pytest
import torch

import oracle as O
from ngram_amd import longest as LG
from ngram_amd.data import device_tokens
from ngram_amd.lib import Lib

pytestmark = pytest.mark.gpu


def _streams(n_train, n_query, vocab, seed):
    """Two shards, and queries half of which are spans of them."""
    rng = np.random.default_rng(seed)
    train = rng.integers(0, vocab, n_train).astype(np.uint16)
    train[rng.random(n_train) < 0.01] = O.BOS
    q = rng.integers(0, vocab, n_query).astype(np.uint16)
    for at in range(0, n_query - 1, 140):
        m = min(int(rng.integers(1, 100)), n_query - at, n_train)
        src = int(rng.integers(0, n_train - m + 1))
        q[at : at + m] = train[src : src + m]
    cut = n_train // 3
    return train, np.array([0, cut, n_train], np.int64), q


@pytest.mark.parametrize("n_train,n_query,vocab", [(40, 1, 3), (700, 255, 2), (5000, 1025, 40), (30000, 4097, 300),
                                                   (200_000, 9000, 50000), (60000, 3000, 1)])
@pytest.mark.parametrize("cap,mask", [(1, "none"), (2, "third"), (9, "none"), (64, "none"), (64, "third"),
                                      (64, "nothing")])
@pytest.mark.parametrize("how", ["together", "one by one", "64-bit"])
def test_longest_match_on_small_streams(gpu, n_train, n_query, vocab, cap, mask, how, monkeypatch):
    monkeypatch.setattr(LG, "_WIDE", set())
    if how == "one by one":
        monkeypatch.setattr(LG, "GROUP_EVENTS", 0)
    if how == "64-bit":
        monkeypatch.setattr(LG, "W_MAX", 0)
    train, bounds, x = _streams(n_train, n_query, vocab, n_train + cap)
    avail = O.segments(x)
    tok, _, _, _ = device_tokens([train[a:b] for a, b in zip(bounds, bounds[1:])])
    xt = torch.from_numpy(x.view(np.int16)).cuda()
    asked = np.ones(n_query, bool)
    if mask != "none":
        asked[:] = False
        if mask == "third":
            asked[::3] = True
    want = [np.where(asked, w, 0) for w in O.longest_match(train, bounds, x, avail, cap)[:3]]
    query = None if mask == "none" else torch.from_numpy(asked).cuda()
    for _ in range(2):  # a call whose sizes are another stream's, then its own
        length, nxt, cnt, ladder = LG.longest_match(tok, xt, LG._segments(xt, Lib()), cap, query=query)
        assert np.array_equal(length.cpu().numpy().view(np.uint32), want[0])
        assert np.array_equal(nxt.cpu().numpy().view(np.uint16), want[1])
        assert np.array_equal(cnt.cpu().numpy().view(np.uint32), want[2])
        for k, eligible, matched in ladder:
            assert matched == int((want[0] >= k).sum()) and eligible == int((asked & (avail >= k)).sum())
        assert len(ladder) >= int(want[0].max())


@pytest.mark.parametrize("overflows", [(1,), (3,), ("lists",), (2, "lists"), "together"])
def test_a_group_that_overflows_marks_only_the_levels_that_do(gpu, overflows, monkeypatch):
    """Levels counted together whose count reports a full escape table (forced here on counts that hold a given level, or
    on counts of several levels): each is counted again by itself, and only one that overflows alone takes the 64-bit
    count from then on."""
    monkeypatch.setattr(LG, "_WIDE", set())
    groups, count_group, count32 = [], LG._count_group, LG.count32

    def grouped(*args):
        groups.append([k for k, _, _ in args[6]])
        return count_group(*args)

    def counted(*args, **kw):
        c = count32(*args, **kw)
        if len(groups[-1]) > 1 if overflows == "together" else set(overflows) & set(groups[-1]):
            c.stat[2] = 2
        return c

    monkeypatch.setattr(LG, "_count_group", grouped)
    monkeypatch.setattr(LG, "count32", counted)
    train, bounds, x = _streams(30000, 4097, 300, 11)
    tok, _, _, _ = device_tokens([train[a:b] for a, b in zip(bounds, bounds[1:])])
    xt = torch.from_numpy(x.view(np.int16)).cuda()
    want = O.longest_match(train, bounds, x, O.segments(x), 64)
    for _ in range(2):
        length, nxt, cnt, _ = LG.longest_match(tok, xt, LG._segments(xt, Lib()), 64)
        assert np.array_equal(length.cpu().numpy().view(np.uint32), want[0])
        assert np.array_equal(nxt.cpu().numpy().view(np.uint16), want[1])
        assert np.array_equal(cnt.cpu().numpy().view(np.uint32), want[2])
    ks = {k for g in groups for k in g}
    assert "lists" in ks and len(ks) > 2 and len(groups[0]) > 1
    assert LG._WIDE == (set() if overflows == "together" else set(overflows) & ks)
    assert LG._WIDE or overflows == "together"


def test_list_levels_past_one_batch_are_counted_in_batches(gpu, monkeypatch):
    """List levels of more positions than a batch takes are not counted at once: their count's buffers would grow with
    the number of levels, and past 2^32 positions its offsets would wrap."""
    batches, count_batch, lists_emit = [], LG._count_batch, []

    def batched(*args):
        batches.append([args[7][k - 1][2] for k, _, _ in args[6]])
        return count_batch(*args)

    class Watched(Lib):
        def __call__(self, name, *args):
            if name == "ng_lm_lists_emit":
                lists_emit.append(name)
            return super().__call__(name, *args)

    train, bounds, x = _streams(30000, 4097, 300, 12)
    tok, _, _, _ = device_tokens([train[a:b] for a, b in zip(bounds, bounds[1:])])
    xt = torch.from_numpy(x.view(np.int16)).cuda()
    want = O.longest_match(train, bounds, x, O.segments(x), 64)
    monkeypatch.setattr(LG, "_WIDE", set())
    monkeypatch.setattr(LG, "_count_batch", batched)
    for limit in (1 << 28, 200):
        monkeypatch.setattr(LG, "BATCH_EVENTS", limit)
        batches.clear(), lists_emit.clear()
        length, nxt, cnt, _ = LG.longest_match(tok, xt, LG._segments(xt, Lib()), 64, elib=Watched())
        assert np.array_equal(length.cpu().numpy().view(np.uint32), want[0])
        assert np.array_equal(nxt.cpu().numpy().view(np.uint16), want[1])
        assert np.array_equal(cnt.cpu().numpy().view(np.uint32), want[2])
        assert (len(lists_emit), len(batches) > 1) == ((1, False) if limit > 200 else (0, True))
    assert all(sum(b[:-1]) < 200 for b in batches) and sum(map(sum, batches)) > 200 and not LG._WIDE
