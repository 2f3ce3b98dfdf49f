"""GPU: the TOP rule (a target's count only where it ranks among its context's cnt_top most frequent next tokens) on
the 32-bit count, against the oracle, and the same build on the 64-bit count: thresholds so low that many contexts
have one, partitions overfull, and levels of few positions."""

import numpy as np
import pytest

import oracle as O
from ngram_amd import counts as C
from ngram_amd import data
from ngram_amd import levels as levels_mod
from ngram_amd import partcount as P

pytestmark = pytest.mark.gpu

LEVELS = (1, 2, 3, 8)


@pytest.fixture(scope="module")
def corpus():
    return data.make_corpus("c3", train_tokens=300_000, query_tokens=30_001, shard_tokens=130_000)


@pytest.mark.parametrize("cnt_top", [1, 4, 1024])
@pytest.mark.parametrize("mode", ["plain", "regroup", "escape", "64-bit"])
def test_top_rule_matches_oracle(corpus, cnt_top, mode, monkeypatch):
    if mode == "regroup":  # partitions overfull at 256 distinct pairs: counted again with a bit more
        monkeypatch.setattr(P, "P32_LIMIT", 256)
    if mode == "escape":  # an 8-bit count field: larger counts in the escape table
        monkeypatch.setattr(P, "PACK32_MIN_BITS", 40)
    if mode == "64-bit":
        monkeypatch.setattr(levels_mod, "W_MAX", 0)
    tok, sizes, starts, _ = data.device_tokens(corpus.shards())
    eng = levels_mod.LevelBuild(tok, sizes, starts, LEVELS)
    x, tgt, avail = C.queries(corpus.query, [], "cuda")
    for _ in range(2):  # a build that has learnt nothing, then one with the sizes it found
        res = eng.build(x, tgt, avail, cnt_top=cnt_top, keep=(2, 8), with_mask=True)
        out = res.counts.cpu().numpy()
        mask = np.zeros(x.numel(), np.int32)
        for li, k in enumerate(LEVELS):
            o = O.query_counts(corpus.train, corpus.bounds, corpus.query[:-1], corpus.query[1:],
                               O.segments(corpus.query[:-1]), k, cnt_top=cnt_top)
            assert np.array_equal(out[0, li].view(np.uint32), o["tot"]), f"tot k={k}"
            assert np.array_equal(out[1, li], o["dist"].astype(np.int32)), f"dist k={k}"
            assert np.array_equal(out[2, li].view(np.uint32), o["cnt"]), f"cnt k={k}"
            mask |= (o["tot"] > 0).astype(np.int32) << li
        assert np.array_equal(res.mask.cpu().numpy(), mask)
    assert set(res.kept) == {2, 8}
    assert (out[1, 1] > 4).any() and (mode == "64-bit" or not eng.wide)


@pytest.mark.parametrize("cnt_top", [None, 4])
def test_position_list_that_outgrows_its_room_on_the_64_bit_count(corpus, cnt_top, monkeypatch):
    """A later build whose levels have far more positions with an occurred context than the last one's, but no more
    contexts: the positions listed on the device outrun their room, which the 64-bit count has to notice too."""
    monkeypatch.setattr(levels_mod, "W_MAX", 0)
    tok, sizes, starts, _ = data.device_tokens(corpus.shards())
    eng = levels_mod.LevelBuild(tok, sizes, starts, LEVELS)
    block = corpus.train[1000:9000]
    absent = np.setdiff1d(np.arange(50000), corpus.train)[0]
    for q in (np.append(block, np.full(24_000, absent, np.uint16)), np.tile(block, 4)):
        q = q.astype(np.uint16)
        x, tgt, avail = C.queries(q, [], "cuda")
        out = eng.build(x, tgt, avail, cnt_top=cnt_top).counts.cpu().numpy()
        for li, k in enumerate(LEVELS):
            o = O.query_counts(corpus.train, corpus.bounds, q[:-1], q[1:], O.segments(q[:-1]), k,
                               cnt_top=cnt_top or 1 << 30)
            assert np.array_equal(out[0, li].view(np.uint32), o["tot"]), f"tot k={k}"
            assert np.array_equal(out[1, li], o["dist"].astype(np.int32)), f"dist k={k}"
            assert np.array_equal(out[2, li].view(np.uint32), o["cnt"]), f"cnt k={k}"
    assert eng.reruns > 0
