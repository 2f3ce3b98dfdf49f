"""GPU: the 32-bit count where a level's partitions are the first pass's digit itself (few events: no second pass), where
they go below it, and at the most it takes, against the oracle: with and without records in runs, top 1 and top 8, one
query position and many."""

import math

import numpy as np
import pytest

import oracle as O
from ngram_amd import counts as C
from ngram_amd import data
from ngram_amd import partcount as P

pytestmark = pytest.mark.gpu

LEVELS = (1, 2, 4)


@pytest.fixture(scope="module")
def corpus():
    return data.make_corpus("c3", train_tokens=200_000, query_tokens=20_001, shard_tokens=70_000)


@pytest.mark.parametrize("target,pbits", [(1 << 30, 8), (100, 11), (5, 13), (1, 15)])
@pytest.mark.parametrize("topk", [1, 8])
@pytest.mark.parametrize("queries", [1, 20_000])
@pytest.mark.parametrize("runs", [True, False])
def test_partition_layouts(corpus, target, pbits, topk, queries, runs, monkeypatch):
    monkeypatch.setattr(P, "P32_TARGET", target)
    if not runs:  # every event bit mixed: the words are grouped by context instead
        import ngram_amd.levels as levels_mod

        monkeypatch.setattr(levels_mod.LevelBuild, "_mbits", staticmethod(lambda W, ids, ktop: W))
    q = corpus.query[-(queries + 1) :]
    cb = C.CountBuild(corpus.shards(), levels=LEVELS, level_shards={}, topk=topk)
    cb.start_load(1)
    x, tgt, avail = C.queries(q, [], "cuda")
    for _ in range(2):  # sizes unknown, then learnt
        out = cb.counts(x, tgt, avail).cpu().numpy()
        for li, k in enumerate(LEVELS):
            o = O.query_counts(corpus.train, corpus.bounds, q[:-1], q[1:], O.segments(q[:-1]), k, cnt_top=1 << 30,
                               ntop=topk)
            assert np.array_equal(out[0, li].view(np.uint32), o["tot"]), f"tot k={k}"
            assert np.array_equal(out[1, li].astype(np.uint16), o["dist"]), f"dist k={k}"
            assert np.array_equal(out[2, li].view(np.uint32), o["cnt"]), f"cnt k={k}"
            assert np.array_equal(cb.top_tok[li].cpu().numpy().view(np.uint16), o["top_tok"][:, :topk]), f"top k={k}"
            assert np.array_equal(cb.top_cnt[li].cpu().numpy().view(np.uint32), o["top_cnt"][:, :topk]), f"top k={k}"
    # the second build's partitions, sized from the first one's events and pairs: the first pass's digit itself where they
    # fit it, else at least PART_MIN_BITS
    taken = set()
    for k in LEVELS:
        idb, W = P.w_bits(cb.info[k]["ids"])
        d1, by_range = P.first_digit(W), runs and P.runs_fit(cb.info[k]["ids"], topk)
        used = cb.info[k]["ids"] / (1 << idb) if by_range else 1.0
        want = math.ceil(math.log2(max(1.0, cb.info[k]["pairs"] / target / used)))
        want = max(want, P.PART_MIN_BITS) if want > d1 else d1
        assert cb.info[k]["pbits"] == min(want, P.pbits32_max(cb.info[k]["ids"])), f"k={k}"
        taken.add(cb.info[k]["pbits"])
    assert not cb.engine.wide and not cb.engine.min_pbits  # none was counted again with more
    assert taken == {8} if target == 1 << 30 else queries == 1 or max(taken) >= pbits
