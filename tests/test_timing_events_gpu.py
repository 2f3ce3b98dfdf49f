"""GPU: the launches' timing events of a count build and of a table: recorded where `timed` is set before the build, else
an empty list that says so with a warning."""

import warnings

import pytest
import torch

from ngram_amd import counts as C
from ngram_amd import data
from ngram_amd.count_table import CountTable

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def corpus():
    return data.make_corpus("c3", train_tokens=100_000, query_tokens=10_001, shard_tokens=40_000)


def test_kernel_events_of_a_count_build(corpus):
    cb = C.CountBuild(corpus.shards(), levels=(2, 3), level_shards={})
    cb.start_load(1)
    x, tgt, avail = C.queries(corpus.query, [], "cuda")
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert cb.kernel_events == []  # nothing built yet
        cb.counts(x, tgt, avail)
    with pytest.warns(RuntimeWarning, match="timed"):
        assert cb.kernel_events == []
    cb.engine.timed = True
    cb.counts(x, tgt, avail).cpu()
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        events = cb.kernel_events
    assert {2, 3} == {k for _, k, *_ in events}
    assert all(e0.elapsed_time(e1) >= 0 for _, _, _, e0, e1, _ in events)
    assert {"qindex", "scan_emit", "count", "pos_gather"} <= {name for name, *_ in events}


@pytest.mark.parametrize("timed", [True, False])
def test_events_of_a_table(corpus, timed):
    tok, sizes, starts, _ = data.device_tokens(corpus.shards())
    ct = CountTable.from_device(tok, sizes, starts, [2, 3])
    assert ct.events == []
    ct.timed = timed
    ct.build()
    x, tgt, avail = C.queries(corpus.query, [], "cuda")
    ct.query_device(x, tgt, avail)
    torch.cuda.synchronize()
    if timed:
        assert {2, 3} == {k for _, k, *_ in ct.events}
        assert all(e0.elapsed_time(e1) >= 0 for _, _, e0, e1 in ct.events)
    else:
        with pytest.warns(RuntimeWarning, match="timed"):
            assert ct.events == []
