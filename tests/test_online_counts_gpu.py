"""GPU: the count rows of a range of steps answered all at once (OnlineRows.counts: searches over each context's
occurrences in step order) against the same range advanced step by step on the incremental state: overlapping and
out-of-order spans, parts, steps without queries, ranges that start late or are empty, contexts longer than the stream,
a hot context, both rules."""

import numpy as np
import pytest
import torch

from ngram_amd import online
from ngram_amd.online import OnlineRows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,parts,vocab", [(1, 1, 3), (2, 1, 1), (40, 3, 2), (257, 1, 1), (6000, 5, 20), (6000, 2, 3)])
@pytest.mark.parametrize("rule,lo,hi", [("step", 0, 12), ("step", 3, 5), ("step", 4, 4), ("segment", 0, 0)])
def test_counts_match_the_stepwise_state(gpu, n, parts, vocab, rule, lo, hi):
    rng = np.random.default_rng(n * 5 + parts)
    tok = rng.integers(0, vocab, n).astype(np.uint16)
    tok[rng.random(n) < 0.02] = 50256
    bounds = [0, *sorted(rng.choice(np.arange(1, n), parts - 1, replace=False).tolist()), n] if parts > 1 else [0, n]
    a = rng.integers(0, n + 1, 6 * parts)
    b = np.minimum(a + rng.integers(0, max(2, n // 3), 6 * parts), n)
    rows = OnlineRows(tok, bounds, np.stack([a, b, rng.integers(0, 10, 6 * parts)], 1))
    levels = [3, 1, 2, 6, 60, 2]  # in any order, one of them twice
    _, want, at = rows._range_rows((), (1,), 0, levels, lo, hi, rule)
    got, at2 = rows._range_counts(levels, lo, hi, rule)
    assert torch.equal(torch.sort(at).values, torch.sort(at2).values)
    for name in ("tot", "dist", "cnt"):
        assert torch.equal(got[name], want[name]), name
    if n >= 6000 and (lo, hi) in ((0, 12), (0, 0)):  # the streams' draws leave counted contexts to compare
        assert int(got["tot"].max()) > 3


def test_calls_at_the_edge_of_what_is_taken(gpu):
    """No levels raise ValueError; a level past the kernels' longest context raises once a query is asked of it, and a
    range without queries asks none."""
    n = 1000
    tok = np.random.default_rng(0).integers(0, 5, n).astype(np.uint16)
    rows = OnlineRows(tok, [0, n], [(0, 500, 2), (500, n, 5)])
    with pytest.raises(ValueError):
        rows.segment_counts([])
    with pytest.raises(RuntimeError):
        rows.segment_counts([65])
    out = [np.full((n, 1), 7, t) for t in (np.uint32, np.uint16, np.uint32)]
    with pytest.raises(RuntimeError):
        rows.counts([65], 0, 6, *out)
    for lo, hi in ((0, 0), (0, 2), (3, 5), (6, 9)):
        rows.counts([65], lo, hi, *out)
    assert all((o == 7).all() for o in out)


@pytest.mark.parametrize("trained", [0, 1, 2, 300, 4800])
@pytest.mark.parametrize("spread", [1, 3_000_000])
@pytest.mark.parametrize("in_order", [True, False])
def test_a_stream_of_which_few_positions_are_trained(gpu, trained, spread, in_order, monkeypatch):
    """Picking the trained positions out before they are sorted gives the state and the count rows that sorting the whole
    stream gives, and keeps lists only as long as they are."""
    n, m = 20_000, max(1, trained // 40)
    rng = np.random.default_rng(trained)
    tok = rng.integers(0, 6, n).astype(np.uint16)
    tok[rng.random(n) < 0.01] = 50256
    at = rng.choice(n // 50 - 1, m, replace=False) * 50
    if in_order:
        at = np.sort(at)
    size = np.full(m, 40) if trained >= 40 else np.full(m, trained)
    spans = np.stack([at, at + size, rng.integers(0, 7, m) * spread], 1)
    got = {}
    for few in (1, 1 << 40):
        monkeypatch.setattr(online, "FEW_MIN", few)
        rows = OnlineRows(tok, [0, n // 3, n], spans if few == 1 else spans[::-1])  # in order (or not), and the other way
        rows.prepare([1, 3], [1, 3], 4, [1, 3, 9])
        lists = [rows.state["q_pos"]] + [lv["occ"] for lv in rows.state["levels"].values()]
        out = [np.zeros((n, 3), t) for t in (np.uint32, np.uint16, np.uint32)]
        rows.counts([3, 1, 9], 0, 7 * spread, *out)
        got[few] = [t.cpu().numpy() for t in lists] + out
        if few == 1:
            assert all(t.untyped_storage().nbytes() <= 4 * t.numel() for t in lists)
    for a, b in zip(*got.values()):
        assert np.array_equal(a, b)
    assert trained < 300 or got[1][-3].max() > 1
