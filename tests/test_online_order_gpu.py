"""GPU: an online stream's layout and training order made on the device (ng_online_tau, ng_online_layout,
ng_online_avail, ng_online_order and a stable sort), against a position-by-position restatement: overlapping, empty and
out-of-order spans, parts and end-of-text tokens, contexts longer than a part, steps close together and far apart."""

import numpy as np
import pytest

from ngram_amd import online
from ngram_amd.online import NONE, OnlineRows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,parts", [(1, 1), (2, 2), (17, 3), (300, 1), (5000, 7)])
@pytest.mark.parametrize("spread", [1, 40_000_000])
def test_training_order(gpu, n, parts, spread):
    rng = np.random.default_rng(n + parts)
    tok = rng.integers(0, 50, n).astype(np.uint16)
    tok[rng.random(n) < 0.05] = 50256
    bounds = [0, *sorted(rng.choice(np.arange(1, n), parts - 1, replace=False).tolist()), n] if parts > 1 else [0, n]
    lo = rng.integers(0, n + 1, 3 * parts)
    hi = np.minimum(lo + rng.integers(0, max(2, n // 4), 3 * parts), n)
    spans = np.stack([lo, hi, rng.integers(0, 9, 3 * parts) * spread], 1)
    rows = OnlineRows(tok, bounds, spans)
    tau, tau_in = np.full(n, NONE, np.int64), np.full(n, NONE, np.int64)
    part = np.searchsorted(bounds, np.arange(n), side="right") - 1
    for a, b, s in spans:
        tau_in[a:b] = np.minimum(tau_in[a:b], s)
        tau[a:b] = np.minimum(tau[a:b], s)
        if b > a and b < n and part[b] == part[b - 1]:
            tau[b] = min(tau[b], s)
    assert np.array_equal(rows.tau.cpu().numpy().view(np.uint32), tau)
    assert np.array_equal(rows.tau_in.cpu().numpy().view(np.uint32), tau_in)
    avail, has_next = np.zeros(n, np.int64), np.zeros(n, np.int64)
    for g in range(n):
        avail[g] = 1 if tok[g] == 50256 or g == bounds[part[g]] else avail[g - 1] + 1
        has_next[g] = g + 1 < n and part[g + 1] == part[g]
    assert np.array_equal(rows.avail.cpu().numpy(), avail)
    assert np.array_equal(rows.has_next.cpu().numpy(), has_next)
    levels = [1, 2, 5, 20]
    got = rows._by_step([(rows.tau_in, 0)] + [(rows.tau, k) for k in levels], rows.max_step + 1)
    for (order, steps), k in zip(got, [0, *levels]):
        if k == 0:
            step = tau_in
        else:
            step = np.full(n, NONE, np.int64)
            for g in range(n):
                if g - k + 1 >= bounds[part[g]] and has_next[g]:
                    m = tau[g - k + 1 : g + 2].max()
                    step[g] = m + 1 if m != NONE else NONE
        want = np.flatnonzero(step != NONE)
        want = want[np.argsort(step[want], kind="stable")]
        assert np.array_equal(order.cpu().numpy(), want), k
        for s in {0, 1, int(spread), int(spans[:, 2].max()) + 1, *step[want].tolist()}:
            assert steps.before(int(s)) == int((step[want] < s).sum()), (k, s)


@pytest.mark.parametrize("m,top", [(40, 40), (40, 1100), (40, 1200), (40, 1_000_000), (3000, 7000), (3000, 7100)])
def test_bounds_of_steps_close_together_and_apart(gpu, m, top, monkeypatch):
    """A few spans whose steps are far apart keep bounds of the steps in use, not of every step up to the last (host
    arrays of a million entries per level otherwise); both forms give the same bounds and the same largest step."""
    rng = np.random.default_rng(m)
    n = 8000
    at = np.linspace(0, n, m + 1).astype(np.int64)
    steps = np.append(np.sort(rng.choice(top - 1, m - 1, replace=False)), top - 1)
    spans = np.stack([at[:-1], at[1:], rng.permutation(steps)], 1)
    tok = rng.integers(0, 9, n).astype(np.uint16)
    got = {}
    for table in (online.STEP_TABLE, 0):
        monkeypatch.setattr(online, "STEP_TABLE", table)
        rows = OnlineRows(tok, [0, n], spans)
        got[table] = rows._by_step([(rows.tau_in, 0), (rows.tau, 2)], rows.max_step + 1)
    for (o1, b1), (o2, b2) in zip(*got.values()):
        assert np.array_equal(o1.cpu().numpy(), o2.cpu().numpy())
        assert len(b1.steps) <= 2 * m + 1026
        for s in (0, 1, top // 2, top, *steps[:50].tolist()):
            assert b1.before(int(s)) == b2.before(int(s)), s
    assert rows._most([b for _, b in got[0]]) == rows._most([b for _, b in list(got.values())[0]])


@pytest.mark.parametrize("times", [3, 70_000])
def test_spans_that_cover_the_stream_many_times(gpu, times):
    """Spans overlap freely, so their lengths add up to far more than the stream: at 70,000 times 2^20 positions to more
    than a launch has threads for (16 positions each)."""
    n = 1 << 20
    rng = np.random.default_rng(times)
    lo = rng.integers(0, 50, times)
    steps = rng.permutation(np.arange(5, 5 + times))
    rows = OnlineRows(np.zeros(n, np.uint16), [0, n], np.stack([lo, np.full(times, n), steps], 1))
    want = np.full(n, steps.min(), np.int64)
    for g in range(50):
        want[g] = steps[lo <= g].min() if (lo <= g).any() else NONE
    assert np.array_equal(rows.tau_in.cpu().numpy().view(np.uint32), want)
