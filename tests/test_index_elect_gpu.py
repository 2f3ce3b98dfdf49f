"""GPU: query indexes of sizes around a block and above, of contexts as frequent as they get (one token only: one
lane a block inserts for the rest) and rare ones: the same contexts, one id each, whatever inserted."""

import numpy as np
import pytest
import torch

from ngram_amd.lib import Lib
from ngram_amd.qindex import QueryIndex

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 255, 256, 257, 5000, 300_001])
@pytest.mark.parametrize("vocab,k", [(1, 1), (1, 5), (50, 2), (40_000, 1), (40_000, 6)])
@pytest.mark.parametrize("listed", [False, True])
def test_contexts_and_ids(gpu, n, vocab, k, listed):
    rng = np.random.default_rng(n + vocab + k)
    N = n + n // 3 if listed else n
    x = (rng.random(N) ** 4 * vocab).astype(np.uint16)
    avail = np.minimum(np.arange(1, N + 1), rng.integers(1, 4 * k + 1, N)).astype(np.int32)
    pos = np.sort(rng.permutation(N)[:n]).astype(np.int32) if listed else None
    qi = QueryIndex(Lib(), torch.from_numpy(x.view(np.int16)).cuda(), torch.from_numpy(avail).cuda(), k,
                    positions=None if pos is None else torch.from_numpy(pos).cuda(), compact=listed)
    p = np.arange(n) if pos is None else pos
    valid = avail[p] >= k
    ids = qi.ctx_of.cpu().numpy()
    assert np.array_equal(ids >= 0, valid)
    pv = p[valid].astype(np.int64)
    rows = np.stack([x[pv - j] for j in range(k)], 1) if len(pv) else np.zeros((0, k), np.uint16)
    uniq, inv = np.unique(rows, axis=0, return_inverse=True)
    assert int(qi.n) == len(uniq)
    first = np.full(len(uniq), -1, np.int64)
    first[inv.reshape(-1)] = ids[valid]
    assert np.array_equal(first[inv.reshape(-1)], ids[valid]) and len(np.unique(first)) == len(uniq)
    rep = qi.rep.cpu().numpy()
    if len(pv):  # an id's representative is a position of its context
        r = rep[first].astype(np.int64)
        assert np.array_equal(np.stack([x[r - j] for j in range(k)], 1), uniq)
