"""GPU: the count mixture's features against the oracle at the edges of the tiled kernel (positions around a tile, few
and many levels, outputs at unaligned places) and over totals on both sides of every power of two, where float32's log2
rounds up or not."""

import numpy as np
import pytest
import torch

import oracle as O
from ngram_amd import exact_match
from ngram_amd.lib import Lib, i32

pytestmark = pytest.mark.gpu


def _counts(n, L, rng):
    edge = np.array([(1 << b) + d for b in range(33) for d in range(-300, 301) if 0 <= (1 << b) + d < 1 << 32], np.uint32)
    c = np.empty((3, L, n), np.int32)
    c[0] = np.where(rng.random((L, n)) < 0.7, rng.choice(edge, (L, n)), rng.integers(0, 1 << 32, (L, n))).astype(
        np.uint32).view(np.int32)
    c[1] = np.minimum(rng.integers(0, 4, (L, n)) ** 8, 65535)
    c[2] = rng.integers(0, 1 << 31, (L, n))
    return c


@pytest.mark.parametrize("n", [1, 3, 255, 256, 257, 4099])
@pytest.mark.parametrize("L", [1, 2, 3, 7, 16, 17])
def test_features_match_the_oracle(gpu, n, L):
    c = _counts(n, L, np.random.default_rng(n * 31 + L))
    for got, want in zip(exact_match.features(torch.from_numpy(c).cuda()), O.features(c)):
        assert np.array_equal(got.cpu().numpy(), want)


def test_features_at_unaligned_outputs(gpu):
    n, L = 513, 3
    c = _counts(n, L, np.random.default_rng(5))
    dev = torch.from_numpy(c).cuda()
    f = [torch.empty(n * L + 1, dtype=torch.float32, device="cuda")[1:] for _ in range(3)]
    b = [torch.empty(n * L + 1, dtype=torch.int64, device="cuda")[1:] for _ in range(2)]
    Lib()("ng_features", dev, i32(L), n, i32(25), *f, *b)
    for got, want in zip([*f, *b], O.features(c)):
        assert np.array_equal(got.cpu().numpy().reshape(n, L), want)


def test_every_total_near_a_power_of_two(gpu):
    tot = np.concatenate([np.arange(max(0, (1 << b) - 70_000), min(1 << 32, (1 << b) + 3), dtype=np.uint64)
                          for b in range(17, 33)]).astype(np.uint32)
    c = np.zeros((3, 1, len(tot)), np.int32)
    c[0, 0] = tot.view(np.int32)
    got = exact_match.features(torch.from_numpy(c).cuda(), 40)[3].cpu().numpy()
    lg = np.log2(tot.astype(np.float32).astype(np.float64)).astype(np.float32)
    assert np.array_equal(got[:, 0], np.clip(np.floor(lg), 0, 39).astype(np.int64))
