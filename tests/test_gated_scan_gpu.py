"""GPU: the gated level scan whose waves choose per span between probing every position and listing the set ones
(ng_scan_emit's mode 4), against the dense scan (mode 0) of the same gate: the same hit bitmap and, as a multiset, the
same events."""

import numpy as np
import pytest
import torch

from ngram_amd.lib import Lib, i32, u64
from ngram_amd.qindex import QueryIndex

pytestmark = pytest.mark.gpu


# lengths around a wave's group (2048 positions) and its span (8 groups); one block makes its waves walk many spans
@pytest.mark.parametrize("L,grid", [(32, 1), (2048, 1), (2080, 3), (16384, 1), (65536 + 32, 1), (300_000 // 32 * 32, 1),
                                    (300_000 // 32 * 32, 5), (1 << 20, 64)])
@pytest.mark.parametrize("density", [0.0, 0.004, 0.3, 0.5, 0.97, -1.0])
@pytest.mark.parametrize("k,pre", [(2, 0), (2, 1), (6, 1)])
def test_gated_scan_matches_the_dense_one(gpu, L, grid, density, k, pre):
    lib = Lib()
    rng = np.random.default_rng(L * 7 + grid + k)
    host = rng.integers(0, 9, L).astype(np.uint16)
    host[:32] = 0xFFFF
    host[rng.random(L) < 0.01] = 0xFFFF
    tok = torch.from_numpy(host.view(np.int16)).cuda()
    q = rng.integers(0, 9, 4000).astype(np.uint16)
    x = torch.from_numpy(q.view(np.int16)).cuda()
    avail = torch.from_numpy(np.arange(1, 4001, dtype=np.int32)).cuda()
    vi = QueryIndex(lib, x, avail, k)
    if density < 0:  # dense and sparse spans side by side, empty ones among them
        bits = (rng.random(L) < np.repeat(rng.choice([0.0, 0.01, 0.6, 1.0], L // 4096 + 1), 4096)[:L])
    else:
        bits = rng.random(L) < density
    gate = torch.from_numpy(np.packbits(bits, bitorder="little").view(np.int32)).cuda()
    flag = torch.tensor([pre], dtype=torch.int32, device="cuda")
    R = -(-L // (grid * 8192)) * 8192
    got = []
    for mode in (0, 4):
        out = torch.full((L // 32,), -7, dtype=torch.int32, device="cuda")
        ev = torch.empty(grid * R, dtype=torch.int64, device="cuda")
        n = torch.empty(grid, dtype=torch.int32, device="cuda")
        flags = torch.zeros(2, dtype=torch.int32, device="cuda")
        dh = torch.empty((256, grid), dtype=torch.int32, device="cuda")
        lib("ng_scan_emit", tok, L, i32(k), gate, out, vi.table, u64(vi.cap), vi.rep, x, ev, u64(R), n, flags,
            i32(grid), i32(mode), dh, grid, flag, i32(0), i32(0), i32(0))
        counts = n.cpu().numpy()
        e = ev.cpu().numpy().reshape(grid, R)
        assert int(flags[0].item()) == 0
        events = np.concatenate([e[b, : counts[b]] for b in range(grid)])
        digits = np.bincount(events.view(np.uint64) >> np.uint64(56), minlength=256)
        assert np.array_equal(dh.cpu().numpy().sum(1), digits)
        got.append((out.cpu().numpy(), np.sort(events)))
    assert np.array_equal(got[0][0], got[1][0])
    assert np.array_equal(got[0][1], got[1][1])
    if density >= 0.3 and L >= 16384 and k == 2:
        assert len(got[0][1]) > 100
