"""GPU: the query masks longest_match takes and refuses: any shape that broadcasts over the positions, as a device tensor
or a single host value; a mask in host memory, or of another length, raises before anything is launched on it."""

import numpy as np
import pytest
import torch

import oracle as O
from ngram_amd import longest as LG
from ngram_amd.data import device_tokens
from ngram_amd.lib import Lib

pytestmark = pytest.mark.gpu


def _call(query):
    rng = np.random.default_rng(5)
    train = rng.integers(0, 30, 4000).astype(np.uint16)
    x = rng.integers(0, 30, 700).astype(np.uint16)
    tok, _, _, _ = device_tokens([train])
    xt = torch.from_numpy(x.view(np.int16)).cuda()
    want = O.longest_match(train, np.array([0, len(train)], np.int64), x, O.segments(x), 8)
    return want, [t.cpu().numpy() for t in LG.longest_match(tok, xt, LG._segments(xt, Lib()), 8, query=query)[:3]]


@pytest.mark.parametrize("make", [lambda n: torch.ones(n, dtype=torch.bool)[::2],  # another length
                                  lambda n: torch.ones(n, dtype=torch.bool),  # host memory
                                  lambda n: torch.ones(n, dtype=torch.uint8),
                                  lambda n: torch.ones(n + 1, dtype=torch.bool, device="cuda")])
def test_masks_that_are_refused(gpu, make):
    with pytest.raises(RuntimeError):
        _call(make(700))


@pytest.mark.parametrize("make", [lambda n: torch.ones(n, dtype=torch.bool, device="cuda"),
                                  lambda n: torch.ones(2 * n, dtype=torch.bool, device="cuda")[::2],  # strided
                                  lambda n: torch.ones(n, dtype=torch.int64, device="cuda"),
                                  lambda n: torch.ones(1, dtype=torch.bool, device="cuda"),
                                  lambda n: torch.tensor(True)])  # one host value: torch takes it
def test_masks_that_ask_for_every_position(gpu, make):
    want, got = _call(make(700))
    for w, g in zip(want, got):
        assert np.array_equal(g.view(w.dtype), w)
