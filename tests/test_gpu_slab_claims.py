"""Slab claims in small pools whose cursor goes round many times: bitmaps of even and odd
word counts, below and above the window that a claim looks at after a full word."""
import numpy as np
import pytest
import torch

import scenarios as S
from indexingpu_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("words", [2, 3, 15, 17, 33])
def test_claims_round_a_small_pool(words):
    """A first-in first-out set of keys with one-slab records, at most about half the pool:
    every insert finds a slab, whatever part of the bitmap is full at the cursor."""
    per = max(1, words // 2 - 1)  # each insert of a batch claims a bitmap word of its own
    rounds = 64
    rng = np.random.default_rng(words)
    keys, lens = W.unique_random_keys(rng, per * rounds, 1, 3)
    vals = W.make_values(keys, lens, 2)
    g = S.GpuBackend(16, pool_bytes=words * 32 * 128)
    assert g.t.pool_slabs() == words * 32
    held = 10 * words // per
    for r in range(rounds):
        b = slice(r * per, (r + 1) * per)
        assert np.asarray(g.insert(keys[b], lens[b], vals[b], None, 3, 2)).all()
        if r >= held:
            e = slice((r - held) * per, (r - held + 1) * per)
            assert np.asarray(g.erase(keys[e], lens[e], 3)).all()
    live = slice(max(0, rounds - held) * per, rounds * per)
    fv, fl = g.find(keys[live], lens[live], 3, 2)
    assert (np.asarray(fl).reshape(-1) == 2).all()
    assert np.array_equal(np.asarray(fv).reshape(-1, 2), vals[live])
    g.t.check_device_error()
    ok, *_, msg = g.validate()
    assert ok, msg
    torch.cuda.synchronize()
