"""Device memory that closed indexes leave for the next ones: reused without a trace of the
old index, bounded, and given back."""
import numpy as np
import pytest
import torch

import scenarios as S
from indexingpu_amd import masstree as MT
from indexingpu_amd import workloads as W

pytestmark = pytest.mark.gpu


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()


def test_reused_memory_holds_nothing_of_the_old_index():
    o = None
    for seed in (1, 2, 3):
        d = W.plain_batch_workload(30_000, seed=seed, n_find=20_000, n_erase=10_000)
        g, o = S.GpuBackend(16, pool_bytes=64 << 20), S.OracleBackend()
        assert g.items() == []
        assert np.array_equal(g.insert(d["keys"], d["lens"], d["values"], None, 8, 2),
                              o.insert(d["keys"], d["lens"], d["values"], None, 8, 2))
        for a, b in zip(g.find(d["find_keys"], d["find_lens"], 8, 2),
                        o.find(d["find_keys"], d["find_lens"], 8, 2)):
            assert np.array_equal(np.asarray(a), np.asarray(b))
        assert np.array_equal(g.erase(d["erase_keys"], d["erase_lens"], 8),
                              o.erase(d["erase_keys"], d["erase_lens"], 8))
        assert g.items() == o.items()
        g.t.close()


@pytest.mark.parametrize("pools_mib", [(600,), (600, 700, 500), (16 << 10,)], ids=str)
def test_kept_memory_is_bounded_and_given_back(pools_mib):
    MT.release_memory()
    before, total = _free()
    live = [MT.GpuMasstree(pool_bytes=m << 20) for m in pools_mib]
    assert before - _free()[0] >= sum(m << 20 for m in pools_mib)
    for t in live:
        t.close()
    kept = before - _free()[0]
    assert kept <= total // 32 + (64 << 20)  # (and what the driver keeps for itself)
    MT.release_memory()
    assert before - _free()[0] <= (64 << 20)
