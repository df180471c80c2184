"""Writes applied border node by border node (batches of any size, by the knob) against the
oracle: split and full nodes at every fanout edge, more requests of a node than one tile
takes, two kinds of entry with one slice, trie layers and push-downs, inline, long and
multi-slab values, erases that empty nodes and layers, and mixed batches."""
import numpy as np
import pytest

import scenarios as S
from indexingpu_amd import workloads as W

pytestmark = pytest.mark.gpu


def _eq(a, b):
    assert np.array_equal(np.asarray(a), np.asarray(b))


def _check(g, o):
    assert g.items() == o.items()
    ok, *_, msg = g.validate()
    assert ok, msg


def _unique(rng, n, mk, alphabet, prefix=0):
    lens = rng.integers(1, mk + 1, size=n).astype(np.uint32)
    keys = rng.integers(0, alphabet, size=(n, mk), dtype=np.uint64).astype(np.uint32)
    keys[:, :prefix] &= 1
    keys[np.arange(mk)[None, :] >= lens[:, None]] = 0
    _, first = np.unique(W.key_hash64(keys, lens), return_index=True)
    first = np.sort(first)
    return np.ascontiguousarray(keys[first]), lens[first]


SHAPES = {
    # (slice alphabet, max key slices, binary prefix slices, max value slices)
    "wide": (1 << 32, 3, 0, 2),         # almost every entry its own slice
    "crowded": (1 << 12, 2, 0, 1),      # ends-here and continues entries with one slice
    "layers": (5, 12, 6, 3),            # shared prefixes, push-downs, deep layers
    "long": (1 << 20, 40, 0, 70),       # multi-slab records
}


@pytest.mark.parametrize("fanout", [(0, 0), (2, 3), (3, 4), (13, 15)], ids=str)
@pytest.mark.parametrize("shape", list(SHAPES))
def test_grouped_writes(shape, fanout):
    alphabet, mk, prefix, mv = SHAPES[shape]
    rng = np.random.default_rng(11)
    keys, lens = _unique(rng, 6000, mk, alphabet, prefix)
    n = len(lens)
    vlens = rng.integers(0, mv + 1, size=n).astype(np.uint32)
    vals = rng.integers(0, 1 << 32, size=(n, mv), dtype=np.uint64).astype(np.uint32)
    g, o = S.GpuBackend(16, pool_bytes=256 << 20, fanout=fanout), S.OracleBackend()
    g.t.set_write_groups(1)

    def both(op, at, v=vals, vl=vlens, **kw):
        if op == "erase":
            _eq(g.erase(keys[at], lens[at], mk), o.erase(keys[at], lens[at], mk))
        else:
            _eq(getattr(g, op)(keys[at], lens[at], v[at], vl[at], mk, mv, **kw),
                getattr(o, op)(keys[at], lens[at], v[at], vl[at], mk, mv, **kw))

    order = rng.permutation(n)
    cut = n // 8
    both("insert", order[:cut])
    both("insert", order[:5])                       # all stored already
    both("insert", order[cut // 2: 3 * cut])        # half the tree and twice as many new
    both("insert", order[3 * cut:], upsert=True)    # many requests per node
    _check(g, o)
    v2, vl2 = vals ^ np.uint32(0xA5A5A5A5), np.roll(vlens, 1)
    both("update", order[:n // 3], v2, vl2)
    both("insert", order[n // 4: n // 2], v2, vl2, upsert=True)
    for a, b in zip(g.find(keys, lens, mk, mv), o.find(keys, lens, mk, mv)):
        _eq(a, b)
    both("erase", order[::3])
    both("update", order[:n // 2])                  # some stored, some gone
    _check(g, o)
    by_key = np.lexsort(keys.T[::-1])
    both("erase", by_key[n // 4: 3 * n // 4])       # runs of neighbours: nodes that empty
    _check(g, o)
    both("insert", by_key[n // 4: n // 2])          # in key order, into one stretch
    both("erase", order)                            # everything
    _check(g, o)
    both("insert", order)
    _check(g, o)


@pytest.mark.parametrize("tile", [16, 64])
@pytest.mark.parametrize("n", [1, 63, 64, 1000, 50_000])
def test_grouped_mixed_batches(n, tile):
    """Mixed batches whose writes are grouped; the finds' outputs stay their own."""
    wl = W.MixedWorkload(60_000, key_len=3, seed=n, find_frac=0.5, insert_frac=0.25)
    g, o = S.GpuBackend(tile, pool_bytes=256 << 20), S.OracleBackend()
    g.t.set_mixed_split(0)
    g.t.set_write_groups(1)
    _eq(g.insert(wl.keys, wl.lens, wl.values, None, 3, 2),
        o.insert(wl.keys, wl.lens, wl.values, None, 3, 2))
    for _ in range(3):
        bt = wl.batch(n)
        vl = np.full(len(bt["types"]), 2, np.uint32)
        for a, b in zip(g.mixed(bt["types"], bt["keys"], bt["lens"], bt["values"], vl, 3, 2),
                        o.mixed(bt["types"], bt["keys"], bt["lens"], bt["values"], vl, 3, 2)):
            _eq(a, b)
    _check(g, o)


def test_grouped_writes_out_of_slabs():
    """A pool that runs out inside grouped writes: what succeeded is the oracle's, the tree
    is whole, and freed slabs serve the failed keys."""
    d = W.plain_batch_workload(8000, seed=3, n_find=16, n_erase=16)
    keys, lens, vals = d["keys"], d["lens"], d["values"]
    g = S.GpuBackend(16, pool_bytes=4096 * 128)
    g.t.set_write_groups(1)
    r = g._zeros(len(lens), np.uint8)
    g.t.insert(g._d(keys), 8, g._d(lens), g._d(vals), 2, None, len(lens), results=r)
    got = g._h(r, np.uint8).astype(bool)
    assert g.t.device_error() == 1
    assert 1000 < got.sum() < 4096
    fv, fl = g.find(keys, lens, 8, 2)
    assert np.array_equal(np.asarray(fl) == 2, got)
    assert np.array_equal(np.asarray(fv)[got], vals[got])
    ok, *_, msg = g.validate()
    assert ok, msg
    at = np.flatnonzero(got)
    assert np.asarray(g.erase(keys[at], lens[at], 8)).all()
    late = np.flatnonzero(~got)[:500]
    assert np.asarray(g.insert(keys[late], lens[late], vals[late], None, 8, 2)).all()
    ok, *_, msg = g.validate()
    assert ok, msg
