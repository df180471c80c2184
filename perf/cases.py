"""Performance cases of the GPU Masstree: what programs have it do, through its host API.

A case is a dict of plain values; `kind` names the calls of one pass:

  find     one read-only find batch over a resident index
  load     a new index, one insert batch into it, one find batch over the loaded keys
  churn    one insert batch into a resident index (one key in ten is stored already), one
           erase batch of the new keys (and one in ten that is not stored)
  update   one update (or upsert) batch over resident keys, one find batch of them
  mixed    two mixed batches of finds, inserts and erases; the second erases what the
           first inserted and inserts what it erased, so a pass leaves the entries as they were
  scan     one batch of range scans over a resident index
  batched  a sequence of such mixed batches in one multi_batch call

Keys are rows of u32 slices.  `prefix` = 0: 2 or more random slices; `prefix` = p: the
first p slices are one of 256 random rows (hierarchical keys: a path, a table id), the
rest random.  `min_len`..`max_len` is the key length in slices (uniform), `value_len`
the value length.  Half of a find batch's keys are stored (a uniform sample), half are
fresh; the finds of mixed batches are Zipf(0.99) over the stored keys.  Everything is
drawn on the GPU from the seed.  Outputs are whole numbers, so there is no exact().
"""
import math

import torch

from indexingpu_amd import REQUEST_ERASE, REQUEST_FIND, REQUEST_INSERT, GpuMasstree

M = 1 << 20
LINE = 64        # bytes of a random access to HBM
PREFIXES = 256
CHUNK = 1 << 24  # rows drawn or gathered by one torch call


def listed():
    var = dict(prefix=0, min_len=2, max_len=8, value_len=2)
    path = dict(prefix=12, min_len=16, max_len=16, value_len=2)
    return [
        # point lookups of one request: a handful of keys, where launches and latency count
        dict(name="find_few", kind="find", keys=100_000, batch=100, concurrent=False,
             prefix=0, min_len=2, max_len=2, value_len=1),
        # the 64-bit-key index with 32-bit values, a million keys and a million lookups
        dict(name="find_fixed_1m", kind="find", keys=1_000_000, batch=1_000_000,
             concurrent=False, prefix=0, min_len=2, max_len=2, value_len=1),
        # the largest index and batch: an analytics join probing 64M variable-length keys
        dict(name="find_varlen_64m", kind="find", keys=64 * M, batch=64 * M, concurrent=False,
             **var),
        # lookups of hierarchical keys, through many trie layers
        dict(name="find_prefixed", kind="find", keys=4 * M, batch=1_000_003, concurrent=False,
             **path),
        # a document store: long keys (up to 160 bytes) and 256-byte values
        dict(name="find_long", kind="find", keys=400_000, batch=300_001, concurrent=False,
             prefix=0, min_len=8, max_len=40, value_len=64),
        # bulk load of an index from nothing
        dict(name="load_16m", kind="load", keys=16 * M, **var),
        # a small transaction's writes
        dict(name="churn_few", kind="churn", keys=1_000_000, batch=1_000, **var),
        # ingest and retention: large insert and erase batches on a resident index
        dict(name="churn_4m", kind="churn", keys=16 * M, batch=4 * M, **var),
        # refresh of stored values, then reading them back
        dict(name="update_1m", kind="update", keys=4 * M, batch=1_000_000, upsert=False,
             prefix=0, min_len=2, max_len=8, value_len=8),
        # a key-value service's steps: 90% finds, 5% inserts, 5% erases on 64M keys
        dict(name="mixed_1m", kind="mixed", keys=64 * M, batch=M,
             prefix=0, min_len=4, max_len=4, value_len=2),
        # range queries with limits of 1 to 100 entries
        dict(name="scan_64k", kind="scan", keys=16 * M, batch=65_536, limit=100, upper=False,
             prefix=0, min_len=4, max_len=4, value_len=2),
        # a queue of uneven mixed batches (1K to 256K requests) over hierarchical keys
        dict(name="batched_24", kind="batched", keys=4 * M, batches=24, batch=256 * 1024, **path),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))

    kind = rng.choice(["find", "find", "load", "churn", "churn", "update", "mixed", "scan",
                       "batched"])
    shape = rng.choice(["fixed", "var", "var", "path", "long"])
    case = dict(kind=kind, keys=spread(2_000, 16 * M))
    if shape == "fixed":
        n = rng.choice([2, 4])
        case.update(prefix=0, min_len=n, max_len=n, value_len=rng.choice([1, 2]))
    elif shape == "var":
        case.update(prefix=0, min_len=2, max_len=rng.randint(3, 8), value_len=rng.randint(1, 8))
    elif shape == "path":
        p = rng.randint(2, 12)
        case.update(prefix=p, min_len=p + 2, max_len=p + rng.randint(2, 4),
                    value_len=rng.randint(1, 4))
        case.update(keys=min(case["keys"], 4 * M))
    else:
        case.update(keys=min(case["keys"], 400_000), prefix=0, min_len=rng.randint(4, 8),
                    max_len=rng.randint(9, 40), value_len=rng.randint(16, 64))
    if kind == "load":
        return case
    if kind == "find":
        case.update(batch=min(spread(50, 4 * case["keys"]), 16 * M), concurrent=rng.random() < 0.2)
    elif kind == "churn":
        case.update(batch=spread(20, case["keys"] // 2))
    elif kind == "update":
        case.update(batch=spread(20, case["keys"]), upsert=rng.random() < 0.5)
    elif kind == "mixed":
        case.update(batch=min(spread(100, case["keys"]), M))
    elif kind == "scan":
        case.update(batch=spread(10, 65_536), limit=rng.randint(1, 100),
                    upper=rng.random() < 0.5)
    else:
        case.update(batch=min(spread(200, case["keys"]), 256 * 1024), batches=rng.randint(2, 24))
    return case


# ------------------------------------------------------------------ inputs
def _slices(gen, n, m):
    out = torch.empty((n, m), dtype=torch.int32, device="cuda")
    for part in out.split(CHUNK):
        part.random_(-(1 << 31), 1 << 31, generator=gen)
    return out


class _Keys:
    """Draws keys (rows, lengths) and values of a case."""

    def __init__(self, case, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)
        self.case = case
        self.mk, self.mv = case["max_len"], case["value_len"]
        if case["prefix"]:
            self.prefixes = _slices(self.gen, PREFIXES, case["prefix"])

    def index(self, high, n):
        return torch.randint(0, high, (n,), generator=self.gen, device="cuda")

    def keys(self, n):
        c = self.case
        rows = _slices(self.gen, n, self.mk)
        if c["prefix"]:
            rows[:, :c["prefix"]] = self.prefixes[self.index(PREFIXES, n)]
        if c["min_len"] == self.mk:
            return rows, None  # every key has max_key_length slices
        lens = torch.randint(c["min_len"], self.mk + 1, (n,), generator=self.gen, device="cuda",
                             dtype=torch.int32)
        return rows, lens

    def values(self, n):
        return _slices(self.gen, n, self.mv)

    def zipf(self, n, high, theta=0.99):
        """Ranks in [0, high) (the stored keys are random, so a rank serves as a place)."""
        zetan = float(torch.arange(1, high + 1, device="cuda", dtype=torch.float64).pow(-theta).sum())
        zeta2 = 1.0 + 0.5 ** theta
        eta = (1 - (2.0 / high) ** (1 - theta)) / (1 - zeta2 / zetan)
        u = torch.rand(n, generator=self.gen, device="cuda", dtype=torch.float64)
        r = ((high - 1) * (eta * u - eta + 1).pow(1.0 / (1.0 - theta))).long()
        uz = u * zetan
        r = torch.where(uz < zeta2, torch.ones_like(r), r)
        return torch.where(uz < 1.0, torch.zeros_like(r), r).clamp_(0, high - 1)


def _pick(keys, at):
    rows, lens = keys
    picked = torch.empty((len(at), rows.shape[1]), dtype=rows.dtype, device="cuda")
    for to, part in zip(picked.split(CHUNK), at.split(CHUNK)):
        to.copy_(rows[part])
    return picked, None if lens is None else lens[at]


def _cat(parts):
    rows, lens = zip(*parts)
    return torch.cat(rows), None if lens[0] is None else torch.cat(lens)


def _pool_bytes(case, extra=0):
    words = 1 + case["max_len"] - 1 + case["value_len"]
    slabs = (words + 30) // 31 + 0.25
    if case["prefix"]:
        slabs += 0.05
    return int((case["keys"] + extra) * slabs * 128 * 1.1) + (512 << 20)


def _index(case, extra=0):
    return GpuMasstree(tile_size=16, pool_bytes=_pool_bytes(case, extra))


def _resident(case, k, extra=0):
    """An index holding the case's keys, the keys and their values."""
    index = _index(case, extra)
    keys, values = k.keys(case["keys"]), k.values(case["keys"])
    index.insert(keys[0], k.mk, keys[1], values, k.mv, None, case["keys"])
    return index, keys, values


def _outputs(n, mv):
    return (torch.zeros((n, mv), dtype=torch.int32, device="cuda"),
            torch.zeros(n, dtype=torch.int32, device="cuda"))


def _flags(n):
    return torch.zeros(n, dtype=torch.uint8, device="cuda")


def _mixed_pair(case, k, keys, values, n, taken):
    """Two mixed batches: finds, inserts of fresh keys and erases of stored ones (from
    place `taken` of the end of the stored keys on, which no find of any batch reads),
    then the same finds with the writes the other way round."""
    ni = max(1, n // 20)
    ne = min(max(1, n // 20), case["keys"] // 8)
    nf = max(1, n - ni - ne)
    n = nf + ni + ne
    readable = case["keys"] - case["keys"] // 2
    found = _pick(keys, k.zipf(nf, readable))
    at = case["keys"] - 1 - (taken + torch.arange(ne, device="cuda")) % (case["keys"] // 2)
    old, fresh = _pick(keys, at), k.keys(ni)
    zeros = torch.zeros((nf, k.mv), dtype=torch.int32, device="cuda")
    vals = torch.cat([zeros, k.values(ni), values[at]])
    rows, lens = _cat([found, fresh, old])
    order = torch.randperm(n, generator=k.gen, device="cuda")
    pair = []
    for new, gone in ((REQUEST_INSERT, REQUEST_ERASE), (REQUEST_ERASE, REQUEST_INSERT)):
        types = torch.cat([torch.full((m,), t, dtype=torch.uint8, device="cuda")
                           for m, t in ((nf, REQUEST_FIND), (ni, new), (ne, gone))])
        pair.append(dict(types=types[order].contiguous(), keys=rows[order].contiguous(),
                         lens=None if lens is None else lens[order].contiguous(),
                         values=vals[order].contiguous(),
                         value_lengths=torch.full((n,), k.mv, dtype=torch.int32, device="cuda"),
                         results=_flags(n), n=n))
    return pair, ne


def prepare(case, seed):
    k = _Keys(case, seed)
    kind, n = case["kind"], case.get("batch", 0)
    s = dict(case=case, mk=k.mk, mv=k.mv)
    if kind == "load":
        s["keys"], s["values"] = k.keys(case["keys"]), k.values(case["keys"])
        s["results"] = _flags(case["keys"])
        s["out"] = _outputs(case["keys"], k.mv)
        return s
    if kind == "batched":
        s["index"], keys, values = _resident(case, k, case["batch"] * 2)
        pairs, taken = [], 0
        small = max(100, min(1024, n))
        for b in range(max(1, case["batches"] // 2)):
            size = int(small * (n / small) ** ((b * 0.618034) % 1.0)) if n > small else n
            pair, ne = _mixed_pair(case, k, keys, values, size, taken)
            pairs += pair
            taken += ne
        ends = torch.tensor([0] + [p["n"] for p in pairs]).cumsum(0)
        for name in ("types", "keys", "values", "value_lengths", "results"):
            s[name] = torch.cat([p[name] for p in pairs])
        s["lens"] = None if pairs[0]["lens"] is None else torch.cat([p["lens"] for p in pairs])
        s["offsets"], s["total"], s["batches"] = ends.cuda(), int(ends[-1]), len(pairs)
        return s
    s["index"], keys, values = _resident(case, k, n)
    if kind == "find":
        hits = n // 2
        rows, lens = _cat([_pick(keys, k.index(case["keys"], hits)), k.keys(n - hits)])
        order = torch.randperm(n, generator=k.gen, device="cuda")
        s["keys"], s["out"] = _pick((rows, lens), order), _outputs(n, k.mv)
    elif kind == "churn":
        fresh, other = k.keys(n - n // 10), k.keys(n // 10)
        stored = _pick(keys, k.index(case["keys"], n // 10))
        order = torch.randperm(n, generator=k.gen, device="cuda")
        s["keys"] = _pick(_cat([fresh, stored]), order)
        s["gone"] = _pick(_cat([fresh, other]), torch.randperm(n, generator=k.gen, device="cuda"))
        s["values"], s["results"] = k.values(n), (_flags(n), _flags(n))
    elif kind == "update":
        at = torch.randperm(case["keys"], generator=k.gen, device="cuda")[:n]
        s["keys"], s["values"] = _pick(keys, at), k.values(n)
        s["results"], s["out"] = _flags(n), _outputs(n, k.mv)
    elif kind == "mixed":
        s["pair"], _ = _mixed_pair(case, k, keys, values, n, 0)
    else:
        limit = case["limit"]
        rows, lens = k.keys(n)
        s["lower"] = rows, lens
        s["upper"] = None
        if case["upper"]:
            # a range of about limit / 2 entries, as far as the varying slice has them
            p = case["prefix"]
            step = max(1, int((1 << 31) * limit * (PREFIXES if p else 1) / case["keys"]))
            first = rows[:, p].long() & 0xFFFFFFFF
            up = torch.full_like(rows, -1)
            up[:, :p] = rows[:, :p]
            up[:, p] = (first + step).clamp_(max=0xFFFFFFFF).to(torch.int32)
            s["upper"] = up
        s["limits"] = torch.randint(1, limit + 1, (n,), generator=k.gen, device="cuda",
                                    dtype=torch.int32)
        s["counts"] = torch.zeros(n, dtype=torch.int32, device="cuda")
        s["out"] = _outputs(n * limit, k.mv)
        s["out_keys"] = _outputs(n * limit, k.mk)
    return s


# ------------------------------------------------------------------ one pass
def _find(s, keys, n):
    values, lengths = s["out"]
    s["index"].find(keys[0], s["mk"], keys[1], values, s["mv"], lengths, n,
                    concurrent=s["case"].get("concurrent", False))
    return values, lengths


def run(s):
    case, mk, mv = s["case"], s["mk"], s["mv"]
    kind, n = case["kind"], case.get("batch", 0)
    if kind == "find":
        return _find(s, s["keys"], n)
    if kind == "load":
        n = case["keys"]
        if s.get("index") is not None:
            s["index"].close()
        s["index"] = _index(case)
        s["index"].insert(s["keys"][0], mk, s["keys"][1], s["values"], mv, None, n,
                          results=s["results"])
        return s["results"], _find(s, s["keys"], n)
    index = s["index"]
    if kind == "churn":
        rows, lens = s["keys"]
        index.insert(rows, mk, lens, s["values"], mv, None, n, results=s["results"][0])
        index.erase(s["gone"][0], mk, s["gone"][1], n, results=s["results"][1])
        return s["results"]
    if kind == "update":
        rows, lens = s["keys"]
        if case["upsert"]:
            index.insert(rows, mk, lens, s["values"], mv, None, n, update_if_exists=True,
                         results=s["results"])
        else:
            index.update(rows, mk, lens, s["values"], mv, None, n, results=s["results"])
        return s["results"], _find(s, s["keys"], n)
    if kind == "mixed":
        for b in s["pair"]:
            index.mixed_batch(b["types"], b["keys"], mk, b["lens"], b["values"], mv,
                              b["value_lengths"], b["results"], b["n"])
        return [(b["results"], b["values"], b["value_lengths"]) for b in s["pair"]]
    if kind == "batched":
        index.multi_batch(s["types"], s["keys"], mk, s["lens"], s["values"], mv,
                          s["value_lengths"], s["results"], s["offsets"], s["batches"],
                          s["total"])
        return s["results"], s["values"], s["value_lengths"]
    rows, lens = s["lower"]
    index.scan(rows, lens, mk, case["limit"], n, upper_keys=s["upper"], counts=s["counts"],
               values=s["out"][0], max_value_length=mv, value_lengths=s["out"][1],
               out_keys=s["out_keys"][0], out_key_lengths=s["out_keys"][1],
               per_query_limits=s["limits"])
    return s["counts"], s["out"], s["out_keys"]


# ------------------------------------------------------------------ what it cannot do without
def work(case):
    """Bytes of one pass: the requests' inputs and outputs once, one line of the index for
    a lookup's entry and one (or the record's own bytes) for a stored key's record."""
    mk, mv = case["max_len"], case["value_len"]
    length = (case["min_len"] + mk) / 2
    key = 4 * length + (4 if case["min_len"] != mk else 0)
    record = max(LINE, 4 * (length + mv))

    def finds(n, hits):
        return n * (key + LINE + 4) + hits * (record + 4 * mv)

    def writes(n, values):
        # the entry's line read and written, the record written (or freed), the flag
        return n * (key + 2 * LINE + 1) + (n * (record + 4 * mv) if values else 0)

    kind, n = case["kind"], case.get("batch", 0)
    if kind == "find":
        b = finds(n, n // 2)
    elif kind == "load":
        # a fresh index shares its border lines between about ten entries
        b = case["keys"] * (key + 2 * LINE / 10 + 1 + record + 4 * mv) + finds(case["keys"], case["keys"])
    elif kind == "churn":
        b = writes(n, True) + writes(n, False)
    elif kind == "update":
        b = writes(n, True) + finds(n, n)
    elif kind in ("mixed", "batched"):
        if kind == "batched":
            n = 2 * sum(int(1024 * (n / 1024) ** ((i * 0.618034) % 1.0)) if n > 1024 else n
                        for i in range(max(1, case["batches"] // 2)))
        else:
            n *= 2
        b = finds(0.9 * n, 0.9 * n) + writes(0.05 * n, True) + writes(0.05 * n, False)
    else:
        rows = n * (case["limit"] + 1) / 2
        b = n * (2 * key + LINE + 4) + rows * (record + 4 * (length + mv + 2) + 2 * LINE / 10)
    return dict(bytes=float(b), flops=0.0)
