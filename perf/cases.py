"""The calls that programs using this library make, as measurable cases.

A case is a dict of plain values.  `path` says which calls it makes:

  upload_ids     upload_from_ids (host ids) or upload_from_device_ids
  upload_bitset  upload_from_device_bitset
  set_op         set_operation of two bitmaps
  multi_and      multi_and of several predicates
  contains       contains_batch, a batch of point queries
  decode         enumerate_ids or decompress_to_bitset
  topk           topk_filtered, the bitmap-gated brute-force search

A new bitmap's outputs are its arrays where the inputs fix how many containers
it holds.  Where they do not (sparse or clustered ids, intersections, compressed
operands), the pass goes on to decompress_to_bitset, the flat bitset that a
search takes, and that is its output.

Inputs are made on the GPU from the seed alone.  Bitmaps that a path reads are
uploads; compressed ones (`layout` "keep": array, bitmap and run containers as
the portable format chooses them) are loaded from portable-format bytes, as a
program with stored filters does.  A result bitmap is freed when the next pass
on the same state starts, as a program that builds one filter per request does.
"""
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "cu-roaring-bitmap_amd", "python"))

import curoaring as cr  # noqa: E402

OPS = {"and": cr.AND, "or": cr.OR, "andnot": cr.ANDNOT, "xor": cr.XOR}
MODES = {"contains": cr.QUERY_CONTAINS, "wavefront": cr.QUERY_WAVEFRONT, "partitioned": cr.QUERY_PARTITIONED}


def listed():
    return [
        # A tag held by a thousand of 1.5M items, from the program's own list of ids.
        {"name": "upload_ids_1k", "path": "upload_ids", "ids": "uniform", "n": 1000, "universe": 1_500_000, "host": True},
        # The benchmark's headline: an index over 2^30 rebuilt from 100M unsorted device ids, about 10% duplicates.
        {"name": "upload_ids_100m", "path": "upload_ids", "ids": "uniform", "n": 100_000_000, "universe": 1 << 30,
         "host": False},
        # A mask computed on the GPU over 10^9 rows, 70% set: stored as its complement.
        {"name": "upload_bitset_1e9", "path": "upload_bitset", "universe": 1_000_000_000, "density": 0.7},
        # Two filters of a 16M-row collection joined for one request: small, so latency counts.
        {"name": "set_op_16m_or", "path": "set_op", "layout": "bitmap", "universe": 1 << 24, "a": "uniform",
         "a_density": 0.01, "b": "uniform", "b_density": 0.1, "op": "or"},
        # A sparse stored filter less a run-heavy one (deleted ranges) at 2^30, handed to a search as a flat bitset.
        {"name": "set_op_mixed_andnot", "path": "set_op", "layout": "keep", "universe": 1 << 30, "a": "uniform",
         "a_density": 0.001, "b": "runs", "b_density": 0.2, "op": "andnot"},
        # Eight attribute predicates over 2^30 rows combined into one filter.
        {"name": "multi_and_8", "path": "multi_and", "universe": 1 << 30, "count": 8, "density": 0.5},
        # A batch of candidate ids checked against a compressed stored filter, in the default mode.
        {"name": "contains_1m_keep", "path": "contains", "layout": "keep", "universe": 1 << 30, "kind": "uniform",
         "density": 0.01, "n": 1_000_003, "order": "uniform", "mode": "contains"},
        # A join's 100M random probes of an all-bitmap filter.
        {"name": "contains_100m", "path": "contains", "layout": "bitmap", "universe": 1 << 30, "kind": "uniform",
         "density": 0.1, "n": 100_000_000, "order": "uniform", "mode": "partitioned"},
        # A filter handed on as its sorted row numbers.
        {"name": "enumerate_100m", "path": "decode", "layout": "bitmap", "universe": 1 << 30, "kind": "uniform",
         "density": 0.1, "to": "ids"},
        # The benchmark's search: 10M x 128 vectors, 1024 queries, a 10% filter.
        {"name": "topk_10m_10pct", "path": "topk", "n_base": 10_000_000, "dim": 128, "n_q": 1024, "k": 10,
         "selectivity": 0.1},
        # A selective filter (about 10K rows pass) and a deep result list, 96 dimensions.
        {"name": "topk_1m_1pct_k100", "path": "topk", "n_base": 1_000_003, "dim": 96, "n_q": 1000, "k": 100,
         "selectivity": 0.01},
        # An unfiltered search of a mid-size collection with a small batch of queries, 100 dimensions.
        {"name": "topk_300k_q64", "path": "topk", "n_base": 300_007, "dim": 100, "n_q": 64, "k": 10, "selectivity": 1.0},
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def _density(rng, lo, hi):
    return round(lo * (hi / lo) ** rng.random(), 5)


def draw(rng):
    """One more case: universes of 10^5 to 2^30, 10^3 to 10^8 ids or queries, 10^4 to 10^7 vectors."""
    path = rng.choice(["upload_ids", "upload_bitset", "set_op", "multi_and", "contains", "decode", "topk", "topk"])
    universe = _log_uniform(rng, 100_000, 1 << 30)
    if path == "upload_ids":
        n = _log_uniform(rng, 1000, 100_000_000)
        return {"path": path, "ids": rng.choice(["uniform", "uniform", "clustered", "sorted"]), "n": n,
                "universe": max(universe, 1 << 20, min(1 << 30, 4 * n)), "host": n <= 1_000_000 and rng.random() < 0.5}
    if universe % 65536 < 4096:  # a last key wide enough to hold values whatever the seed
        universe = min(1 << 30, universe + 4096)
    if path == "upload_bitset":
        return {"path": path, "universe": universe, "density": _density(rng, 0.001, 0.95)}
    if path == "set_op":
        return {"path": path, "layout": rng.choice(["bitmap", "keep"]), "universe": max(universe, 1 << 20),
                "a": rng.choice(["uniform", "runs"]), "a_density": _density(rng, 0.002, 0.45),
                "b": rng.choice(["uniform", "runs"]), "b_density": _density(rng, 0.002, 0.45),
                "op": rng.choice(sorted(OPS))}
    if path == "multi_and":
        return {"path": path, "universe": universe, "count": rng.randint(2, 8), "density": _density(rng, 0.1, 0.9)}
    kind = rng.choice(["uniform", "runs"])
    if path == "contains":
        mode = rng.choice(sorted(MODES))
        return {"path": path, "layout": rng.choice(["bitmap", "keep"]), "universe": max(universe, 1 << 20), "kind": kind,
                "density": _density(rng, 0.0005, 0.45),
                "n": _log_uniform(rng, 1000, 100_000_000 if mode == "partitioned" else 10_000_000),
                "order": rng.choice(["uniform", "clustered"]), "mode": mode}
    if path == "decode":
        return {"path": path, "layout": rng.choice(["bitmap", "keep"]), "universe": max(universe, 1 << 20), "kind": kind,
                "density": _density(rng, 0.0005, 0.2), "to": rng.choice(["ids", "bitset"])}
    n_base = _log_uniform(rng, 10_000, 10_000_000)
    selectivity = rng.choice([1.0, _density(rng, 0.001, 0.9)])
    dim = rng.choice([32, 64, 96, 100, 128, rng.randint(17, 128)])
    # at most the largest listed search's rows x queries x dimensions
    most = int(1_000_000 * 1024 * 128 / (n_base * selectivity * dim))
    return {"path": path, "n_base": n_base, "dim": dim, "n_q": max(1, min(_log_uniform(rng, 1, 1024), most)),
            "k": _log_uniform(rng, 1, 200), "selectivity": selectivity}


# ---- inputs ------------------------------------------------------------------
class Bitmap:
    """Owns a device bitmap: freed when replaced or dropped."""

    def __init__(self, g):
        self.g = g

    def free(self):
        if self.g is not None:
            cr.free_async(self.g)
            self.g = None

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass


class _Mem:
    def __init__(self, ptr, n, typestr):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (ptr, False), "version": 2}


class Views:
    """Tensors over the library's device memory, one made for each address and length."""

    def __init__(self):
        self.made = {}

    def of(self, ptr, n, typestr):
        if not ptr or not n:
            return 0
        key = (ptr, n, typestr)
        t = self.made.get(key)
        if t is None:
            t = self.made[key] = torch.as_tensor(_Mem(ptr, n, typestr), device="cuda")
        return t

    def bitmap(self, g):
        n = g.n_containers
        return {"n": n, "cardinality": g.total_cardinality, "universe": g.universe_size, "negated": g.negated,
                "keys": self.of(g.keys, n, "<i2"), "types": self.of(g.types, n, "|u1"),
                "offsets": self.of(g.offsets, n, "<i4"), "cards": self.of(g.cardinalities, n, "<i2"),
                "index": self.of(g.key_index, g.max_key + 1, "<i2"),
                "bitmaps": self.of(g.bitmap_data, 1024 * g.n_bitmap_containers, "<i8"),
                "arrays": self.of(g.array_data, g.array_pool_bytes // 2, "<i2"),
                "runs": self.of(g.run_data, g.run_pool_bytes // 2, "<i2")}


def _generator(seed, part=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 64 + part)
    return g


def _cut(words, universe):
    """Clears the bits of the last word past the universe."""
    if universe % 32:
        words[-1] &= (1 << (universe % 32)) - 1
    return words


def _random_words(universe, density, g):
    """A flat bitset (int32 words), each bit set with probability `density` (to 1/65536): the binary digits of the
    density, lowest first, OR or AND a fresh random word in."""
    n = (universe + 31) // 32
    p = max(1, min(65535, round(density * 65536)))
    words = torch.zeros((n + 1) // 2, device="cuda", dtype=torch.int64)
    low = (p & -p).bit_length() - 1
    for b in range(low, 16):
        r = torch.randint(-(1 << 63), (1 << 63) - 1, words.shape, device="cuda", generator=g, dtype=torch.int64)
        words = words | r if (p >> b) & 1 else words & r
    return _cut(words.view(torch.int32)[:n].clone(), universe)


def _run_words(universe, coverage, g):
    """A flat bitset of runs of 1000 to 65535 set bits, with gaps that leave `coverage` of the universe set."""
    n = (universe + 31) // 32
    count = int(universe * coverage / 33_000) + 2
    length = torch.randint(1000, 65536, (count,), device="cuda", generator=g)
    gap = 64 + (torch.rand(count, device="cuda", generator=g) * 2 * 33_268 * (1 - coverage) / coverage).to(torch.int64)
    gap[0] = 64  # so that the smallest universes hold a run too
    end = torch.cumsum(length + gap, 0)
    start = end - length
    keep = end < universe - 64
    start, end = start[keep], end[keep]
    first, last = start >> 5, end >> 5  # the words that hold a run's first bit and the bit after its last
    step = torch.zeros(n + 1, device="cuda", dtype=torch.int32)
    step[first + 1] += 1
    step[last] -= 1  # a run spans over 30 words and gaps over one, so neither index repeats
    words = -torch.cumsum(step[:n], 0).to(torch.int32)  # whole words inside runs: all ones
    ones = torch.full_like(start, 0xFFFFFFFF)
    words[first] |= ((ones << (start & 31)) & 0xFFFFFFFF).to(torch.int32)
    words[last] |= ((1 << (end & 31)) - 1).to(torch.int32)
    return words


def _words(kind, universe, density, g):
    return _run_words(universe, density, g) if kind == "runs" else _random_words(universe, density, g)


def _bitmap(kind, universe, density, layout, g):
    b = Bitmap(cr.upload_from_device_bitset(_words(kind, universe, density, g), universe))
    if layout == "bitmap":
        return b
    stored = cr.portable_serialize(b.g)
    b.free()
    return Bitmap(cr.portable_deserialize(stored, universe, cr.PROMOTE_KEEP_DEFAULT))


def _ids(order, n, universe, g):
    if order == "clustered":  # runs of 1000 to 65535 consecutive ids, shuffled
        count = n // 33_000 + 2
        longest = min(65536, universe // 2)
        length = torch.randint(1000, longest, (count,), device="cuda", generator=g)
        start = torch.randint(0, universe - longest, (count,), device="cuda", generator=g)
        owner = torch.repeat_interleave(torch.arange(count, device="cuda"), length)
        first = (torch.cumsum(length, 0) - length)[owner]
        ids = start[owner] + torch.arange(owner.numel(), device="cuda") - first
        ids = ids[torch.randint(0, ids.numel(), (n,), device="cuda", generator=g)]
    else:
        ids = torch.randint(0, universe, (n,), device="cuda", generator=g)
        again = torch.randint(0, n, (n,), device="cuda", generator=g)
        ids = torch.where(torch.rand(n, device="cuda", generator=g) < 0.1, ids[again], ids)  # about 10% repeats
    if order == "sorted":
        ids = torch.sort(ids)[0]
    return ids.to(torch.int32)


def _queries(order, n, universe, g):
    if order == "clustered":  # groups of 4096 in one 65536-wide window each, sorted
        groups = (n + 4095) // 4096
        window = torch.randint(0, max(1, universe >> 16), (groups, 1), device="cuda", generator=g)
        at = torch.randint(0, min(65536, universe), (groups, 4096), device="cuda", generator=g)
        return ((window << 16) + torch.sort(at, 1)[0]).reshape(-1)[:n].to(torch.int32).contiguous()
    return torch.randint(0, universe, (n,), device="cuda", generator=g).to(torch.int32)


def _to_flat(case):
    """Whether the number of containers that a pass makes depends on the seed."""
    if case["path"] == "set_op":
        return case["layout"] == "keep" or case["op"] not in ("or", "xor") or "runs" in (case["a"], case["b"])
    if case["path"] != "upload_ids":
        return False
    tail = case["universe"] % 65536 or 65536
    return case["ids"] == "clustered" or case["n"] * tail < 20 * case["universe"]


def prepare(case, seed):
    path, g = case["path"], _generator(seed)
    s = {"case": case, "views": Views(), "result": None}
    if path == "upload_ids":
        ids = _ids(case["ids"], case["n"], case["universe"], g)
        s["ids"] = ids.cpu().numpy().view("uint32") if case["host"] else ids
    elif path == "upload_bitset":
        s["words"] = _random_words(case["universe"], case["density"], g)
    elif path == "set_op":
        s["a"] = _bitmap(case["a"], case["universe"], case["a_density"], case["layout"], g)
        s["b"] = _bitmap(case["b"], case["universe"], case["b_density"], case["layout"], _generator(seed, 1))
    elif path == "multi_and":
        s["inputs"] = [_bitmap("uniform", case["universe"], case["density"], "bitmap", _generator(seed, i))
                       for i in range(case["count"])]
    elif path == "contains":
        s["bitmap"] = _bitmap(case["kind"], case["universe"], case["density"], case["layout"], g)
        s["ids"] = _queries(case["order"], case["n"], case["universe"], g)
        s["out"] = torch.empty_like(s["ids"])
    elif path == "decode":
        s["bitmap"] = _bitmap(case["kind"], case["universe"], case["density"], case["layout"], g)
        if case["to"] == "ids":  # room for any filter of this kind
            room = min(case["universe"], int(1.2 * case["universe"] * case["density"]) + 200_000)
            s["out"] = torch.full((room,), -1, device="cuda", dtype=torch.int64)
        else:
            s["out"] = torch.empty((case["universe"] + 31) // 32, device="cuda", dtype=torch.int32)
    elif path == "topk":
        s["base"] = torch.randn(case["n_base"], case["dim"], device="cuda", generator=g)
        s["queries"] = torch.randn(case["n_q"], case["dim"], device="cuda", generator=g)
        s["dist"] = torch.empty(case["n_q"], case["k"], device="cuda")
        s["ids"] = torch.empty(case["n_q"], case["k"], device="cuda", dtype=torch.int64)
        s["filter"] = None
        if case["selectivity"] < 1:
            s["filter"] = _bitmap("uniform", case["n_base"], case["selectivity"], "bitmap", _generator(seed, 1))
    if _to_flat(case):
        s["flat"] = torch.empty((case["universe"] + 31) // 32, device="cuda", dtype=torch.int32)
    return s


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "contains":
        cr.contains_batch(state["bitmap"].g, state["ids"], state["out"], MODES[case["mode"]])
        return state["out"]
    if path == "decode":
        if case["to"] == "ids":
            cr.enumerate_ids(state["bitmap"].g, state["out"], state["out"].numel())
        else:
            cr.decompress_to_bitset(state["bitmap"].g, state["out"])
        return state["out"]
    if path == "topk":
        f = state["filter"]
        cr.topk_filtered(state["base"], state["queries"], case["k"], f.g if f else None, state["dist"], state["ids"])
        return {"dist": state["dist"], "ids": state["ids"]}
    if state["result"] is not None:
        state["result"].free()
    if path == "upload_ids":
        upload = cr.upload_from_ids if case["host"] else cr.upload_from_device_ids
        r = upload(state["ids"], case["universe"])
    elif path == "upload_bitset":
        r = cr.upload_from_device_bitset(state["words"], case["universe"])
    elif path == "multi_and":
        r = cr.multi_and([b.g for b in state["inputs"]])
    else:
        r = cr.set_operation(state["a"].g, state["b"].g, OPS[case["op"]])
    state["result"] = Bitmap(r)
    if "flat" in state:
        cr.decompress_to_bitset(r, state["flat"])
        return {"cardinality": r.total_cardinality, "negated": r.negated, "flat": state["flat"]}
    return state["views"].bitmap(r)


# ---- what a pass cannot do without ---------------------------------------------
def _stored_bytes(kind, universe, density, layout):
    """Container payloads and 9 bytes of metadata each, of a bitmap of this kind."""
    keys = (universe + 65535) // 65536
    if layout == "bitmap":
        return 8201 * keys
    if kind == "runs":
        return 4 * int(universe * density / 33_268 + 2) + 9 * keys
    return (min(8192, 2 * int(65536 * density)) + 9) * keys


def work(case):
    path = case["path"]
    if path == "topk":
        rows = int(case["n_base"] * case["selectivity"])
        filt = case["n_base"] // 8 if case["selectivity"] < 1 else 0
        return {"bytes": 4 * case["dim"] * (rows + case["n_q"]) + filt + 12 * case["n_q"] * case["k"],
                "flops": 2 * rows * case["n_q"] * case["dim"]}
    universe = case["universe"]
    keys = (universe + 65535) // 65536
    if path == "upload_ids":
        if _to_flat(case):
            return {"bytes": 4 * case["n"] + universe // 8, "flops": 0}
        return {"bytes": 4 * case["n"] + 8201 * keys + 2 * keys, "flops": 0}
    if path == "upload_bitset":
        return {"bytes": universe // 8 + 8201 * keys + 2 * keys, "flops": 0}
    if path == "multi_and":
        return {"bytes": 8201 * keys * (case["count"] + 1) + 2 * keys, "flops": 0}
    if path == "set_op":
        read = [_stored_bytes(case[x], universe, case[x + "_density"], case["layout"]) for x in "ab"]
        return {"bytes": sum(read) + (universe // 8 if _to_flat(case) else 8201 * keys), "flops": 0}
    held = _stored_bytes(case["kind"], universe, case["density"], case["layout"])
    if path == "contains":
        return {"bytes": 8 * case["n"] + min(held, 8 * case["n"]), "flops": 0}
    return {"bytes": held + (8 * int(universe * case["density"]) if case["to"] == "ids" else universe // 8), "flops": 0}


def tolerance(case):
    """Bitmaps, answers and ids are exact.  A search's distances are fp32 sums of at most 128 squares; two rows whose
    distances agree to that precision may change places."""
    if case["path"] != "topk":
        return "exact"
    return {"rel": 1e-6, "max": 4e-6, "differ": 2e-3}


def exact(case, seed):
    """A search's distances in 64 bits; the other paths' outputs are whole numbers."""
    if case["path"] != "topk":
        return None
    g = _generator(seed)
    base = torch.randn(case["n_base"], case["dim"], device="cuda", generator=g)
    queries = torch.randn(case["n_q"], case["dim"], device="cuda", generator=g).double()
    rows = None
    if case["selectivity"] < 1:
        words = _random_words(case["n_base"], case["selectivity"], _generator(seed, 1))
        bits = (words[:, None] >> torch.arange(32, device="cuda", dtype=torch.int32)) & 1
        rows = torch.nonzero(bits.reshape(-1)[:case["n_base"]])[:, 0]
    n, k, best = base.shape[0] if rows is None else rows.numel(), case["k"], None
    for at in range(0, n, 1 << 17):
        x = (base[at:at + (1 << 17)] if rows is None else base[rows[at:at + (1 << 17)]]).double()
        d = (queries * queries).sum(1)[:, None] + (x * x).sum(1)[None, :] - 2 * queries @ x.t().contiguous()
        d = d if best is None else torch.cat([best, d], 1)
        best = torch.topk(d, min(k, d.shape[1]), dim=1, largest=False, sorted=True)[0]
    if best is None:
        best = torch.zeros(case["n_q"], 0, device="cuda", dtype=torch.float64)
    if best.shape[1] < k:
        best = torch.cat([best, torch.full((case["n_q"], k - best.shape[1]), float("inf"), device="cuda").double()], 1)
    return {"dist": best, "ids": None}
