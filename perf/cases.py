"""Performance cases: what programs have the tree do, over the range of sizes.

A case names one call pattern (`op`), the tree it runs on (`kind`, `width`
pairs per node, `tile` lanes per read tile, `keys` initial keys) and its
sizes. Every pass goes through the public Python API the way a program calls
it: output buffers are kept by the program, the tree is long-lived (except in
`build`), and writes rotate through the program's own key sets, so a pass can
follow any number of others and the tree stays at its size.

  find     n lookups at a snapshot (half present, half uniform draws)
  range    n range queries of about `span` keys at a snapshot
  request  one served request, launch by launch: snapshot, lookups, ranges and
           inserts of n operations (80/10/10), release; a reclamation every
           64 requests
  step     one step of a batch loop: snapshot, `finds` lookups and `ranges`
           ranges at it, `erases` and `inserts`, release, reclaim
  mixed    one concurrent_insert_range (versioned: reads see the state before
           the call) or concurrent_find_erase call, then a reclamation; erased
           keys are inserted again by the next pass
  batches  one run_batches call of `batches` uneven batches (60/20/10/10
           find/insert/erase/range), n operations in all, through the launch
           graph, then the reclamation and the statistics of a served step
  build    a new tree, all keys in one insert (or a bulk build of sorted
           keys), then as many lookups; the old tree is dropped
"""
from __future__ import annotations

import math

import torch

import mvgpubtree_amd as mv

DEV = "cuda:0"
KEY_TOP = 0xFFFFFFFE  # keys are 1 .. KEY_TOP - 1


def listed():
    return [
        # the smallest read a serving program makes: one short lookup list
        {"name": "find_64", "op": "find", "kind": "versioned", "width": 32, "tile": 16, "keys": 1_000_000,
         "n": 64, "span": 0, "concurrent": False},
        # a large lookup batch on a large index
        {"name": "find_1m", "op": "find", "kind": "versioned", "width": 32, "tile": 16, "keys": 40_000_000,
         "n": 1_000_000, "span": 0, "concurrent": False},
        # a large scan batch on a large index
        {"name": "range_500k", "op": "range", "kind": "versioned", "width": 32, "tile": 16, "keys": 40_000_000,
         "n": 500_000, "span": 32, "concurrent": False},
        # one request of an online service, one launch per operation kind
        {"name": "request_1k", "op": "request", "kind": "versioned", "width": 32, "tile": 16, "keys": 4_000_000,
         "n": 1_000, "span": 32},
        # the batch loop of an index under inserts and scans
        {"name": "step_insert_range_1m", "op": "step", "kind": "versioned", "width": 32, "tile": 16,
         "keys": 40_000_000, "finds": 0, "ranges": 500_000, "span": 32, "inserts": 500_000, "erases": 0},
        # the batch loop of an index whose keys expire, at the narrow node and an odd size
        {"name": "step_erase_find_600k", "op": "step", "kind": "versioned", "width": 16, "tile": 16,
         "keys": 10_000_000, "finds": 300_007, "ranges": 0, "span": 0, "inserts": 150_001, "erases": 150_001},
        # the one-launch mixed calls: scans beside inserts, lookups beside erases
        {"name": "mixed_insert_range_200k", "op": "mixed", "kind": "versioned", "width": 32, "tile": 16,
         "keys": 10_000_000, "reads": 100_003, "writes": 99_997, "span": 8, "call": "insert_range"},
        {"name": "mixed_find_erase_1m", "op": "mixed", "kind": "plain", "width": 16, "tile": 16,
         "keys": 40_000_000, "reads": 500_000, "writes": 500_000, "span": 0, "call": "find_erase"},
        # served steps: a few requests, a busy step, and an offline replay
        {"name": "batches_3k", "op": "batches", "kind": "versioned", "width": 32, "tile": 16, "keys": 4_000_000,
         "n": 3_001, "batches": 3, "span": 32},
        {"name": "batches_64k", "op": "batches", "kind": "versioned", "width": 32, "tile": 16, "keys": 10_000_000,
         "n": 65_521, "batches": 24, "span": 32},
        {"name": "batches_4m", "op": "batches", "kind": "versioned", "width": 32, "tile": 16, "keys": 40_000_000,
         "n": 4_000_000, "batches": 480, "span": 64},
        # a new index from random keys
        {"name": "build_1m", "op": "build", "kind": "plain", "width": 16, "tile": 16, "keys": 1_000_000,
         "bulk": False},
    ]


def _log(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))


def draw(rng):
    op = rng.choice(["find", "find", "range", "request", "step", "step", "mixed", "mixed", "batches", "batches",
                     "build"])
    width = rng.choice([16, 32, 32])
    tile = 16 if width == 16 or rng.random() < 0.7 else 32
    keys = _log(rng, 30_000, 40_000_000)
    c = {"op": op, "kind": "versioned", "width": width, "tile": tile, "keys": keys}
    if op in ("find", "range"):
        c["kind"] = rng.choice(["versioned", "versioned", "plain"])
        c["n"] = _log(rng, 1, 1_000_000 if op == "find" else 400_000)
        c["span"] = 0 if op == "find" else rng.choice([4, 8, 32, 50])
        c["concurrent"] = rng.random() < 0.25
    elif op == "request":
        c["n"] = _log(rng, 16, 16_384)
        c["span"] = rng.choice([8, 32])
    elif op == "step":
        w = _log(rng, 100, min(500_000, keys // 8))
        r = _log(rng, 100, 500_000)
        scan = rng.random() < 0.5
        c |= {"finds": 0 if scan else r, "ranges": r if scan else 0, "span": rng.choice([8, 32]) if scan else 0,
              "inserts": w, "erases": rng.choice([0, w])}
    elif op == "mixed":
        c["call"] = rng.choice(["insert_range", "find_erase"])
        # a plain tree's ranges beside inserts may see them or not: lookups of other keys may not
        c["kind"] = "versioned" if c["call"] == "insert_range" else rng.choice(["versioned", "plain"])
        c |= {"reads": _log(rng, 100, 500_000), "writes": _log(rng, 100, min(500_000, keys // 8)),
              "span": rng.choice([8, 32]) if c["call"] == "insert_range" else 0}
    elif op == "batches":
        c["n"] = _log(rng, 500, min(3_000_000, keys))
        c["batches"] = max(1, min(_log(rng, 1, 400), c["n"] // 40))
        c["span"] = rng.choice([16, 32])
    else:
        c["kind"] = rng.choice(["versioned", "plain"])
        c["keys"] = min(keys, _log(rng, 20_000, 4_000_000))
        c["bulk"] = rng.random() < 0.3
    return c


def _sizes(c):
    """Finds, ranges, inserts and erases of one pass."""
    if c["op"] == "find":
        return c["n"], 0, 0, 0
    if c["op"] == "range":
        return 0, c["n"], 0, 0
    if c["op"] == "request":
        r = i = c["n"] // 10
        return c["n"] - r - i, r, i, 0
    if c["op"] == "step":
        return c["finds"], c["ranges"], c["inserts"], c["erases"]
    if c["op"] == "mixed":
        if c["call"] == "insert_range":
            return 0, c["reads"], c["writes"], 0
        return c["reads"], 0, c["writes"], c["writes"]  # erased, and inserted again
    if c["op"] == "batches":
        f = sum(b[0] for b in _batch_sizes(c))
        i = sum(b[1] for b in _batch_sizes(c))
        e = sum(b[2] for b in _batch_sizes(c))
        return f, c["n"] - f - i - e, i, e
    return c["keys"], 0, c["keys"], 0


def _batch_sizes(c):
    """(finds, inserts, erases, ranges) of each batch: sizes spread over a factor of about 2000."""
    nb, n = c["batches"], c["n"]
    weight = [math.exp(7.6 * ((k * 0.6180339887) % 1.0)) for k in range(nb)]
    total, sizes, left = sum(weight), [], n - 8 * nb
    for k in range(nb):
        s = 8 + int(left * weight[k] / total)
        sizes.append(s)
    sizes[0] += n - sum(sizes)
    out = []
    for s in sizes:
        f, i, e = (6 * s) // 10, (2 * s) // 10, s // 10
        out.append((f, i, e, s - f - i - e))
    return out


def work(c):
    """Bytes a pass cannot do without: a lookup its key, result and one 128-byte line of its leaf; a range its
    bounds, its pairs (read and written) and its count; a write its pair and its leaf read and written (and the
    version copy on a versioned tree)."""
    f, r, i, e = _sizes(c)
    node = 8 * c["width"]
    per_write = 8 + 2 * node + (node if c["kind"] == "versioned" else 0)
    if c["op"] == "build":  # a pair's share of a node: nodes are about two thirds full
        return {"bytes": c["keys"] * (8 + 12) + f * (8 + 128), "flops": 0}
    return {"bytes": f * (8 + 128) + r * (12 + 16 * c.get("span", 0)) + (i + e) * per_write, "flops": 0}


# ---- inputs --------------------------------------------------------------------


def _i32(k64):
    """uint32 bit patterns in int32 tensors."""
    return torch.where(k64 >= 2**31, k64 - 2**32, k64).to(torch.int32).contiguous()


def _keys(n, g):
    """n distinct uniform keys in random order (one from each of n equal slices of the key space)."""
    step = (KEY_TOP - 1) // n
    k = torch.arange(n, device=DEV, dtype=torch.int64) * step + 1
    k += torch.randint(0, step, (n,), device=DEV, generator=g)
    return k[torch.randperm(n, device=DEV, generator=g)]


def _values(n, g):
    return torch.randint(0, 2**31 - 1, (n,), device=DEV, generator=g, dtype=torch.int32)


def _lookups(n, present, g, absent=None):
    """Half present keys, half absent ones (or uniform draws, nearly all absent), shuffled."""
    h = n // 2
    hit = present[torch.randint(0, present.numel(), (n - h,), device=DEV, generator=g)]
    miss = torch.randint(1, KEY_TOP, (h,), device=DEV, generator=g) if absent is None else absent[:h]
    return torch.cat([hit, miss])[torch.randperm(n, device=DEV, generator=g)]


def _bounds(n, span, keys, g):
    width = math.ceil(span * KEY_TOP / keys)
    lo = torch.randint(1, KEY_TOP, (n,), device=DEV, generator=g)
    return lo, torch.clamp(lo + width, max=KEY_TOP + 1)


def _tree(c, pool):
    cls = mv.GpuVersionedBTree if c["kind"] == "versioned" else mv.GpuBlinkTree
    t = cls(pool_nodes=pool, node_width=c["width"])
    t.set_read_tile(c["tile"] if c["tile"] < c["width"] else 0)
    return t


def _op_stream(c, sets, present, g):
    """run_batches input: int32 rows {type, key, arg, slot} and offsets. sets = (inserted keys, erased keys)."""
    ins, era = sets
    f, r, i, e = _sizes(c)
    ik, iv = ins, _values(i, g)
    fk = _lookups(f, present, g)
    lo, hi = _bounds(r, c["span"], c["keys"], g)
    rows, offs, at = [], [0], [0, 0, 0, 0]

    def rec(ty, key, arg, slot):
        m = key.numel()
        z = torch.zeros(m, dtype=torch.int32, device=DEV)
        return torch.stack([z + ty, _i32(key), z if arg is None else arg, z if slot is None else slot], 1)

    slots = torch.arange(max(r, 1), dtype=torch.int32, device=DEV)
    every = torch.cat([rec(mv.OP_FIND, fk, None, None), rec(mv.OP_INSERT, ik, iv, None),
                       rec(mv.OP_ERASE, era, None, None), rec(mv.OP_RANGE, lo, _i32(hi), slots[:r])])
    first = [0, f, f + i, f + i + e]
    for nf, ni, ne, nr in _batch_sizes(c):
        part = []
        for q, m in enumerate((nf, ni, ne, nr)):
            part.append(torch.arange(first[q] + at[q], first[q] + at[q] + m, device=DEV))
            at[q] += m
        idx = torch.cat(part)
        rows.append(idx[torch.randperm(idx.numel(), device=DEV, generator=g)])
        offs.append(offs[-1] + idx.numel())
    ops = every[torch.cat(rows)].contiguous()
    return ops, torch.tensor(offs, dtype=torch.int64, device=DEV)


def prepare(case, seed):
    c = case
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    s = {"case": c, "k": 0}
    f, r, i, e = _sizes(c)
    n = c["keys"]
    if c["op"] == "build":
        k = _keys(n, g)
        if c["bulk"]:
            k = torch.sort(k).values
        s["keys"], s["values"] = _i32(k), _values(n, g)
        s["query"] = _i32(_lookups(n, k, g))
        s["out"] = torch.empty(n, dtype=torch.int32, device=DEV)
        s["pool"] = n // (c["width"] // 4) + 4096
        s["tree"] = None
        return s
    # key sets that the passes write: sets[j] are present at the start for j
    # below `here`; a pass inserts one set and erases another
    writes = max(i, e)
    count = 0 if writes == 0 else 2 if c["op"] == "batches" else 64 if c["op"] == "request" else 4
    if c["op"] == "batches":
        i = e = writes
    extra = n // 100 if c["op"] in ("find", "range") and c["kind"] == "versioned" else f if c["op"] == "mixed" else 0
    every = _keys(n + count * writes + extra, g)
    base, sets = every[:n], [every[n + j * writes:n + (j + 1) * writes] for j in range(count)]
    per_node = c["width"] // 4
    copies = (64 if c["op"] == "request" else 2) * 2 * writes
    s["tree"] = t = _tree(c, every.numel() // per_node + copies + extra + (1 << 20))
    start = [base]
    if c["op"] in ("step", "mixed") and e:  # the set the first pass erases
        start.append(sets[0])
    if c["op"] == "batches":
        start.append(sets[0])
    start = torch.cat(start)
    t.insert(_i32(start), _values(start.numel(), g))
    if c["kind"] == "versioned" and c["op"] in ("find", "range"):
        s["snapshot"] = t.take_snapshot()
        late = every[n + count * writes:]
        if extra:  # the index has moved on since the snapshot
            t.insert(_i32(late), _values(extra, g))
    if c["op"] == "batches":
        f, r, i, e = _sizes(c)
        # the writes of pass k undo those of pass k - 1 (as far as they overlap)
        s["ops"], s["offsets"] = zip(*[_op_stream(c, (sets[1 - j][:i], sets[j][:e]), base, g) for j in range(2)])
        L = 4 * c["span"]
        s["results"] = torch.zeros(c["n"], dtype=torch.int32, device=DEV)
        s["pairs"] = torch.full((max(r, 1) * L,), -1, dtype=torch.int64, device=DEV)
        s["stats"] = torch.zeros(8, dtype=torch.int64).pin_memory()
        s["slots"], s["L"] = max(r, 1), L
        t.reserve_batches(c["n"], c["batches"])
        return s
    if f:
        # lookups beside erases name no key that a pass writes: what such a lookup finds is up to the order
        miss = every[n + count * writes:] if c["op"] == "mixed" else None
        s["fk"] = _i32(_lookups(f, base, g, miss))
        s["fo"] = torch.empty(f, dtype=torch.int32, device=DEV)
    if r:
        lo, hi = _bounds(r, c["span"], n, g)
        s["lo"], s["hi"], s["L"] = _i32(lo), _i32(hi), 4 * c["span"]
        s["pairs"] = torch.full((r * s["L"],), -1, dtype=torch.int64, device=DEV)
        s["counts"] = torch.zeros(r, dtype=torch.int32, device=DEV)
    s["sets"] = [_i32(k) for k in sets]
    s["vals"] = [_values(writes, g) for _ in range(count)]
    return s


# ---- one pass ------------------------------------------------------------------


def _reads(s, ts, concurrent=False):
    t, out = s["tree"], {}
    if "fk" in s:
        t.find(s["fk"], s["fo"], timestamp=ts, concurrent=concurrent)
        out["found"] = s["fo"]
    if "lo" in s:
        t.range_query(s["lo"], s["hi"], s["L"], result=s["pairs"], counts=s["counts"], timestamp=ts,
                      concurrent=concurrent)
        out["pairs"], out["counts"] = s["pairs"], s["counts"]
    return out


def run(state):
    s = state
    c, t, k = s["case"], s["tree"], s["k"]
    s["k"] = k + 1
    op = c["op"]
    if op in ("find", "range"):
        return _reads(s, s.get("snapshot", mv.LATEST), c["concurrent"])
    if op == "request":
        ts = t.take_snapshot()
        out = _reads(s, ts)
        if s["sets"]:
            t.insert(s["sets"][k % 64], s["vals"][k % 64])
        t.release_snapshot(ts)
        if k % 64 == 63:
            t.reclaim()
        return out
    if op == "step":
        ts = t.take_snapshot()
        out = _reads(s, ts)
        if c["erases"]:
            t.erase(s["sets"][k % 4])
        t.insert(s["sets"][(k + 1) % 4], s["vals"][(k + 1) % 4])
        t.release_snapshot(ts)
        t.reclaim()
        return out
    if op == "mixed":
        if c["call"] == "insert_range":
            t.concurrent_insert_range(s["sets"][k % 4], s["vals"][k % 4], s["lo"], s["hi"], s["L"],
                                      result=s["pairs"], counts=s["counts"])
            out = {"pairs": s["pairs"], "counts": s["counts"]}
        else:
            t.concurrent_find_erase(s["fk"], s["sets"][k % 4], find_results=s["fo"])
            t.insert(s["sets"][(k + 1) % 4], s["vals"][(k + 1) % 4])
            out = {"found": s["fo"]}
        if c["kind"] == "versioned":
            t.reclaim()
        return out
    if op == "batches":
        j = k % 2
        t.run_batches(s["ops"][j], s["offsets"][j], results=s["results"], pairs=s["pairs"],
                      pair_slots=s["slots"], average_range_length=s["L"], use_graph=True)
        t.reclaim()
        t.memory_stats_async(s["stats"])
        return {"results": s["results"], "pairs": s["pairs"]}
    old = t
    t = s["tree"] = _tree(c, s["pool"])
    if c["bulk"]:
        t.bulk_build(s["keys"], s["values"])
    else:
        t.insert(s["keys"], s["values"])
    t.find(s["query"], s["out"])
    if old is not None:
        old.close()
    return {"found": s["out"]}
