"""GPU parity of launches whose operations are divided over more tiles: call
sizes at the edges where a tile takes one, two, ... operations, against the
oracle; and repeated keys of one call, of which the last wins in each aligned
group of `node_width` operations."""
from __future__ import annotations

import numpy as np
import pytest

import mvgpubtree_amd as mv
import oracle
from mvgpubtree_amd import workloads as wl

from conftest import to_dev, to_np

pytestmark = pytest.mark.gpu

# (node width, read tile): tiles of 16 lanes are divided over 32768 (finds), tiles of 32 over 16384
SHAPES = [(16, 0), (32, 16), (32, 0), (64, 32)]


@pytest.mark.parametrize("nw,lanes", SHAPES)
@pytest.mark.parametrize("kind", ["versioned", "plain"])
@pytest.mark.parametrize("n", [1, 5, 4097, 6145, 16385, 49999, 140001])
def test_calls_of_every_division(dev, nw, lanes, kind, n):
    rng = np.random.default_rng(n + nw)
    versioned = kind == "versioned"
    tree = (mv.GpuVersionedBTree if versioned else mv.GpuBlinkTree)(pool_nodes=1 << 17, node_width=nw)
    tree.set_read_tile(lanes)
    ref = oracle.MVMap()
    keys = wl.unique_keys(rng, 30_000 + n)
    vals = wl.value_of(keys)
    tree.insert(to_dev(keys[:30_000], dev), to_dev(vals[:30_000], dev))
    ref.insert(keys[:30_000], vals[:30_000])
    snaps = []
    if versioned:
        snaps.append(tree.take_snapshot())
        assert snaps[0] == ref.take_snapshot()
    new = keys[-n:]
    tree.insert(to_dev(new, dev), to_dev(vals[-n:], dev))
    ref.insert(new, vals[-n:])
    gone = rng.permutation(keys)[:n]
    tree.erase(to_dev(gone, dev))
    ref.erase(gone)
    q = rng.choice(keys, size=n)
    lo = rng.integers(1, 0xFFFFFF00, size=n, dtype=np.uint64).astype(np.uint32)
    hi = np.minimum(lo.astype(np.uint64) + wl.span_for(8, keys.size), 0xFFFFFFFE).astype(np.uint32)
    for ts in snaps + [mv.LATEST]:
        for conc in (False, True):
            f = to_np(tree.find(to_dev(q, dev), timestamp=ts, concurrent=conc))
            p, c = tree.range_query(to_dev(lo, dev), to_dev(hi, dev), 32, timestamp=ts, concurrent=conc)
            rp, rc = ref.range_query(lo, hi, 32, ts)
            assert np.array_equal(f, ref.find(q, ts))
            assert np.array_equal(to_np(c), rc)
            assert np.array_equal(to_np(p, np.uint64), rp)
    assert tree.error_flags() == 0
    assert tree.validate_tree_structure()[0] == ref.size()


@pytest.mark.parametrize("nw", [16, 32, 64])
@pytest.mark.parametrize("mixed", [False, True])
def test_last_of_a_repeated_key_wins_within_a_group(dev, nw, mixed):
    rng = np.random.default_rng(nw)
    for n in (2, nw, 4 * nw, 6000, 20_000):
        tree = mv.GpuVersionedBTree(pool_nodes=1 << 16, node_width=nw)
        # every aligned group of nw operations repeats its own few keys
        keys = (rng.integers(0, 5, size=n) + (np.arange(n) // nw) * 5 + 1).astype(np.uint32)
        vals = np.arange(1, n + 1, dtype=np.uint32)
        if mixed:
            none = to_dev(np.empty(0, np.uint32), dev)
            tree.concurrent_insert_range(to_dev(keys, dev), to_dev(vals, dev), none, none, 4)
        else:
            tree.take_snapshot()  # not the first call of an empty tree
            tree.insert(to_dev(keys, dev), to_dev(vals, dev))
        want = {}
        for k, v in zip(keys.tolist(), vals.tolist()):
            want[k] = v
        k = np.array(sorted(want), np.uint32)
        got = to_np(tree.find(to_dev(k, dev)))
        assert np.array_equal(got, np.array([want[x] for x in k.tolist()], np.uint32))
        assert tree.error_flags() == 0


@pytest.mark.parametrize("n", [9_000, 10_400, 10_650, 10_900, 11_800])
def test_insert_that_grows_the_tree_past_the_division_line(dev, n):
    """The tree holds about 3000 nodes, a fraction of four times the call's
    writes, and gains a third of them while the call runs: every wave must
    divide the call the same way."""
    rng = np.random.default_rng(n)
    tree = mv.GpuVersionedBTree(pool_nodes=1 << 16, node_width=16)
    keys = wl.unique_keys(rng, 30_000 + n)
    vals = wl.value_of(keys)
    tree.insert(to_dev(keys[:30_000], dev), to_dev(vals[:30_000], dev))
    tree.insert(to_dev(keys[30_000:], dev), to_dev(vals[30_000:], dev))
    assert np.array_equal(to_np(tree.find(to_dev(keys, dev))), vals)
    assert tree.validate_tree_structure()[0] == keys.size

@pytest.mark.parametrize("nw", [16, 32, 64])
@pytest.mark.parametrize("spare", [200, 30_000])
def test_slots_of_a_workgroup_are_all_accounted_for(dev, nw, spare):
    """Updates that copy every leaf, no leaf twice, and absent keys that copy
    none: after reclamation the pool holds the tree's nodes and nothing else,
    both where the pool allows the workgroups' reservations (spare well above
    three slots a write) and where it does not."""
    rng = np.random.default_rng(nw + spare)
    keys = wl.unique_keys(rng, 60_000)
    probe = mv.GpuVersionedBTree(pool_nodes=1 << 16, node_width=nw)
    probe.bulk_build(to_dev(np.sort(keys), dev), to_dev(wl.value_of(np.sort(keys)), dev))
    nodes = probe.memory_stats().live_nodes
    tree = mv.GpuVersionedBTree(pool_nodes=nodes + spare, node_width=nw)
    ks = np.sort(keys)
    tree.bulk_build(to_dev(ks, dev), to_dev(wl.value_of(ks), dev))
    absent = wl.absent_keys(rng, 3000, ks)
    for r in range(6):
        s = tree.take_snapshot()
        some = rng.choice(ks, size=150, replace=False)
        tree.insert(to_dev(some, dev), to_dev(np.full(150, r + 1, np.uint32), dev))
        tree.erase(to_dev(absent, dev))  # copies nothing
        tree.release_snapshot(s)
        tree.reclaim()
        assert np.all(to_np(tree.find(to_dev(some, dev))) == r + 1)
        assert tree.error_flags() == 0
        m = tree.memory_stats()
        assert m.live_nodes == nodes and m.retired_pending == 0
    assert tree.validate_tree_structure()[0] == ks.size
