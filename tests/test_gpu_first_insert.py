"""GPU parity of a tree's first insert, which sorts its pairs and lays the
nodes out: sizes at the edges of a leaf, of a level and of the sort's
segments, repeated and reserved keys, pools with and without room for the
sort, later writes, a snapshot and a write on another stream right behind it,
and concurrent readers beside it."""
from __future__ import annotations

import numpy as np
import pytest

import mvgpubtree_amd as mv
import oracle
from mvgpubtree_amd import workloads as wl

from conftest import to_dev, to_np

pytestmark = pytest.mark.gpu

KINDS = {"versioned": mv.GpuVersionedBTree, "plain": mv.GpuBlinkTree}


def check(tree, keys, vals, dev, extra=None):
    ks = np.sort(keys)
    order = np.argsort(keys)
    f = to_np(tree.find(to_dev(keys, dev)))
    assert np.array_equal(f, vals)
    if extra is not None:
        assert np.all(to_np(tree.find(to_dev(extra, dev))) == mv.NOT_FOUND)
    assert tree.validate_tree_structure()[0] == keys.size
    ex = tree.export()
    assert np.array_equal((ex & 0xFFFFFFFF).astype(np.uint32), ks)
    assert np.array_equal((ex >> 32).astype(np.uint32), vals[order])


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("nw", [16, 32, 64])
@pytest.mark.parametrize("n", [63, 64, 65, 140, 511, 513, 4001, 131073, 300007])
def test_sizes(dev, kind, nw, n):
    rng = np.random.default_rng(n + nw)
    keys = wl.unique_keys(rng, n + 5000)
    if n > 100:  # both ends of the key space
        keys[:2] = [1, 0xFFFFFFFE]
        keys = np.unique(keys)
        keys = keys[rng.permutation(keys.size)]
    new, keys = keys[n:], keys[:n]
    tree = KINDS[kind](pool_nodes=n // (nw // 4) + 40_000, node_width=nw)
    tree.insert(to_dev(keys, dev), to_dev(wl.value_of(keys), dev))
    assert tree.error_flags() == 0
    st = tree.memory_stats()
    assert st.live_nodes + st.free_nodes == st.capacity_nodes and st.retired_total == 0
    check(tree, keys, wl.value_of(keys), dev, extra=new)
    # the tree goes on like any other
    tree.insert(to_dev(new, dev), to_dev(wl.value_of(new), dev))
    gone = keys[: n // 3]
    tree.erase(to_dev(gone, dev))
    left = np.concatenate([keys[n // 3:], new])
    assert tree.error_flags() == 0
    check(tree, left, wl.value_of(left), dev, extra=gone)


@pytest.mark.parametrize("kind", KINDS)
def test_repeated_and_reserved_keys(dev, kind):
    rng = np.random.default_rng(3)
    n = 20_000
    keys = rng.integers(1, 6000, size=n, dtype=np.uint32)
    keys[rng.permutation(n)[:50]] = 0
    keys[rng.permutation(n)[:50]] = 0xFFFFFFFF
    vals = np.arange(1, n + 1, dtype=np.uint32)
    tree = KINDS[kind](pool_nodes=1 << 15)
    tree.insert(to_dev(keys, dev), to_dev(vals, dev))
    assert tree.error_flags() == mv.FLAG_INVALID_KEY
    want = {k: v for k, v in zip(keys.tolist(), vals.tolist()) if k not in (0, 0xFFFFFFFF)}
    k = np.array(sorted(want), np.uint32)
    check(tree, k, np.array([want[x] for x in k.tolist()], np.uint32), dev)
    only = KINDS[kind](pool_nodes=1 << 12)
    only.insert(to_dev(np.zeros(100, np.uint32), dev), to_dev(vals[:100], dev))
    assert only.error_flags() == mv.FLAG_INVALID_KEY and only.validate_tree_structure()[0] == 0
    only.insert(to_dev(k[:10], dev), to_dev(k[:10], dev))
    assert np.array_equal(to_np(only.find(to_dev(k[:10], dev))), k[:10])


@pytest.mark.parametrize("kind", KINDS)
def test_pool_without_room_for_the_sort(dev, kind):
    """16 bytes a key of scratch do not fit behind the nodes: the keys go in one by one."""
    rng = np.random.default_rng(4)
    keys = wl.unique_keys(rng, 20_000)
    tree = KINDS[kind](pool_nodes=4500)
    tree.insert(to_dev(keys, dev), to_dev(wl.value_of(keys), dev))
    assert tree.error_flags() == 0
    check(tree, keys, wl.value_of(keys), dev)


def test_streams_behind_the_first_insert(dev):
    """A snapshot on a second stream and a write on a third, unordered with the
    first insert by the caller: the snapshot sees all of it or none, the write
    is kept, and nothing of it shows at the snapshot."""
    import torch
    rng = np.random.default_rng(5)
    n = 400_000
    keys = wl.unique_keys(rng, n + 1000)
    dk, dv = to_dev(keys[:n], dev), to_dev(wl.value_of(keys[:n]), dev)
    wk, wv = to_dev(keys[n:], dev), to_dev(wl.value_of(keys[n:]), dev)
    a, b, c = torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(3):
        tree = mv.GpuVersionedBTree(pool_nodes=1 << 18)
        torch.cuda.synchronize()
        tree.insert(dk, dv, stream=a)
        s = tree.take_snapshot(stream=b)
        with torch.cuda.stream(b):
            at_s = tree.find(dk, timestamp=s, stream=b, concurrent=True)
        tree.insert(wk, wv, stream=c)
        torch.cuda.synchronize()
        got = to_np(at_s)
        assert np.array_equal(got, wl.value_of(keys[:n])) or np.all(got == mv.NOT_FOUND)
        assert np.all(to_np(tree.find(wk, timestamp=s)) == mv.NOT_FOUND)
        assert np.array_equal(to_np(tree.find(to_dev(keys, dev))), wl.value_of(keys))
        assert tree.error_flags() == 0
        assert tree.validate_tree_structure()[0] == keys.size


@pytest.mark.parametrize("kind", KINDS)
def test_concurrent_readers_beside_the_first_insert(dev, kind):
    import torch
    rng = np.random.default_rng(6)
    n = 300_000
    keys = wl.unique_keys(rng, n)
    vals = wl.value_of(keys)
    dk, dv = to_dev(keys, dev), to_dev(vals, dev)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    tree = KINDS[kind](pool_nodes=1 << 18)
    q, want = dk[:3000].contiguous(), vals[:3000]  # they all lock the one leaf of the empty tree
    outs = [torch.zeros(3000, dtype=torch.int32, device=dev) for _ in range(6)]
    torch.cuda.synchronize()
    for i, o in enumerate(outs):
        if i == 1:
            tree.insert(dk, dv, stream=a)
        tree.find(q, o, stream=b, concurrent=True)
    torch.cuda.synchronize()
    for o in outs:  # each key: its value, or not there yet
        got = to_np(o)
        assert np.all((got == want) | (got == mv.NOT_FOUND))
    assert tree.error_flags() == 0
    check(tree, keys, vals, dev)


def test_captured_first_insert_is_not_laid_out(dev):
    """Under capture the call keeps to launches a replay may repeat: a replay inserts the keys again."""
    import torch
    rng = np.random.default_rng(7)
    keys = wl.unique_keys(rng, 9000)
    tree = mv.GpuBlinkTree(pool_nodes=1 << 15)
    dk, dv = to_dev(keys[:5000], dev), to_dev(wl.value_of(keys[:5000]), dev)
    more = to_dev(keys[5000:], dev), to_dev(wl.value_of(keys[5000:]), dev)
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        tree.insert(dk, dv, stream=s)
    g.replay()
    torch.cuda.synchronize()
    tree.insert(*more)
    torch.cuda.synchronize()
    for _ in range(2):
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(to_np(tree.find(to_dev(keys, dev))), wl.value_of(keys))
    assert tree.validate_tree_structure()[0] == keys.size
