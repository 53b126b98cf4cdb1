"""Reclamations issued on two streams with no write between them run one after
the other: no slot is lost, freed twice or handed to two owners."""
from __future__ import annotations

import numpy as np
import pytest

import mvgpubtree_amd as mv
from mvgpubtree_amd import workloads as wl

from conftest import to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [700, 90_000, 400_001])
def test_reclaims_on_two_streams(dev, n):
    import torch
    rng = np.random.default_rng(n)
    keys = wl.unique_keys(rng, max(n, 2_000))
    order = np.argsort(keys)
    vals = wl.value_of(keys)
    tree = mv.GpuVersionedBTree(pool_nodes=keys.size // 4 + 5 * n + (1 << 12))
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    tree.insert(to_dev(keys, dev), to_dev(vals, dev))
    torch.cuda.synchronize()
    live = tree.memory_stats().live_nodes
    cur = vals.copy()
    for k in range(6):
        snaps = []
        for part in range(3):  # three epochs of copies
            snaps.append(tree.take_snapshot(stream=a))
            pick = rng.permutation(keys.size)[:n]
            new = ((keys[pick] ^ np.uint32(k * 31 + part)) & np.uint32(0x7FFFFFFF)).astype(np.uint32)
            dk, dv = to_dev(keys[pick], dev), to_dev(new, dev)
            torch.cuda.synchronize()
            tree.insert(dk, dv, stream=a)
            torch.cuda.synchronize()
            cur[pick] = new
        for s, st in zip(snaps, (a, b, a) if k % 2 else (b, a, b)):  # each frees one epoch's copies
            tree.release_snapshot(s)
            tree.reclaim(stream=st)
        tree.reclaim(stream=b)
        torch.cuda.synchronize()
        m = tree.memory_stats()
        assert m.retired_pending == 0 and m.live_nodes == live
        assert m.live_nodes + m.free_nodes == m.capacity_nodes
        assert m.reclaimed_nodes == m.retired_total
        assert np.array_equal(to_np(tree.find(to_dev(keys[order], dev))), cur[order])
    assert tree.error_flags() == 0
    assert tree.validate_tree_structure()[0] == keys.size
