"""Reclamation in one launch: entry counts around its workgroups' and threads'
shares, a ring that wraps, parked slots merged with freed copies, and no slot
lost or handed out twice."""
from __future__ import annotations

import numpy as np
import pytest

import mvgpubtree_amd as mv
from mvgpubtree_amd import workloads as wl

from conftest import to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 1_025, 65_537, 120_000, 600_001])
def test_rounds_of_updates_and_reclamations(dev, n):
    rng = np.random.default_rng(n)
    size = max(3 * n // 2, 2_000)
    pool = size // 5 + 2 * n + (1 << 12)
    tree = mv.GpuVersionedBTree(pool_nodes=pool)
    keys = wl.unique_keys(rng, size)
    vals = wl.value_of(keys)
    tree.insert(to_dev(keys, dev), to_dev(vals, dev))
    order = np.argsort(keys)
    cur = vals.copy()
    live = tree.memory_stats().live_nodes
    for k in range(5):  # more entries than the ring holds: it wraps
        snap = tree.take_snapshot()
        pick = rng.permutation(size)[:n]
        new = ((keys[pick] ^ np.uint32(k * 77 + 5)) & np.uint32(0x7FFFFFFF)).astype(np.uint32)
        tree.insert(to_dev(keys[pick], dev), to_dev(new, dev))
        before = tree.memory_stats()
        assert before.retired_pending > 0
        cur[pick] = new
        tree.release_snapshot(snap)
        tree.reclaim()
        st = tree.memory_stats()
        assert st.retired_pending == 0 and st.live_nodes == live
        assert st.live_nodes + st.free_nodes == st.capacity_nodes
        assert st.reclaimed_nodes == before.retired_total
        assert np.array_equal(to_np(tree.find(to_dev(keys[order], dev))), cur[order])
    assert tree.error_flags() == 0
    assert tree.validate_tree_structure()[0] == size
