"""GPU parity of the 16-lane reader on plain trees, at the counts where a tile's
groups of walks and the launch's division change, against the sorted state."""
from __future__ import annotations

import numpy as np
import pytest

import mvgpubtree_amd as mv
import oracle
from mvgpubtree_amd import workloads as wl

from conftest import to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nw", [16, 32, 64])
@pytest.mark.parametrize("n", [1, 2, 5, 15, 17, 65, 40_001, 140_003, 530_001])
def test_plain_reads(dev, nw, n):
    rng = np.random.default_rng(nw + n)
    tree = mv.GpuBlinkTree(pool_nodes=1 << 16, node_width=nw)
    tree.set_read_tile(16 if nw > 16 else 0)
    keys = wl.unique_keys(rng, 60_000)
    keys[:2] = (1, 0xFFFFFFFE)
    vals = wl.value_of(keys)
    for part in range(3):  # the first is laid out, the others split its leaves
        a, b = part * 20_000, (part + 1) * 20_000
        tree.insert(to_dev(keys[a:b], dev), to_dev(vals[a:b], dev))
    gone = rng.permutation(60_000)[:9_000]
    tree.erase(to_dev(keys[gone], dev))
    left = np.delete(np.arange(60_000), gone)
    ref = oracle.SortedState(keys[left], vals[left])
    ends = np.array([1, 0xFFFFFFFE, 0, 0xFFFFFFFF], np.uint32)
    q = rng.choice(np.concatenate([keys, keys + np.uint32(1), ends]), size=n)
    assert np.array_equal(to_np(tree.find(to_dev(q, dev))), ref.find(q))
    lo = rng.choice(np.concatenate([keys, ends]), size=n)
    hi = np.minimum(lo.astype(np.uint64) + rng.choice([0, 1, wl.span_for(6, left.size), wl.span_for(40, left.size)],
                                                      size=n).astype(np.uint64), 0xFFFFFFFF).astype(np.uint32)
    cap = 16
    p, c = tree.range_query(to_dev(lo, dev), to_dev(hi, dev), cap)
    rp, rc = ref.range_query(lo, hi, cap)
    assert np.array_equal(to_np(c), rc)
    live = np.arange(cap)[None, :] < np.minimum(rc, cap)[:, None]
    assert np.array_equal(to_np(p, np.uint64).reshape(-1, cap)[live], np.asarray(rp, np.uint64).reshape(-1, cap)[live])
    assert tree.error_flags() & ~mv.FLAG_RANGE_OVERFLOW == 0
    assert tree.validate_tree_structure()[0] == left.size
