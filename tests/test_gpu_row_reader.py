"""GPU parity of the 16-lane reader of quiescent launches (one, two and four walks
of a tile in flight; one, two and four pairs a lane) against the oracle: counts
at the edges of its groups and tiles, version chains, and the extremes of keys
and bounds."""
from __future__ import annotations

import numpy as np
import pytest

import mvgpubtree_amd as mv
import oracle
from mvgpubtree_amd import workloads as wl

from conftest import to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nw", [16, 32, 64])
@pytest.mark.parametrize("n", [1, 3, 15, 17, 63, 65, 40_001, 200_003, 530_001])
def test_reads_through_version_chains(dev, nw, n):
    rng = np.random.default_rng(nw + n)
    tree = mv.GpuVersionedBTree(pool_nodes=1 << 17, node_width=nw)
    tree.set_read_tile(16 if nw > 16 else 0)
    ref = oracle.MVMap()
    keys = wl.unique_keys(rng, 20_000)
    keys[:2] = (1, 0xFFFFFFFE)
    stamps = []
    for part in range(4):
        some = rng.permutation(keys)[: 9_000]
        vals = (some * np.uint32(7) + np.uint32(part)) & np.uint32(0xFFFFFFFE)
        tree.insert(to_dev(some, dev), to_dev(vals, dev))
        ref.insert(some, vals)
        gone = rng.permutation(keys)[: 2_000]
        tree.erase(to_dev(gone, dev))
        ref.erase(gone)
        stamps.append(tree.take_snapshot())
        assert stamps[-1] == ref.take_snapshot()
    ends = np.array([1, 0xFFFFFFFE, 0, 0xFFFFFFFF], np.uint32)
    q = rng.choice(np.concatenate([keys, keys + np.uint32(1), ends]), size=n)
    lo = rng.choice(np.concatenate([keys, ends]), size=n)
    hi = np.minimum(lo.astype(np.uint64) + rng.choice([0, 1, wl.span_for(6, keys.size), wl.span_for(40, keys.size)],
                                                      size=n).astype(np.uint64), 0xFFFFFFFF).astype(np.uint32)
    hi[::7] = rng.choice(np.concatenate([keys, ends]), size=hi[::7].size) >> np.uint32(1)
    few = min(n, 300)  # long answers: more pairs than fit, at the edges of the output
    long_hi = rng.choice(np.array([0xFFFFFFFE, 0xFFFFFFFF], np.uint32), size=few)
    for ts in stamps + [mv.LATEST]:
        assert np.array_equal(to_np(tree.find(to_dev(q, dev), timestamp=ts)), ref.find(q, ts))
        for a, b, cap in ((lo, hi, 8), (lo[:few], long_hi, 32)):
            if cap == 32 or np.any(b > a):
                p, c = tree.range_query(to_dev(a, dev), to_dev(b, dev), cap, timestamp=ts)
                rp, rc = ref.range_query(a, b, cap, ts)
                assert np.array_equal(to_np(c), rc)
                live = np.arange(cap)[None, :] < np.minimum(rc, cap)[:, None]
                assert np.array_equal(to_np(p, np.uint64).reshape(-1, cap)[live], rp.reshape(-1, cap)[live])
    assert tree.error_flags() & ~(1 << 4) == 0  # long answers may overflow, nothing else
    assert tree.validate_tree_structure()[0] == ref.size()
