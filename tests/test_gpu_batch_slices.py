"""GPU parity of the sorted batched form's passes over slices of the call's
operations, whatever batches the slices hold, against the batch-by-batch
replay."""
from __future__ import annotations

import numpy as np
import pytest

import mvgpubtree_amd as mv
import oracle
from mvgpubtree_amd import workloads as wl

from conftest import to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nw,lanes", [(16, 0), (32, 16), (64, 32)])
@pytest.mark.parametrize("sizes", [[1], [0, 0, 3, 0], [5] * 3000, [30_000, 1, 0, 1, 9_000], [2] * 40 + [20_000] + [0] * 5000])
def test_sorted_form_slices_and_divisions(dev, nw, lanes, sizes):
    """Calls whose slices of operations hold one batch, many, empty ones, and
    more than a slice's LDS copy takes, in the sorted form at every division of
    its passes, against the batch-by-batch replay."""
    rng = np.random.default_rng(len(sizes) + nw)
    keys = wl.unique_keys(rng, 20_000 + sum(sizes))
    tree = mv.GpuVersionedBTree(pool_nodes=1 << 17, node_width=nw)
    tree.set_read_tile(lanes)
    tree.set_worker_mode(2)
    init = keys[:20_000]
    tree.insert(to_dev(init, dev), to_dev(wl.value_of(init), dev))
    at, batches = 20_000, []
    for s in sizes:
        n_i, n_e, n_r = s // 4, s // 8, s // 5
        ik = keys[at:at + n_i]
        at += s
        ek = rng.choice(init, size=n_e, replace=False)
        lo = rng.integers(1, 0xFFFFFF00, size=n_r, dtype=np.uint64).astype(np.uint32)
        hi = np.minimum(lo.astype(np.uint64) + wl.span_for(6, 20_000), 0xFFFFFFFE).astype(np.uint32)
        batches.append(wl.Batch(insert_keys=ik, insert_values=wl.value_of(ik), erase_keys=ek,
                                find_keys=rng.choice(keys, size=s - n_i - n_e - n_r), range_lo=lo, range_hi=hi))
    ops, offs, slots = wl.to_ops(batches, seed=1)
    L = 24
    pairs = to_dev(np.full(max(slots, 1) * L, 0xFFFFFFFFFFFFFFFF, np.uint64), dev)
    res = to_np(tree.run_batches(to_dev(ops, dev), to_dev(offs, dev), pairs=pairs, pair_slots=max(slots, 1),
                                 average_range_length=L))
    assert tree.error_flags() == 0
    want_r, want_p, ref = oracle.replay_batches(init, wl.value_of(init), ops, offs, L, max(slots, 1))
    assert np.array_equal(res, want_r)
    assert np.array_equal(to_np(pairs, np.uint64), want_p)
    assert tree.validate_tree_structure()[0] == ref.size()
