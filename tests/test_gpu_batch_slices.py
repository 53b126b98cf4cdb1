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


@pytest.mark.parametrize("mode", [2, 3])
@pytest.mark.parametrize("nb,n", [(1, 1), (7, 16384), (4096, 16384), (4097, 9000), (3, 16385)])
def test_small_calls_and_their_limits(dev, mode, nb, n):
    """Calls at the limits of the form made for small ones: as many operations
    and batches as it takes, one more of each, all writes to a few hot leaves
    (many batches write one leaf) beside spread ones, reserved keys, through
    the graph and without it, against the replay; a batch that writes one key
    twice is rejected whole."""
    rng = np.random.default_rng(nb + n)
    init = np.sort(wl.unique_keys(rng, 30_000))
    cut = np.sort(rng.integers(0, n + 1, size=nb - 1)) if nb > 1 else np.empty(0, int)
    offs = np.concatenate([[0], cut, [n]]).astype(np.uint64)
    ops = np.zeros((n, 4), np.uint32)
    ops[:, 0] = rng.choice([mv.OP_FIND, mv.OP_INSERT, mv.OP_ERASE, mv.OP_RANGE], size=n, p=[0.3, 0.4, 0.2, 0.1])
    hot = init[1000:1040]
    for b in range(nb):
        lo, hi = int(offs[b]), int(offs[b + 1])
        k = np.where(rng.random(hi - lo) < 0.3, rng.choice(hot, size=hi - lo), rng.choice(init, size=hi - lo) + 1)
        w = (ops[lo:hi, 0] == mv.OP_INSERT) | (ops[lo:hi, 0] == mv.OP_ERASE)
        _, first = np.unique(k, return_index=True)
        dup = np.ones(hi - lo, bool)
        dup[first] = False
        ops[lo:hi, 0] = np.where(w & dup, mv.OP_FIND, ops[lo:hi, 0])  # one write per key and batch
        ops[lo:hi, 1] = k
    ops[:, 2] = rng.integers(1, 1 << 31, size=n)
    r = ops[:, 0] == mv.OP_RANGE
    ops[r, 2] = np.minimum(ops[r, 1].astype(np.uint64) + wl.span_for(5, init.size), 0xFFFFFFFE)
    ops[r, 3] = np.arange(r.sum())
    slots, L = max(int(r.sum()), 1), 16
    want_r, want_p, ref = oracle.replay_batches(init, wl.value_of(init), ops, offs, L, slots)
    for graph in (False, True):
        tree = mv.GpuVersionedBTree(pool_nodes=1 << 16, node_width=32 if graph else 16)
        tree.set_worker_mode(mode)
        tree.bulk_build(to_dev(init, dev), to_dev(wl.value_of(init), dev))
        if graph:
            tree.reserve_batches(n, nb)
        pairs = to_dev(np.full(slots * L, 0xFFFFFFFFFFFFFFFF, np.uint64), dev)
        base = to_dev(np.zeros(1, np.uint32), dev)
        res = to_np(tree.run_batches(to_dev(ops, dev), to_dev(offs, dev), pairs=pairs, pair_slots=slots,
                                     average_range_length=L, snapshot_base=base, use_graph=graph))
        assert tree.error_flags() in (0, mv.FLAG_RANGE_OVERFLOW)
        assert np.array_equal(res, want_r)
        assert np.array_equal(to_np(pairs, np.uint64), want_p)
        assert int(to_np(base)[0]) == 0 and tree.take_snapshot() == nb
        assert tree.validate_tree_structure()[0] == ref.size()
        tree.clear_error_flags()
        if n > 4:  # the same call with one key written twice by its last non-trivial batch
            bad = ops.copy()
            b = int(np.nonzero(np.diff(offs.astype(np.int64)) >= 2)[0][-1])
            i = int(offs[b])
            bad[i:i + 2, 0] = (mv.OP_INSERT, mv.OP_ERASE)
            bad[i + 1, 1] = bad[i, 1]
            before = tree.export()
            tree.run_batches(to_dev(bad, dev), to_dev(offs, dev), pairs=pairs, pair_slots=slots,
                             average_range_length=L, use_graph=graph)
            assert tree.error_flags() == mv.FLAG_BAD_BATCH
            assert np.array_equal(before, tree.export())


def test_small_call_in_a_pool_with_few_slots(dev):
    """Erases of absent keys copy nothing: a call of many of them and a few
    inserts fits a pool whose spare slots cover only the inserts' copies."""
    rng = np.random.default_rng(9)
    init = np.sort(wl.unique_keys(rng, 20_000))
    probe = mv.GpuVersionedBTree(pool_nodes=1 << 14)
    probe.bulk_build(to_dev(init, dev), to_dev(wl.value_of(init), dev))
    tree = mv.GpuVersionedBTree(pool_nodes=probe.memory_stats().live_nodes + 700)
    tree.bulk_build(to_dev(init, dev), to_dev(wl.value_of(init), dev))
    absent = wl.absent_keys(rng, 4000, init)
    some = rng.choice(init, size=60, replace=False)
    ops = np.zeros((4060, 4), np.uint32)
    ops[:, 0] = mv.OP_ERASE
    ops[:, 1] = np.concatenate([absent, some])
    ops[4000:, 0] = mv.OP_INSERT
    ops[4000:, 2] = 5
    ops = ops[rng.permutation(4060)]
    offs = np.array([0, 1000, 4060], np.uint64)
    _, keep = np.unique(ops[:, 1], return_index=True)
    assert keep.size == 4060
    res = to_np(tree.run_batches(to_dev(ops, dev), to_dev(offs, dev)))
    assert tree.error_flags() == 0
    assert np.all(res == 0)  # absent keys erased, present keys updated
    assert np.all(to_np(tree.find(to_dev(some, dev))) == 5)
