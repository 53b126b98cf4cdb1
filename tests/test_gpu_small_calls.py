"""GPU tests of small batched calls (at most 16384 operations) where they could
go wrong beside their results: rejected calls, the pool slots they take, and
readers on another stream, against the batch-by-batch replay."""
from __future__ import annotations

import numpy as np
import pytest

import mvgpubtree_amd as mv
import oracle
from mvgpubtree_amd import workloads as wl

from conftest import to_dev, to_np

pytestmark = pytest.mark.gpu


def _mixed_ops(rng, init, n, nb):
    """n operations in nb batches over the keys of `init`, one write per key and call."""
    ops = np.zeros((n, 4), np.uint32)
    k = rng.permutation(init)[:n]
    ops[:, 0] = rng.choice([mv.OP_FIND, mv.OP_INSERT, mv.OP_ERASE], size=n, p=[0.4, 0.4, 0.2])
    ops[:, 1] = k + rng.integers(0, 2, size=n).astype(np.uint32)  # half of them absent
    _, first = np.unique(ops[:, 1], return_index=True)
    dup = np.ones(n, bool)
    dup[first] = False
    ops[dup, 0] = mv.OP_FIND
    ops[:, 2] = rng.integers(1, 1 << 31, size=n)
    offs = np.concatenate([[0], np.sort(rng.integers(0, n + 1, size=nb - 1)), [n]]).astype(np.uint64)
    return ops, offs


@pytest.mark.parametrize("where", ["first", "last_wave", "second_round", "last", "one_a_wave", "every"])
@pytest.mark.parametrize("n", [1024, 16384])
def test_unknown_types_reject_a_call_of_many_waves(dev, n, where):
    """An unknown operation type anywhere in a call that fills every wave of
    the checking workgroup: results and tree stay as they were, and a valid
    call on the same handle then runs as if the bad one had not been sent."""
    rng = np.random.default_rng(n)
    init = np.sort(wl.unique_keys(rng, 20_000))
    tree = mv.GpuVersionedBTree(pool_nodes=1 << 16)
    tree.bulk_build(to_dev(init, dev), to_dev(wl.value_of(init), dev))
    ops, offs = _mixed_ops(rng, init, n, 5)
    at = {"first": [0], "last_wave": [1023], "second_round": [min(1024 + 70, n - 1)], "last": [n - 1],
          "one_a_wave": np.arange(0, n, 64), "every": np.arange(n)}[where]
    bad = ops.copy()
    bad[at, 0] = 9
    res = to_dev(np.full(n, 0xABCD1234, np.uint32), dev)
    before = tree.export()
    tree.run_batches(to_dev(bad, dev), to_dev(offs, dev), results=res)
    assert tree.error_flags() == mv.FLAG_BAD_BATCH
    assert np.all(to_np(res) == 0xABCD1234)
    assert np.array_equal(before, tree.export())
    tree.clear_error_flags()
    want, _, ref = oracle.replay_batches(init, wl.value_of(init), ops, offs, 1, 1)
    tree.run_batches(to_dev(ops, dev), to_dev(offs, dev), results=res)
    assert tree.error_flags() == 0
    assert np.array_equal(to_np(res), want)
    assert tree.validate_tree_structure()[0] == ref.size()


def _update_ops(rng, init, n, nb, noop):
    """nb batches of writes: updates and erases of present keys, each batch its
    own distinct keys, and a share `noop` of erases of absent keys."""
    ops, offs = [], [0]
    absent = wl.absent_keys(rng, n, init)
    at = 0
    for m in np.diff(np.linspace(0, n, nb + 1).astype(int)):
        k = int(m * noop)
        o = np.zeros((m, 4), np.uint32)
        o[:k, 0], o[:k, 1] = mv.OP_ERASE, absent[at:at + k]
        o[k:, 0], o[k:, 1] = mv.OP_INSERT, rng.choice(init, size=m - k, replace=False)
        o[k:, 2] = rng.integers(1, 1 << 31, size=m - k)
        at += k
        ops.append(o[rng.permutation(m)])
        offs.append(offs[-1] + m)
    return np.concatenate(ops), np.array(offs, np.uint64)


@pytest.mark.parametrize("nw", [16, 32, 64])
@pytest.mark.parametrize("n,nb", [(1, 1), (300, 3), (1025, 1), (9000, 40), (16383, 3)])
@pytest.mark.parametrize("noop", [0.0, 0.7, 1.0])
def test_slots_taken_are_the_copies_made(dev, nw, n, nb, noop):
    """Calls in the default mode retire as many slots as a call that runs
    batch after batch: one per copy of a leaf, none for writes that change
    nothing; the others are free again when the call ends, also under a live
    snapshot, and a reclamation gives the copies' back."""
    rng = np.random.default_rng(n + nw)
    init = np.sort(wl.unique_keys(rng, 40_000))
    ops, offs = _update_ops(rng, init, n, nb, noop)
    seen = []
    for mode in (0, 3):
        tree = mv.GpuVersionedBTree(pool_nodes=1 << 19, node_width=nw)
        tree.set_worker_mode(mode)
        tree.bulk_build(to_dev(init, dev), to_dev(wl.value_of(init), dev))
        live = tree.memory_stats().live_nodes
        snap = tree.take_snapshot()
        stats = []
        for _ in range(3):
            tree.run_batches(to_dev(ops, dev), to_dev(offs, dev))
            st = tree.memory_stats()
            stats.append((st.retired_total, st.live_nodes))
            assert st.live_nodes + st.free_nodes == st.capacity_nodes
            assert st.live_nodes == live + st.retired_pending
        if noop == 1.0:
            assert stats[-1] == (0, live)
        assert tree.memory_stats().peak_live_nodes == stats[-1][1]
        seen.append((stats, tree.export()))
        tree.release_snapshot(snap)
        tree.reclaim()
        st = tree.memory_stats()
        assert st.live_nodes == live and st.retired_pending == 0 and st.reclaimed_nodes == st.retired_total
        # the free slots are distinct: every one can be used, and the tree stays whole
        tree.insert(to_dev(init, dev), to_dev(wl.value_of(init), dev))
        assert tree.error_flags() == 0
        assert np.array_equal(to_np(tree.find(to_dev(init, dev))), wl.value_of(init))
        assert tree.validate_tree_structure()[0] == init.size
    assert seen[0][0] == seen[1][0]
    assert np.array_equal(seen[0][1], seen[1][1])


@pytest.mark.parametrize("no_alloc", [False, True])
def test_slots_of_calls_that_reclaim(dev, no_alloc):
    """Small calls of the sorted form that reclaim in the call free the copies
    they made, and record the epoch."""
    rng = np.random.default_rng(3)
    init = np.sort(wl.unique_keys(rng, 40_000))
    tree = mv.GpuVersionedBTree(pool_nodes=1 << 17, node_width=32)
    tree.set_worker_mode(2)
    tree.bulk_build(to_dev(init, dev), to_dev(wl.value_of(init), dev))
    live = tree.memory_stats().live_nodes
    total = 0
    for k, (n, nb) in enumerate([(900, 3), (16384, 30), (1, 1), (5000, 4096)]):
        ops, offs = _update_ops(rng, init, n, nb, 0.5)
        ref = mv.GpuVersionedBTree(pool_nodes=1 << 18, node_width=32)
        ref.set_worker_mode(0)
        ref.bulk_build(to_dev(init, dev), to_dev(wl.value_of(init), dev))
        ref.run_batches(to_dev(ops, dev), to_dev(offs, dev))
        total += ref.memory_stats().retired_total
        tree.run_batches(to_dev(ops, dev), to_dev(offs, dev), no_alloc=no_alloc)
        st = tree.memory_stats()
        assert st.live_nodes == live and st.retired_pending == 0
        assert st.live_nodes + st.free_nodes == st.capacity_nodes
        assert st.retired_total == st.reclaimed_nodes == total
        assert tree.memory_series()[-1].freed_nodes == ref.memory_stats().retired_total
    assert tree.error_flags() == 0
    assert tree.validate_tree_structure()[0] == init.size


@pytest.mark.parametrize("fill", [0, 14])
def test_nearly_full_pools(dev, fill):
    """A call of erases of absent keys, updates and inserts that split (at
    fill 14 every node of every level is full) into pools of every spare size:
    where the form that takes a slot only for what it stores finds room, the
    default form does."""
    rng = np.random.default_rng(17)
    init = np.sort(wl.unique_keys(rng, 20_000))
    vals = wl.value_of(init)
    probe = mv.GpuVersionedBTree(pool_nodes=1 << 14)
    probe.bulk_build(to_dev(init, dev), to_dev(vals, dev), fill=fill)
    live = probe.memory_stats().live_nodes
    for n, inserts in ((1, 1), (40, 40), (2000, 60)):
        absent = wl.absent_keys(rng, n, init)
        ops = np.zeros((n, 4), np.uint32)
        ops[:, 0], ops[:, 1] = mv.OP_ERASE, absent
        ops[:inserts, 0], ops[:inserts, 2] = mv.OP_INSERT, 7
        ops = ops[rng.permutation(n)]
        offs = np.array([0, n // 2, n], np.uint64)
        leaf = np.searchsorted(init[::fill or 10], ops[:, 1], side="right")
        groups = len(set(zip(leaf.tolist(), (np.arange(n) >= n // 2).tolist())))  # (leaf, batch) pairs written
        near = [groups + k for k in (-1, 0, 1, 5, 20, 60, 130, 200, 300)]
        for spare in near + [4, 8, 16, 40, 80, 120, 160, 240, 400, 900, 4200, 6500, 30_000, 33_000]:
            if spare < 2:
                continue
            flags = []
            for mode in (0, 3):
                tree = mv.GpuVersionedBTree(pool_nodes=live + spare)
                tree.set_worker_mode(mode)
                tree.bulk_build(to_dev(init, dev), to_dev(vals, dev), fill=fill)
                res = to_np(tree.run_batches(to_dev(ops, dev), to_dev(offs, dev)))
                flags.append(tree.error_flags())
                if flags[-1] == 0:
                    assert np.array_equal(res, (ops[:, 0] == mv.OP_INSERT).astype(np.uint32))
                    assert tree.validate_tree_structure()[0] == init.size + inserts
            assert flags[1] == 0 or flags[0] != 0, (n, spare, flags)


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("spare", [3600, 200_000])
def test_few_operations_in_many_batches(dev, spare, graph):
    """Fewer than 16384 operations in more batches than the small form takes:
    the default mode holds a slot only for a copy it makes there too, so the
    call fits a pool that has room for its copies and not for its writes, and
    gives back what it did not use of a larger one; in one window and several."""
    rng = np.random.default_rng(23)
    init = np.sort(wl.unique_keys(rng, 20_000))
    n, nb = 9000, 5000
    ops, _ = _update_ops(rng, init, n, 1, 0.9)
    offs = np.concatenate([[0], np.sort(rng.integers(0, n + 1, size=nb - 1)), [n]]).astype(np.uint64)
    probe = mv.GpuVersionedBTree(pool_nodes=1 << 14)
    probe.bulk_build(to_dev(init, dev), to_dev(wl.value_of(init), dev))
    live = probe.memory_stats().live_nodes
    want, _, ref = oracle.replay_batches(init, wl.value_of(init), ops, offs, 1, 1)
    tree = mv.GpuVersionedBTree(pool_nodes=live + spare)
    tree.bulk_build(to_dev(init, dev), to_dev(wl.value_of(init), dev))
    if graph:
        tree.reserve_batches(20_000, nb)  # a larger call's reservation covers it
    tree.set_batch_window(4000 if graph else 0)
    for k in range(2):  # (the second call finds the present keys updated and the absent ones absent as well)
        res = to_np(tree.run_batches(to_dev(ops, dev), to_dev(offs, dev), use_graph=graph))
        assert tree.error_flags() == 0
        assert np.array_equal(res, want)
        st = tree.memory_stats()
        assert 0 < st.retired_total <= (k + 1) * n // 10
        assert st.live_nodes == live + st.retired_total == st.capacity_nodes - st.free_nodes
    tree.reclaim()
    st = tree.memory_stats()
    assert st.live_nodes == live and st.reclaimed_nodes == st.retired_total
    assert tree.validate_tree_structure()[0] == ref.size()


@pytest.mark.parametrize("nw", [16, 32, 64])
@pytest.mark.parametrize("nb", [3, 4500])
def test_latest_reads_beside_small_calls(dev, nw, nb):
    """MVBT_CONCURRENT reads of the latest version on one stream while small
    calls run on another: leaves are written under their locks, so keys that no
    call writes read exactly, written ones as before or after some call, ranges
    stay sorted, and no leaf is left locked."""
    import torch
    rng = np.random.default_rng(nw + nb)
    init = np.sort(wl.unique_keys(rng, 60_000))
    vals = wl.value_of(init) & np.uint32(0x3FFFFFFF)
    still, moved = init[::2], init[1::2]
    tree = mv.GpuVersionedBTree(pool_nodes=1 << 20, node_width=nw)
    tree.bulk_build(to_dev(init, dev), to_dev(vals, dev))
    calls = []
    for k in range(24):  # updates (values of bit 31), erases and inserts of the moving keys, in turn
        n = 9000
        ops = np.zeros((n, 4), np.uint32)
        ops[:, 1] = rng.choice(moved, size=n, replace=False)
        ops[:, 0] = rng.choice([mv.OP_INSERT, mv.OP_ERASE], size=n, p=[0.7, 0.3])
        ops[:, 2] = ops[:, 1] | np.uint32(0x80000000)
        offs = np.concatenate([[0], np.sort(rng.integers(0, n + 1, size=nb - 1)), [n]]).astype(np.uint64)
        calls.append((to_dev(ops, dev), to_dev(offs, dev), torch.empty(n, dtype=torch.int32, device=dev)))
    q = rng.permutation(init)
    lo = rng.choice(init, size=4000)
    hi = np.minimum(lo.astype(np.uint64) + wl.span_for(40, init.size), 0xFFFFFFFE).astype(np.uint32)
    L = 128
    dq, dlo, dhi = to_dev(q, dev), to_dev(lo, dev), to_dev(hi, dev)
    tree.reserve_batches(9000, nb)
    torch.cuda.synchronize()
    sr, sw = torch.cuda.Stream(), torch.cuda.Stream()
    finds, ranges = [], []
    for ops, offs, res in calls:
        with torch.cuda.stream(sw):
            tree.run_batches(ops, offs, results=res, stream=sw)
        with torch.cuda.stream(sr):
            finds.append(tree.find(dq, stream=sr, concurrent=True))
            ranges.append(tree.range_query(dlo, dhi, L, stream=sr, concurrent=True))
    torch.cuda.synchronize()
    assert tree.error_flags() == 0
    unmoved = np.isin(q, still)
    want = vals[np.searchsorted(init, q)]
    for f in finds:
        got = to_np(f)
        assert np.array_equal(got[unmoved], want[unmoved])
        m = ~unmoved
        assert np.all((got[m] == want[m]) | (got[m] == (q[m] | np.uint32(0x80000000))) | (got[m] == 0xFFFFFFFF))
    a, b = np.searchsorted(still, lo), np.searchsorted(still, hi)
    for p, c in ranges:
        p, c = to_np(p, np.uint64).reshape(-1, L), to_np(c)
        assert c.max() <= L
        for i in range(0, lo.size, 37):
            k = (p[i, :c[i]] & np.uint64(0xFFFFFFFF)).astype(np.uint32)
            assert np.all(np.diff(k.astype(np.int64)) > 0)
            assert np.array_equal(k[np.isin(k, still)], still[a[i]:b[i]])
    state = dict(zip(init.tolist(), vals.tolist()))
    for ops, _, _ in calls:
        o = to_np(ops).reshape(-1, 4)
        for ty, k, v in zip(o[:, 0].tolist(), o[:, 1].tolist(), o[:, 2].tolist()):
            if ty == mv.OP_INSERT:
                state[k] = v
            else:
                state.pop(k, None)
    assert tree.validate_tree_structure()[0] == len(state)  # (a locked leaf fails this)
    got = to_np(tree.find(dq))
    assert np.array_equal(got, np.array([state.get(k, 0xFFFFFFFF) for k in q.tolist()], np.uint32))
