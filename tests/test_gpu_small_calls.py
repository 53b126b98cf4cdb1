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
