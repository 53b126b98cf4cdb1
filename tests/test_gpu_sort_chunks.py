"""The stable sort under a tree's first insert, at the edges of its chunks: less
than one element a thread, several chunks a workgroup, few distinct digits; the
last of a repeated key has to win."""
from __future__ import annotations

import numpy as np
import pytest

import mvgpubtree_amd as mv

from conftest import to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [64, 513, 131_073, 1_048_575, 1_048_577, 2_100_001])
@pytest.mark.parametrize("spread", [1 << 6, 1 << 20, 0xFFFFFFFD])
def test_sorted_first_insert_keeps_order_of_equal_keys(dev, n, spread):
    rng = np.random.default_rng(n ^ spread)
    keys = rng.integers(1, spread + 1, size=n, dtype=np.uint64).astype(np.uint32)
    vals = np.arange(n, dtype=np.uint32)
    tree = mv.GpuBlinkTree(pool_nodes=n // 3 + (1 << 16))
    tree.insert(to_dev(keys, dev), to_dev(vals, dev))
    distinct, back = np.unique(keys[::-1], return_index=True)  # first from behind = last given
    assert np.array_equal(to_np(tree.find(to_dev(distinct, dev))), vals[::-1][back])
    assert tree.error_flags() == 0
    assert tree.validate_tree_structure()[0] == distinct.size
