"""The row passes of the trait calls: trees added by the branch-free walk (from 1024 rows a compute unit, up to 512 leaves)
and by the plain one, on one- and two-byte bins with category sets and missing-value rules; leaf sums over pieces of 2048
rows. Every one equals the oracle's."""

import numpy as np
import pytest

import oracle
import silvic_amd
from silvic_amd import bin_split, device_node, wide_bin_split
from tests.test_gpu_parity import say

pytestmark = pytest.mark.gpu


def random_tree(data, leaves, rng):
    """A tree of random splits, children after their parent: threshold rules on two-byte features, bin sets on others."""
    left, right, splits, ends = [], [], [], [(-1, False)]
    used = [m for m in data.features if m.num_bins]
    for k in range(leaves - 1):
        leaf = int(rng.integers(0, len(ends)))
        parent, went_right = ends[leaf]
        if parent >= 0:
            (right if went_right else left)[parent] = k
        left.append(~leaf)
        right.append(~len(ends))
        ends[leaf] = (k, False)
        ends.append((k, True))
        m = used[int(rng.integers(0, len(used)))]
        if data.groups[m.group].bin_bits == 16:
            splits.append(wide_bin_split(m.group, m.column, int(rng.integers(0, m.num_bins)), m.num_bins - 1 if k % 2 else None))
        else:
            splits.append(bin_split(m.group, m.column, np.flatnonzero(rng.random(m.num_bins) < 0.5).tolist()))
    return [device_node(s, a, b) for s, a, b in zip(splits, left, right)], rng.standard_normal(leaves).astype(np.float32)


@pytest.mark.parametrize("workload,rows", [(2, 262_143), (2, 262_145), (5, 262_145), (2, 3000)])
def test_added_trees_and_leaf_sums_match_the_oracle(rocm, workload, rows):
    say("row passes", workload, rows)
    rng = np.random.default_rng(rows + workload)
    data = silvic_amd.synthetic(workload, rows=rows, cols=9, seed=3, max_bin=1023 if workload == 5 else None)
    rocm.load(data)
    rocm.init_scores(0, 0.5)
    want = np.full(rows, 0.5, np.float32)
    for leaves in (2, 31, 512, 513):
        nodes, values = random_tree(data, leaves, rng)
        rocm.add_tree(nodes, values)
        want = oracle.add_tree(data, nodes, values, want)
        assert np.array_equal(rocm.scores(0), want), leaves
    g = rng.standard_normal(rows).astype(np.float32)
    h = rng.random(rows).astype(np.float32)
    rocm.set_gradients(g, h)
    rocm.reset_partition()
    leaves = [(0, 0), (0, 1), (1, 255), (256, 256), (300, 0), (512, 2047), (3, 2048), (700, 2049), (0, rows)]
    leaves = [(b, min(c, rows - b)) for b, c in leaves]
    got = rocm.leaf_sums(leaves, 1024.0, 256.0)
    assert np.array_equal(got, np.asarray(oracle.leaf_sums(g, h, np.arange(rows, dtype=np.uint32), leaves, 1024.0, 256.0)).reshape(-1, 2))
