"""Trees that are one long chain: every split cuts one bin off the end of the largest leaf, so the speculative tree is far
deeper than the links a leaf's bound walks up by itself (frontier_bounds) and its bounds end in pointer-jumping rounds. At
one leaf count of each replay's range the tree and the final partition equal the oracle's."""

import numpy as np
import pytest

import oracle
from silvic_amd import from_bins
from tests.test_gpu_parity import compare_trees, quantized_setup, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("leaves", [40, 120, 250, 700])
def test_chain_trees_match_the_oracle(rocm, leaves):
    say("chain", leaves)
    rng = np.random.default_rng(leaves)
    rows = 60_000
    # bins of geometrically falling counts, the gradient's sign alternating from one to the next: the largest leaf is what
    # is left past the last bin cut off
    bins = np.minimum(-25.0 * np.log(rng.random((rows, 4))), 249.0).astype(np.uint8)
    g = np.where(bins[:, 0] % 2, 1.0, -1.0) * (1.0 + bins[:, 0] / 50.0) + 0.01 * rng.standard_normal(rows)
    g = g.astype(np.float32)
    h = np.ones(rows, np.float32)
    data = from_bins(bins, [250] * 4, np.zeros(rows))
    p = oracle.default_params(num_leaves=leaves, num_grad_quant_bins=64)
    p.cfg.min_data_in_leaf = 1
    o_tree, _, o_part = oracle.grow_tree(data, g, h, p, renew=False)
    assert o_tree["leaf_depth"].max() >= 39
    spec, _ = quantized_setup(rocm, data, g, h, seed=p.data_random_seed, num_bins=64)
    n = rocm.reset_partition()
    d = rocm.grow(p.cfg, leaves, -1, spec.grad_scale, spec.hess_scale, np.ones(4, bool), (0, n), n)
    compare_trees(d, dict(o_tree), f"chain {leaves}")
    assert np.array_equal(rocm.partition_rows(n), o_part)
