"""The step kernel that makes the children's histograms and candidates (k_step_children) where its work items change
shape: one column group, a partly filled last group, groups in pairs; jobs of at most and of more partials than one block
takes (160: shares that meet in scratch), with packed partials and with {g, h} planes (64 gradient bins fill a packed word
in 1023 rows). Each tree and the final partition equal the oracle's."""

import numpy as np
import pytest

import oracle
import silvic_amd
from tests.test_gpu_parity import binary_gradients, compare_trees, quantized_setup, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,leaves,qbins", [(30_000, 1, 15, 4), (655_360, 5, 15, 4), (655_361, 5, 15, 4),
                                                    (1_100_001, 9, 31, 64), (120_000, 64, 40, 64)])
def test_children_of_every_item_shape_match_the_oracle(rocm, rows, cols, leaves, qbins):
    say("children", rows, cols, leaves, qbins)
    data = silvic_amd.synthetic(2, rows=rows, cols=cols, seed=cols)
    g, h = binary_gradients(data, 3)
    p = oracle.default_params(num_leaves=leaves, num_grad_quant_bins=qbins)
    o_tree, o_ranges, o_part = oracle.grow_tree(data, g, h, p, renew=False)
    spec, _ = quantized_setup(rocm, data, g, h, seed=p.data_random_seed, num_bins=qbins)
    n = rocm.reset_partition()
    mask = oracle.feature_mask(data.features, 1.0, 2, 0)
    d = rocm.grow(p.cfg, p.num_leaves, p.max_depth, spec.grad_scale, spec.hess_scale, mask, (0, n), n)
    compare_trees(d, dict(o_tree), f"children {rows} x {cols}")
    assert np.array_equal(rocm.partition_rows(n), o_part)
