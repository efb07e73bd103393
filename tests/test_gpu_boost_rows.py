"""The boosting loop's one-pass quantization (words, row ids and gradient codes, four rows a thread) at every remainder of
four rows, with and without a bag, with carried codes (4 bins) and without (16), over iterations whose gradient maxima take
turns in two buffers: trees, scores and the final partition equal the oracle's."""

import numpy as np
import pytest

import silvic_amd
from silvic_amd import _abi
from tests.test_gpu_parity import boost_both, compare_trees, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,params", [(4001, {}), (4002, dict(num_grad_quant_bins=16)), (4003, dict(bagging_fraction=0.7, bagging_freq=1)),
                                         (5, dict(min_data_in_leaf=1)), (6148, dict(objective=_abi.OBJ_REGRESSION, quant_train_renew_leaf=0))])
def test_boosting_over_ragged_rows_matches_the_oracle(rows, params):
    say("ragged boost", rows, params)
    data = silvic_amd.synthetic(2, rows=rows, cols=7, seed=rows)
    p = dict(objective=_abi.OBJ_BINARY, num_leaves=15)
    p.update(params)
    o, t = boost_both(data, p, 5)
    try:
        assert len(t.trees) == len(o.trees)
        for i, (d, ot) in enumerate(zip(t.trees, o.trees)):
            compare_trees(d, ot, f"tree {i}", exact_values=False)
        assert np.array_equal(t.backend.scores(0), o.scores)
    finally:
        t.backend.close()
