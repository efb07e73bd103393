"""What the trait calls keep between calls, and their readbacks in pieces: a split search after one with another feature
table of the same length (the device's table follows the contents), and row arrays of one piece (1 MiB), of a few, and of
more than the staging holds (16 pieces) coming back whole."""

import numpy as np
import pytest

import oracle
import silvic_amd
from silvic_amd import _abi
from tests.test_gpu_parity import compare_split, say

pytestmark = pytest.mark.gpu


def test_split_search_follows_a_changed_feature_table(rocm):
    rng = np.random.default_rng(4)
    cfg = oracle.default_params().cfg
    cfg.min_data_in_leaf = 3
    kinds = (_abi.BINS_NUMERICAL, _abi.BINS_CATEGORICAL)
    tables = []
    for bins in ([20, 255, 7, 64], [20, 255, 7, 64], [64, 7, 255, 20]):
        offs = np.concatenate([[0], np.cumsum(bins)])
        tables.append([silvic_amd.FeatureMeta(b, 0, i, int(offs[i]), kinds[i == 2], i % 2 == len(tables) % 2)
                       for i, b in enumerate(bins)])
    hist = np.stack([rng.integers(-40, 40, 346), rng.integers(1, 60, 346)], 1).astype(np.float64).reshape(-1)
    for k in (0, 1, 0, 2, 1, 1):
        say("table", k)
        feats = tables[k]
        m = feats[0]
        part = hist.reshape(-1, 2)[m.hist_offset:m.hist_offset + m.num_bins].sum(0)
        sums = (float(part[0]), float(part[1]), 5000)
        ev = np.ones(4, bool)
        d, dspl = rocm.find_best_split(hist, feats, ev, sums, 0.01, 0.02, cfg)
        o, ospl = oracle.find_best_split(hist, feats, ev, sums, 0.01, 0.02, cfg)
        compare_split(d, o, f"table {k}")
        assert np.array_equal(dspl, np.asarray(ospl, bool))
        assert list(d.cat_bins[:d.num_cat_bins]) == list(o.cat_bins[:o.num_cat_bins])


@pytest.mark.parametrize("rows", [262_144, 262_145, 4_500_001])
def test_row_arrays_come_back_whole(rocm, rows):
    say("rows back", rows)
    rng = np.random.default_rng(rows)
    data = silvic_amd.from_bins(rng.integers(0, 4, (rows, 1)), [4], rng.random(rows))
    rocm.load(data)
    g = rng.standard_normal(rows).astype(np.float32)
    h = rng.random(rows).astype(np.float32)
    rocm.set_gradients(g, h)
    bg, bh = rocm.gradients()
    assert np.array_equal(bg, g) and np.array_equal(bh, h)
    assert rocm.reset_partition() == rows
    assert np.array_equal(rocm.partition_rows(), np.arange(rows, dtype=np.uint32))
    m = data.features[0]
    rocm.init_scores(0, 0.5)
    rocm.add_tree([silvic_amd.device_node(silvic_amd.bin_split(m.group, m.column, [0, 2]), -1, -2)], [1.0, 2.0])
    want = np.float32(0.5) + np.where(np.isin(data.bin(0), (0, 2)), np.float32(1.0), np.float32(2.0))
    assert np.array_equal(rocm.scores(0), want.astype(np.float32))
