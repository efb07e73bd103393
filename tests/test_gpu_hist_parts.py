"""Histograms whose workgroups take 32 of a byte slab's 64 or 128 columns, and whole rows beyond their sizes: packed partials
(4 quantized bins) and {g, h} pairs (64 bins: flushed every 1023 rows), row ranges that do not come in eights, ragged and tiny
leaves, through the host, slot and fixed-scratch entry points. Integers: every one equals the oracle's."""

import numpy as np
import pytest
import torch

import oracle
import silvic_amd
from silvic_amd import _abi
from tests.test_gpu_parity import quantized_setup, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qbins", [4, 64])
@pytest.mark.parametrize("rows,cols", [(70_001, 50), (70_001, 100), (300_007, 150), (1_700_001, 40)])
def test_histograms_of_column_parts_match_the_oracle(rocm, rows, cols, qbins):
    say("column parts", rows, cols, qbins)
    rng = np.random.default_rng(cols + qbins)
    data = silvic_amd.from_bins(rng.integers(0, 255, (rows, cols), dtype=np.uint8), [255] * cols, rng.random(rows))
    g = rng.standard_normal(rows).astype(np.float32)
    h = (0.1 + rng.random(rows)).astype(np.float32)
    _, packed = quantized_setup(rocm, data, g, h, num_bins=qbins)
    assert rocm.reset_partition() == rows
    order = np.arange(rows, dtype=np.uint32)
    rocm.hist_slots(2)
    out = torch.empty(2 * data.total_bins, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    for b, c in [(0, rows), (3, 1), (7, 65), (1, 2048), (1, 2049), (5, 18_433), (64, rows - 65)]:
        want = oracle.histogram(data, packed, qbins, order[b:b + c])
        assert np.array_equal(rocm.histogram((b, c)), want), (b, c)
        rocm.histogram_slot((b, c), 1)
        assert np.array_equal(rocm.read_slot(1), want), (b, c)
        assert _abi.load_rocm().srocm_histogram_noalloc(rocm._h, _abi.LeafRange(b, c), out.data_ptr(), out.numel(), 1) == _abi.OK
        assert np.array_equal(out.cpu().numpy().astype(np.float64), want), (b, c)
