"""Saved batch configurations of kernels that are gone: an entry under the signature of domain sizes, types and form alone,
as they were recorded for the item-table stencil phase, is not taken up by a batch of the same domains."""
import numpy as np
import pytest

from test_gpu_batch import make_members

pytestmark = pytest.mark.gpu


def _signature(values):
    h = 1469598103934665603
    for v in values:
        for b in range(8):
            h = (h ^ (v >> (8 * b) & 0xff)) * 1099511628211 & (1 << 64) - 1
    return h


def test_entries_of_the_item_tables_are_not_taken(gpu, tmp_path):
    from gridtools_amd import tune
    from gridtools_amd.batch import Batch

    sizes = [(70, 30, 60), (64, 20, 120)]
    key = _signature([3, 1, 1, len(sizes)] + [v for s in sizes for v in (*s, 0)])  # form, FP32 storage, FP64 arithmetic
    path = tmp_path / "tune.txt"
    path.write_text(f"batch {key:016x} 4 8 3 8 2 4 81 123.000\n")
    tune.clear()
    try:
        default = Batch(make_members(gpu, sizes, np.float32), precision=1, wg_per_cu=1).config()
        assert tune.load(path) == 1
        assert Batch(make_members(gpu, sizes, np.float32), precision=1, wg_per_cu=1).config() == default
    finally:
        tune.clear()
