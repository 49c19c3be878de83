"""transform_layout past 64 MiB into rows that start on whole lines (non-temporal), on 16 bytes only, and on elements; either
direction.  Bytes are moved, so results are equal."""
import numpy as np
import pytest

from test_gpu_layout_runs import _exchange

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("to_dense", [True, False])
@pytest.mark.parametrize("n_run,pad", [(80, 4), (80, 2), (80, 3), (82, 2), (83, 3)])
def test_rows(gpu, oracle, n_run, pad, to_dense):
    _exchange(oracle, 300, 350, n_run, np.float64, pad, 0, to_dense)
