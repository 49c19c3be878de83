"""transform_layout of 1- and 2-byte elements along runs that move whole: pieces of 128, 64, 32 and 16 elements of the other
dimension, at the numbers of tiles (1024) and the run lengths where they change.  Bytes are moved, so results are equal."""
import numpy as np
import pytest

from test_gpu_layout_runs import _exchange

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("to_dense", [True, False])
@pytest.mark.parametrize("dtype", [np.uint8, np.uint16])
@pytest.mark.parametrize("n_long,mid,n_run", [(1, 3, 1), (17, 2, 9), (130, 9, 32), (130, 9, 33), (129, 342, 65), (129, 341, 65),
                                              (129, 513, 20), (129, 512, 20), (65, 205, 160), (65, 204, 160)])
def test_pieces(gpu, oracle, n_long, mid, n_run, dtype, to_dense):
    _exchange(oracle, n_long, mid, n_run, dtype, 5, 0, to_dense)
