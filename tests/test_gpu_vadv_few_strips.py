"""FP64 vertical advection of 25 to 32 levels where at most half the SIMDs have a strip (8 levels of load-ahead) and just past
that, at the block's edges and with partial strips, and of 41 and more levels where 9/8 to 3/2 strips per SIMD take two
launches; the bits of the oracle, so the tolerance is zero."""
import numpy as np
import pytest

from test_gpu_vadv_deep import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,nj", [(1, 1), (70, 3), (64, 512), (65, 256), (64, 513)])  # 512 strips: half of 256 CUs' SIMDs
@pytest.mark.parametrize("nk", [24, 25, 31, 32])
def test_load_ahead(gpu, oracle, ni, nj, nk):
    _check(gpu, oracle, ni, nj, nk, np.float64, 0, "native")


@pytest.mark.parametrize("nj", [1151, 1152, 1153, 1535, 1536, 1537])  # strips on 1024 SIMDs: two launches from 9/8 to 3/2
@pytest.mark.parametrize("nk", [41, 80])
def test_two_launches(gpu, oracle, nj, nk):
    _check(gpu, oracle, 50, nj, nk, np.float64, 0, "native")
