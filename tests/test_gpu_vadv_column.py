"""Vertical advection of columns up to 80 levels: every number of 8-level blocks, at the depths where a block fills or
overflows by one level, and the strip counts (64 columns each) that change the wavefronts per SIMD, the load-ahead or
the number of launches; and the two wavefronts per strip that few strips take from 33 to 144 levels, at every number of
blocks.  FP64 and the native FP32 and mixed forms equal the oracle bit for bit, so the tolerance is
zero."""
import numpy as np
import pytest

from test_gpu_vadv_deep import FORMS, _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nk", [2, 3, 7, 8, 9, 15, 16, 17, 24, 25, 32, 33, 40, 41, 48, 49, 56, 57, 64, 65, 72, 73, 80])
@pytest.mark.parametrize("dtype,precision,mode", FORMS)
def test_depths(gpu, oracle, nk, dtype, precision, mode):
    _check(gpu, oracle, 131, 4, nk, dtype, precision, mode)


# two strips per row; strips per SIMD on 256 CUs: 0.9, 1.5, 2.7 and 4.7
@pytest.mark.parametrize("nj", [450, 750, 1400, 2400])
@pytest.mark.parametrize("nk", [2, 8, 9, 20, 31, 34, 42, 56, 61, 70, 80])
@pytest.mark.parametrize("dtype,precision,mode", FORMS)
def test_strips_per_simd(gpu, oracle, nj, nk, dtype, precision, mode):
    _check(gpu, oracle, 65, nj, nk, dtype, precision, mode)


# strips of 64 columns from 150 MiB per field (mixed: 300 MiB): a launch per round, the last one partly filled
@pytest.mark.parametrize("nj,nk,dtype,precision,mode",
                         [(4700, 33, np.float64, 0, "native"), (9400, 33, np.float32, 0, "native"),
                          (7777, 80, np.float32, 1, "mixed")])
def test_launch_per_round(gpu, oracle, nj, nk, dtype, precision, mode):
    _check(gpu, oracle, 65, nj, nk, dtype, precision, mode)


# 512 strips, the most that run on two wavefronts each on 256 CUs, and 513; partial strips; the block edges
@pytest.mark.parametrize("ni,nj", [(1, 1), (70, 3), (64, 512), (65, 256), (64, 513)])
@pytest.mark.parametrize("nk", [32, 33, 48, 81, 103, 104, 105, 112, 113, 136, 144, 145])
@pytest.mark.parametrize("dtype,precision,mode", FORMS)
def test_two_wavefronts_per_strip(gpu, oracle, ni, nj, nk, dtype, precision, mode):
    _check(gpu, oracle, ni, nj, nk, dtype, precision, mode)
