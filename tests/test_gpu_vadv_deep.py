"""Vertical advection of columns past the register buckets (nk > 80): the split of a column over registers, LDS and
the wavefront's scratch, at the depths where a part fills, overflows by one level or ends inside a block of eight
levels.  FP64 and the native FP32 and mixed forms equal the oracle bit for bit, so the tolerance is zero."""
import numpy as np
import pytest

from test_gpu_stencils import oracle_vadv, vadv_case

pytestmark = pytest.mark.gpu

# register parts of 80, 96 and 128 levels, with 16 or 40 LDS levels behind them
DEPTHS = [81, 88, 89, 96, 97, 112, 113, 120, 121, 128, 129, 136, 137, 144, 145, 153, 200]
FORMS = [(np.float64, 0, "native"), (np.float32, 0, "native"), (np.float32, 1, "mixed")]


def _check(gt, oracle, ni, nj, nk, dtype, precision, mode, noalloc=False):
    from gridtools_amd import _abi, stencils
    import ctypes

    print(f"[case] vadv deep {np.dtype(dtype).name} prec={precision} {ni}x{nj}x{nk} noalloc={noalloc}", flush=True)
    f, grid = vadv_case(gt, ni, nj, nk, dtype)
    dtr = 0.15 if dtype == np.float64 else float(np.float32(0.15))
    ref = oracle_vadv(oracle, f, dtr, 3, ni, nj, nk, mode)
    order = ("utens_stage", "u_stage", "wcon", "u_pos", "utens")
    if noalloc:
        s = [f[n].sid(grid.origin) for n in order]
        _abi.call("gt355_vadv_noalloc", precision, *[ctypes.byref(x) for x in s], ctypes.c_double(dtr), ni, nj, nk, None)
    else:
        stencils.vadv(*[f[n] for n in order], dtr, grid, precision=precision)
    got = f["utens_stage"].padded_numpy()[:nk, 3:3 + nj, 3:3 + ni]
    assert np.array_equal(got, ref, equal_nan=True)


@pytest.mark.parametrize("nk", DEPTHS)
@pytest.mark.parametrize("dtype,precision,mode", FORMS)
def test_depths(gpu, oracle, nk, dtype, precision, mode):
    _check(gpu, oracle, 67, 5, nk, dtype, precision, mode)


@pytest.mark.parametrize("nk", [81, 120, 137, 150])
@pytest.mark.parametrize("dtype,precision,mode", FORMS)
def test_several_strips_per_wavefront(gpu, oracle, nk, dtype, precision, mode):
    """More strips than one wavefront per SIMD (1024 on 256 CUs): the next strip's loads start in the sweep before."""
    _check(gpu, oracle, 130, 720, nk, dtype, precision, mode)


@pytest.mark.parametrize("ni,nj,nk", [(1, 1, 81), (64, 3, 137), (5, 40, 300)])
@pytest.mark.parametrize("dtype,precision,mode", FORMS)
def test_no_alloc_entry(gpu, oracle, ni, nj, nk, dtype, precision, mode):
    _check(gpu, oracle, ni, nj, nk, dtype, precision, mode, noalloc=True)
