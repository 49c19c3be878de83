"""The scratch of the vertical advection past 80 levels: what a call keeps allocated, columns of few lanes, buffers that hold
fewer wavefronts than a domain has strips, chunks of rows, and captured shapes that have not run themselves.  FP64 and the
native FP32 and mixed forms equal the oracle bit for bit, so the tolerance is zero."""
import ctypes

import numpy as np
import pytest

from test_gpu_stencils import oracle_vadv, vadv_case
from test_gpu_vadv_deep import FORMS, _check

pytestmark = pytest.mark.gpu

ORDER = ("utens_stage", "u_stage", "wcon", "u_pos", "utens")
STREAMS = []  # kept: a stream made later must not get the handle, and with it the scratch, of one of these


def _stream():
    from gridtools_amd.timing import Stream

    STREAMS.append(Stream())
    return STREAMS[-1]


def _free_bytes():
    from gridtools_amd import _abi

    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert _abi.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_pool_holds_what_the_launch_uses(gpu):
    """512x512 columns of 100 levels keep every ccol/dcol on chip: no more than the pool's 64 MiB are allocated for them
    (all of them would take 417 MB)."""
    from gridtools_amd import stencils

    f, grid = vadv_case(gpu, 512, 512, 100, np.float64)
    st = _stream()
    st.synchronize()
    before = _free_bytes()
    stencils.vadv(*[f[n] for n in ORDER], 0.15, grid, stream=st.handle)
    st.synchronize()
    assert before - _free_bytes() < 128 << 20


# few lanes per strip at depths that leave levels to the scratch, more strips than SIMDs; the last two go to the kernel that
# keeps all levels there, for their depth and for the 256 MiB that the pool gives such domains
@pytest.mark.parametrize("ni,nj,nk", [(1, 1100, 200), (3, 1100, 300), (31, 1030, 153), (32, 1030, 153), (2, 1030, 400),
                                      (2, 1030, 420)])
@pytest.mark.parametrize("dtype,precision,mode", FORMS)
def test_few_lanes(gpu, oracle, ni, nj, nk, dtype, precision, mode):
    _check(gpu, oracle, ni, nj, nk, dtype, precision, mode)


# 64 MiB of scratch: fewer wavefronts than strips; few lanes, all rows at once; not a quarter of the wavefronts, three chunks
# of rows (FP32: two); few lanes in two chunks
@pytest.mark.parametrize("ni,nj,nk", [(40, 1100, 300), (3, 1100, 300), (40, 260, 1200), (3, 2100, 700)])
@pytest.mark.parametrize("dtype,precision,mode", FORMS)
def test_no_alloc_small_buffer(gpu, oracle, ni, nj, nk, dtype, precision, mode):
    _check(gpu, oracle, ni, nj, nk, dtype, precision, mode, noalloc=True)


def test_captured_shapes_that_have_not_run(gpu, oracle):
    """After 300x300x97 (139 MB of ccol/dcol, none of it in scratch) shapes of less ccol/dcol may be captured: in fewer
    wavefronts, or in chunks of rows; one of more may not."""
    from gridtools_amd import _abi, stencils
    from gridtools_amd.timestep import capture

    st = _stream()
    f, grid = vadv_case(gpu, 300, 300, 97, np.float64)
    stencils.vadv(*[f[n] for n in ORDER], 0.15, grid, stream=st.handle)
    st.synchronize()
    for ni, nj, nk in ((40, 260, 700), (3, 2100, 700), (48, 40, 97)):
        print(f"[case] captured vadv {ni}x{nj}x{nk}", flush=True)
        f, grid = vadv_case(gpu, ni, nj, nk, np.float64)
        host = f["utens_stage"].to_numpy()
        ref = oracle_vadv(oracle, f, 0.15, 3, ni, nj, nk, "native")
        graph = capture(st, lambda s: stencils.vadv(*[f[n] for n in ORDER], 0.15, grid, stream=s.handle))
        for _ in range(2):
            f["utens_stage"].from_numpy(host)
            graph.launch(st)
            st.synchronize()
            assert np.array_equal(f["utens_stage"].padded_numpy()[:nk, 3:3 + nj, 3:3 + ni], ref)
    ni, nj, nk = 600, 512, 100
    f, grid = vadv_case(gpu, ni, nj, nk, np.float64)
    sids = [f[n].sid(grid.origin) for n in ORDER]
    _abi.call("gt355_graph_begin", st.handle)
    try:
        rc = _abi.lib().gt355_vadv(0, *sids, ctypes.c_double(0.15), ni, nj, nk, st.handle)
    finally:
        g = ctypes.c_void_p()
        _abi.call("gt355_graph_end", st.handle, ctypes.byref(g))
        if g.value:
            _abi.lib().gt355_graph_destroy(g)
    assert rc == -4 and "outside capture" in _abi.last_error()
