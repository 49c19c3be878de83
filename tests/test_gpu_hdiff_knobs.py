"""GT355_TUNE_hdiff_jb and GT355_TUNE_hdiff_p set alone, on fields whose default shape is the flat pair sweep, the strips or
the rule for large fields: each names a shape of the strips of that width, runs and equals the oracle bit for bit (so the
tolerance is zero); a value that no strip shape of that width has is refused with a status."""
import ctypes

import numpy as np
import pytest

from test_gpu_stencils import hdiff_case, oracle_hdiff

pytestmark = pytest.mark.gpu

KNOBS = [("jb", 4), ("jb", 8), ("jb", 16), ("jb", 32), ("p", 4), ("p", 8), ("jb", 7), ("p", 5)]
# (rows, rows ahead) of the strips: one column per lane, two columns per lane
ONE, PAIRS = {(4, 4), (8, 4), (16, 4), (16, 8), (32, 4), (32, 8)}, {(4, 4), (8, 4), (8, 8), (16, 4), (16, 8)}


@pytest.mark.parametrize("knob,value", KNOBS)
@pytest.mark.parametrize("ni,nj,nk,dtype", [(64, 64, 20, np.float64), (65, 33, 7, np.float64), (64, 64, 20, np.float32),
                                            (520, 40, 9, np.float64), (300, 700, 84, np.float64)])
def test_one_knob(gpu, oracle, monkeypatch, ni, nj, nk, dtype, knob, value):
    from gridtools_amd import _abi

    print(f"[case] hdiff {knob}={value} {np.dtype(dtype).name} {ni}x{nj}x{nk}", flush=True)
    monkeypatch.setenv(f"GT355_TUNE_hdiff_{knob}", str(value))
    shape = (value, 4) if knob == "jb" else (8, value)
    runs = shape in (PAIRS if dtype == np.float32 or ni >= 512 else ONE)
    inp, coeff, out, grid = hdiff_case(gpu, ni, nj, nk, dtype)
    sids = [ctypes.byref(f.sid(grid.origin)) for f in (out, inp, coeff)]
    rc = _abi.lib().gt355_hdiff(0, *sids, ni, nj, nk, None)
    assert rc == (0 if runs else -4), _abi.last_error()
    ref = oracle_hdiff(oracle, inp, coeff, 2, ni, nj, nk, "native") if runs else 0
    assert np.array_equal(out.padded_numpy()[:nk, 2:2 + nj, 2:2 + ni], np.broadcast_to(ref, (nk, nj, ni)))


@pytest.mark.parametrize("cfg", [(2, 2, 6, 1), (2, 4, 8, 1), (1, 16, 4, 0), (2, 16, 4, 0)])
def test_knob_over_a_tuned_entry(gpu, oracle, monkeypatch, cfg):
    """A tuned entry of the strips keeps its other value, one of the flat sweep gives way to the strips'."""
    from gridtools_amd import stencils, tune

    ni, nj, nk = 64, 40, 9
    tune.clear()
    try:
        tune.store("hdiff", (8, 8, ni, nj, nk), cfg)
        monkeypatch.setenv("GT355_TUNE_hdiff_jb", "16")
        inp, coeff, out, grid = hdiff_case(gpu, ni, nj, nk, np.float64)
        stencils.hdiff(out, inp, coeff, grid)
    finally:
        tune.clear()
    ref = oracle_hdiff(oracle, inp, coeff, 2, ni, nj, nk, "native")
    assert np.array_equal(out.padded_numpy()[:nk, 2:2 + nj, 2:2 + ni], ref)
