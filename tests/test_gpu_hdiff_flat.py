"""The flat column-pair hdiff sweep against the oracle, bit for bit (so the tolerance is zero): rows narrower than,
equal to and just past what a wavefront outputs (60 pairs), odd and even widths, row blocks that end short of a whole
block of four rows, single levels, fields whose rows start unaligned, and the shapes the default rule sends to it."""
import numpy as np
import pytest

from test_gpu_stencils import hdiff_case, oracle_hdiff

pytestmark = pytest.mark.gpu

FORMS = [(np.float64, 0, "native"), (np.float32, 0, "native"), (np.float32, 1, "mixed")]
SIZES = [(2, 4, 1), (3, 5, 2), (5, 7, 61), (12, 33, 61), (59, 8, 3), (117, 9, 2), (118, 6, 3), (119, 4, 2), (120, 11, 2),
         (121, 10, 2), (125, 13, 1), (387, 25, 3)]


def _run(gt, oracle, ni, nj, nk, dtype, precision, mode, shift=0):
    from gridtools_amd import stencils
    from gridtools_amd.grid import Grid

    print(f"[case] hdiff flat {np.dtype(dtype).name} prec={precision} {ni}x{nj}x{nk} shift={shift}", flush=True)
    inp, coeff, out, grid = hdiff_case(gt, ni, nj, nk, dtype)
    ref = oracle_hdiff(oracle, inp, coeff, 2, ni, nj, nk, mode)
    if shift:  # the interior without its first columns and rows: an unaligned origin
        grid = Grid(2 + shift, ni - shift, 2 + shift, nj - shift, nk)
    stencils.hdiff(out, inp, coeff, grid, precision=precision)
    full = out.padded_numpy()[:nk]
    assert np.array_equal(full[:, 2 + shift:2 + nj, 2 + shift:2 + ni], ref[:, shift:, shift:])
    # nothing outside the computed domain is written
    full[:, 2 + shift:2 + nj, 2 + shift:2 + ni] = 0
    assert not full.any()


@pytest.mark.parametrize("jb,p", [(4, 8), (2, 6)])
@pytest.mark.parametrize("ni,nj,nk", SIZES + [(119, 2, 3), (120, 3, 2), (64, 5, 4)])
@pytest.mark.parametrize("dtype,precision,mode", FORMS)
def test_sizes_by_rows(gpu, oracle, monkeypatch, jb, p, ni, nj, nk, dtype, precision, mode):
    """Four and two rows per wavefront, with the fewest rows each takes and one less."""
    monkeypatch.setenv("GT355_TUNE_hdiff_impl", "3")
    monkeypatch.setenv("GT355_TUNE_hdiff_jb", str(jb))
    monkeypatch.setenv("GT355_TUNE_hdiff_p", str(p))
    _run(gpu, oracle, ni, nj, nk, dtype, precision, mode)


# the sizes around each line of the default rule: 36, 128 (512 columns) and 400 MiB of FP64 fields
@pytest.mark.parametrize("ni,nj,nk", [(128, 150, 80), (130, 152, 80), (512, 200, 50), (513, 250, 44), (512, 270, 41),
                                      (640, 400, 69), (301, 700, 84)])
@pytest.mark.parametrize("dtype,precision,mode", FORMS)
def test_default_rule_by_size(gpu, oracle, ni, nj, nk, dtype, precision, mode):
    _run(gpu, oracle, ni, nj, nk, dtype, precision, mode)


@pytest.mark.parametrize("ni,nj,nk", SIZES)
@pytest.mark.parametrize("dtype,precision,mode", FORMS)
def test_sizes(gpu, oracle, monkeypatch, ni, nj, nk, dtype, precision, mode):
    monkeypatch.setenv("GT355_TUNE_hdiff_impl", "3")
    _run(gpu, oracle, ni, nj, nk, dtype, precision, mode)


@pytest.mark.parametrize("ni", [66, 67])
@pytest.mark.parametrize("dtype,precision,mode", FORMS)
def test_unaligned_rows(gpu, oracle, monkeypatch, ni, dtype, precision, mode):
    monkeypatch.setenv("GT355_TUNE_hdiff_impl", "3")
    _run(gpu, oracle, ni, 14, 3, dtype, precision, mode, shift=1)


@pytest.mark.parametrize("ni,nj,nk", [(1, 9, 3), (130, 3, 2), (130, 41, 5), (251, 40, 3), (300, 17, 4)])
@pytest.mark.parametrize("dtype,precision,mode", FORMS)
def test_default_rule(gpu, oracle, ni, nj, nk, dtype, precision, mode):
    """Ragged widths by default, with the shapes it refuses (one column, fewer than four rows) on the sweeps."""
    _run(gpu, oracle, ni, nj, nk, dtype, precision, mode)
