"""transform_layout where one of the transposed extents is short and moves as whole runs (lt_run_kernel), against the
oracle: extents of one or two accesses, at and past the longest run, partial lines of the other dimension, either
direction, rows aligned on one side only, a broadcast source dimension, every element size, and arrays large enough
for non-temporal accesses.  Bytes are moved, so results are equal."""
import numpy as np
import pytest

from test_gpu_layout import run_both

pytestmark = pytest.mark.gpu


def _exchange(oracle, n_long, mid, n_run, dtype, pad, off=0, to_dense=True):
    """A padded [run][mid][long_padded] array to a dense [long][mid][run] one, or back; `pad` elements behind each
    padded row, the padded array starting `off` elements into its buffer."""
    rng = np.random.default_rng(n_long * 7 + n_run)
    row = n_long + pad
    padded = rng.integers(0, 100, size=off + n_run * mid * row).astype(dtype)
    dense = rng.integers(0, 100, size=n_long * mid * n_run).astype(dtype)
    dims, p_st, d_st = [n_long, mid, n_run], [1, row, row * mid], [mid * n_run, n_run, 1]
    print(f"[case] layout run {dims} {np.dtype(dtype).name} pad={pad} off={off} to_dense={to_dense}", flush=True)
    from gridtools_amd import layout
    from test_gpu_layout import DevBuf

    d_p, d_d = DevBuf(padded), DevBuf(dense)
    p_ptr = d_p.p.value + off * padded.itemsize
    if to_dense:
        layout.transform_layout(d_d.p.value, p_ptr, dims, d_st, p_st, elem_size=padded.itemsize)
        want = dense.copy()
        oracle.transform_layout(want, padded[off:], dims, d_st, p_st)
        assert np.array_equal(d_d.get(dense), want)
    else:
        layout.transform_layout(p_ptr, d_d.p.value, dims, p_st, d_st, elem_size=padded.itemsize)
        want = padded.copy()
        oracle.transform_layout(want[off:], dense, dims, p_st, d_st)
        assert np.array_equal(d_p.get(padded), want)


@pytest.mark.parametrize("to_dense", [True, False])
@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.float32, np.float64])
@pytest.mark.parametrize("n_long,n_run", [(2, 2), (33, 2), (197, 3), (48, 4), (197, 73), (161, 64), (130, 160), (300, 161)])
def test_runs(gpu, oracle, n_long, n_run, dtype, to_dense):
    """Rows padded to 16-byte multiples (vector accesses on the padded side) and dense rows of every alignment."""
    _exchange(oracle, n_long, 5, n_run, dtype, (-n_long) % 16 + 16, 0, to_dense)


@pytest.mark.parametrize("to_dense", [True, False])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("pad,off", [(1, 0), (15, 1), (0, 3)])
def test_unaligned_rows(gpu, oracle, dtype, pad, off, to_dense):
    _exchange(oracle, 97, 3, 20, dtype, pad, off, to_dense)


def test_broadcast_source(gpu, oracle):
    """A masked (stride 0) source dimension next to the transposed pair."""
    src = np.arange(7 * 40, dtype=np.float64)
    dst0 = np.zeros((40, 6, 7))
    got, want = run_both(oracle, dst0, src, [40, 6, 7], [42, 7, 1], [1, 0, 40])
    assert np.array_equal(got, want)


@pytest.mark.parametrize("to_dense", [True, False])
def test_large_arrays(gpu, oracle, to_dense):
    """64 MiB and more: non-temporal accesses on the aligned side."""
    _exchange(oracle, 301, 219, 137, np.float64, 3, 0, to_dense)
