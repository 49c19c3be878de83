"""Paths that single shapes of the other files do not reach: every block edge of the one-wavefront column sweep (with more than
512 strips, the most that two wavefronts each solve), non-finite top levels past 80 levels there and in the batch's depth
classes, and fields whose row and level strides differ.  Equal to the oracle bit for bit, so the tolerance is zero."""
import numpy as np
import pytest

from test_gpu_inf_top import H, _inject, _oracle, _run, _store
from test_gpu_stencils import SEED
from test_gpu_vadv_deep import FORMS, _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nk", [40, 41, 49, 57, 64, 65, 73, 81, 88, 89, 96, 97, 104, 105, 128, 129, 153])
@pytest.mark.parametrize("dtype,precision,mode", FORMS)
def test_column_sweep_block_edges(gpu, oracle, nk, dtype, precision, mode):
    _check(gpu, oracle, 65, 300, nk, dtype, precision, mode)


@pytest.mark.parametrize("nj", [6144, 6145])  # two strips per row: 12 strips per SIMD on 256 CUs, and more
@pytest.mark.parametrize("nk", [8, 9, 16])
def test_many_strips(gpu, oracle, nk, nj):
    """One wavefront per SIMD for FP64 of 9 to 16 levels past 12 strips per SIMD."""
    _check(gpu, oracle, 65, nj, nk, np.float64, 0, "native")


def _inf_fields(ni, nj, nk, dtype):
    rng = np.random.default_rng(ni * 7 + nk)
    shp = (nk, nj + 2 * H, ni + 2 * H)
    fl = [rng.uniform(-1, 1, shp) for _ in range(2)] + [rng.uniform(-0.5, 0.5, (nk + 1,) + shp[1:])] + \
         [rng.uniform(-1, 1, shp) for _ in range(2)]
    fl = [a.astype(dtype) for a in fl]
    _inject(rng, fl[1], ni, nj, nk, 12)
    fl[2][nk, H:H + nj, H:H + ni + 1] = np.inf  # never read
    return fl


def _inf_reference(oracle, fl, ni, nj, nk, dtype, precision):
    dtr = 0.15 if dtype == np.float64 else float(np.float32(0.15))
    ref = _oracle(oracle, [a.astype(np.float64) for a in fl] if precision else fl, dtr, ni, nj, nk, "native")
    assert np.isnan(ref).any() and np.isinf(ref).any()
    return ref.astype(dtype)


@pytest.mark.parametrize("ni,nj,nk", [(65, 300, 86), (65, 300, 95), (65, 300, 120), (65, 300, 150), (65, 300, 165)])
@pytest.mark.parametrize("dtype,precision", [(np.float64, 0), (np.float32, 0), (np.float32, 1)])
def test_inf_top_deep(gpu, oracle, ni, nj, nk, dtype, precision):
    print(f"[case] vadv inf-top {np.dtype(dtype).name} prec={precision} {ni}x{nj}x{nk}", flush=True)
    fl = _inf_fields(ni, nj, nk, dtype)
    ref = _inf_reference(oracle, fl, ni, nj, nk, dtype, precision)
    np.testing.assert_array_equal(_run(gpu, fl, 0.15, ni, nj, nk, dtype, precision), ref)


@pytest.mark.parametrize("dtype,precision", [(np.float64, 0), (np.float32, 0), (np.float32, 1)])
def test_inf_top_batch(gpu, oracle, dtype, precision):
    """The vertical phase alone: a domain in the shallowest depth class, in one of the middle and in the deepest ones."""
    from gridtools_amd.batch import Batch

    members, refs = [], []
    for ni, nj, nk in [(70, 9, 17), (33, 20, 60), (64, 6, 100), (65, 8, 137)]:
        fl = _inf_fields(ni, nj, nk, dtype)
        refs.append(_inf_reference(oracle, fl, ni, nj, nk, dtype, precision))
        m = dict(zip(("utens_stage", "u_stage", "wcon", "u_pos", "utens"), (_store(gpu, a, dtype) for a in fl)))
        m["grid"] = gpu.make_grid(gpu.halo_descriptor.symmetric(H, ni + 2 * H), gpu.halo_descriptor.symmetric(H, nj + 2 * H), nk)
        members.append(dict(m, phases=2))
    Batch(members, precision=precision).run(0.15)
    gpu.synchronize()
    for m, ref in zip(members, refs):
        nk, nj, ni = ref.shape
        np.testing.assert_array_equal(m["utens_stage"].to_numpy().transpose(2, 1, 0)[:, H:H + nj, H:H + ni], ref)


def _field(gt, name, lo, hi, size, h, dtype, more=(0, 0)):
    """A field with `more` points behind its interior and halo, which only its strides show."""
    from gridtools_amd import inputs

    b = gt.builder().type(dtype).dimensions(size[0] + 2 * h + more[0], size[1] + 2 * h + more[1], size[2]).halos(h, h, 0)
    return b.uniform(SEED, inputs.FIELD_IDS[name], lo, hi).build() if name else b.value(0).build()


@pytest.mark.parametrize("ni,nj,nk", [(61, 9, 4), (130, 33, 5), (64, 20, 7)])
@pytest.mark.parametrize("impl", [None, 1, 2, 3])
@pytest.mark.parametrize("dtype,precision,mode", FORMS)
def test_hdiff_strides(gpu, oracle, monkeypatch, ni, nj, nk, impl, dtype, precision, mode):
    from gridtools_amd import stencils

    if impl is not None:
        monkeypatch.setenv("GT355_TUNE_hdiff_impl", str(impl))
    inp = _field(gpu, "in", -1.0, 1.0, (ni, nj, nk), 2, dtype, (70, 3))
    coeff = _field(gpu, "coeff", 0.0, 0.25, (ni, nj, nk), 2, dtype, (140, 1))
    out = _field(gpu, None, 0, 0, (ni, nj, nk), 2, dtype, (0, 5))
    assert len({(f.strides[1], f.strides[2]) for f in (inp, coeff, out)}) == 3
    grid = gpu.make_grid(gpu.halo_descriptor.symmetric(2, ni + 4), gpu.halo_descriptor.symmetric(2, nj + 4), nk)
    stencils.hdiff(out, inp, coeff, grid, precision=precision)
    # the oracle takes one layout: the points that hdiff reads of each
    a_in, a_co = (np.ascontiguousarray(f.padded_numpy()[:nk, :nj + 4, :ni + 4]) for f in (inp, coeff))
    res, V = np.zeros_like(a_in), oracle.View
    oracle.hdiff(V(res, 2, 2), V(a_in, 2, 2), V(a_co, 2, 2), ni, nj, nk, mode=mode, threads=8)
    full = out.padded_numpy()
    assert np.array_equal(full[:nk, 2:2 + nj, 2:2 + ni], res[:, 2:2 + nj, 2:2 + ni])
    full[:nk, 2:2 + nj, 2:2 + ni] = 0
    assert not full.any()  # nothing outside the domain is written


@pytest.mark.parametrize("ni,nj,nk", [(61, 9, 30), (61, 9, 70), (65, 300, 70), (65, 300, 130)])
@pytest.mark.parametrize("dtype,precision,mode", FORMS)
def test_vadv_strides(gpu, oracle, ni, nj, nk, dtype, precision, mode):
    from gridtools_amd import stencils

    f = {n: _field(gpu, n, -1.0, 1.0, (ni, nj, nk), 3, dtype) for n in ("utens_stage", "u_stage", "u_pos", "utens")}
    f["wcon"] = _field(gpu, "wcon", -0.5, 0.5, (ni, nj, nk + 1), 3, dtype, (70, 2))
    assert f["wcon"].strides[1] != f["utens"].strides[1] and f["wcon"].strides[2] != f["utens"].strides[2]
    grid = gpu.make_grid(gpu.halo_descriptor.symmetric(3, ni + 6), gpu.halo_descriptor.symmetric(3, nj + 6), nk)
    dtr = 0.15 if dtype == np.float64 else float(np.float32(0.15))
    a = {n: np.ascontiguousarray(v.padded_numpy()[:, :nj + 6, :ni + 6]) for n, v in f.items()}
    ref, V = a["utens_stage"].copy(), oracle.View
    oracle.vadv(V(ref, 3, 3), *(V(a[n], 3, 3) for n in ("u_stage", "wcon", "u_pos", "utens")), dtr, ni, nj, nk, mode=mode,
                threads=8)
    stencils.vadv(*[f[n] for n in ("utens_stage", "u_stage", "wcon", "u_pos", "utens")], dtr, grid, precision=precision)
    assert np.array_equal(f["utens_stage"].padded_numpy()[:nk, 3:3 + nj, 3:3 + ni], ref[:nk, 3:3 + nj, 3:3 + ni])
