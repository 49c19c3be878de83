"""The calls whose speed is measured: what a program using this framework has it do per timestep.

Each case is one call (or one timestep) through the Python entry points, on fields laid out by ``DataStore`` with the
halo its stencil needs, over the sizes of the regression tests, the benchmark and the batched workload:

* ``hdiff``: horizontal diffusion, from the reference's verification domain to the benchmark's and a ragged one;
* ``vadv``: vertical advection, from the smallest domain of the batched workload to the benchmark's, a ragged one
  and a deep column;
* ``compose``: hdiff followed by vadv of its result in one call;
* ``timestep``: the large domain's step, composition and boundary conditions;
* ``batch``: uneven domains in one batched call;
* ``tracers``: the expandable prepare_tracers over many members;
* ``layout``: a field to a k-fastest dense array and back.

Precision is "f64" (FP64 storage), "f32" (FP32 storage and arithmetic) or "mixed" (FP32 storage, FP64 arithmetic).
"""
import ctypes
import math

import numpy as np
import torch

from gridtools_amd import boundaries, stencils
from gridtools_amd.batch import Batch
from gridtools_amd.grid import halo_descriptor, make_grid
from gridtools_amd.layout import transform_layout
from gridtools_amd.storage import DataStore
from gridtools_amd.timestep import HdiffVadvTimestepper

HALO = 3  # the benchmark's halo (hdiff needs 2, vadv 1)
DTR = 0.15
DEV = "cuda"


def listed():
    return [
        # the reference's own verification domain: a call whose cost is its latency
        {"name": "hdiff_smallest_f64", "kind": "hdiff", "ni": 12, "nj": 33, "nk": 61, "prec": "f64"},
        # the headline domain in double precision
        {"name": "hdiff_f64", "kind": "hdiff", "ni": 256, "nj": 256, "nk": 80, "prec": "f64"},
        # a subdomain of a decomposition that does not divide evenly (odd sizes), FP32 storage
        {"name": "hdiff_ragged_mixed", "kind": "hdiff", "ni": 387, "nj": 251, "nk": 61, "prec": "mixed"},
        # the smallest subdomain, single precision: one column solve per lane on a mostly idle chip
        {"name": "vadv_smallest_f32", "kind": "vadv", "ni": 48, "nj": 48, "nk": 40, "prec": "f32"},
        # the headline domain in double precision
        {"name": "vadv_f64", "kind": "vadv", "ni": 256, "nj": 256, "nk": 80, "prec": "f64"},
        # an uneven subdomain at a common level count, FP32 storage
        {"name": "vadv_ragged_mixed", "kind": "vadv", "ni": 235, "nj": 198, "nk": 60, "prec": "mixed"},
        # deep columns (137 levels, the deepest of the batched workload), double precision
        {"name": "vadv_deep_f64", "kind": "vadv", "ni": 192, "nj": 160, "nk": 137, "prec": "f64"},
        # the operator on the benchmark's composition domain
        {"name": "compose_f64", "kind": "compose", "ni": 512, "nj": 512, "nk": 80, "prec": "f64"},
        # one timestep of the large domain with its boundary conditions: the largest work
        {"name": "timestep_large_mixed", "kind": "timestep", "ni": 1536, "nj": 1536, "nk": 80, "bc": "fill"},
        # uneven domains of the batched workload's ranges
        {"name": "batch_mixed", "kind": "batch", "domains": 16, "sizes": 2024, "prec": "mixed"},
        # tracer preparation of eleven members on the headline domain
        {"name": "tracers_f64", "kind": "tracers", "ni": 256, "nj": 256, "nk": 80, "members": 11, "prec": "f64"},
        # data exchange with a model that keeps k fastest, on an uneven domain
        {"name": "layout_ragged_f64", "kind": "layout", "ni": 197, "nj": 261, "nk": 73, "prec": "f64"},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["hdiff", "hdiff", "vadv", "vadv", "compose", "timestep", "batch", "tracers", "layout"])
    prec = rng.choice(["f64", "f32", "mixed"])
    if kind == "hdiff":
        return {"kind": kind, "ni": log(12, 512), "nj": log(12, 512), "nk": rng.randint(20, 137), "prec": prec}
    if kind == "vadv":
        return {"kind": kind, "ni": log(32, 512), "nj": log(32, 512), "nk": rng.randint(20, 137), "prec": prec}
    if kind == "compose":
        return {"kind": kind, "ni": log(64, 512), "nj": log(64, 512), "nk": rng.randint(40, 137), "prec": prec}
    if kind == "timestep":
        return {"kind": kind, "ni": log(64, 1536), "nj": log(64, 1536), "nk": rng.randint(40, 80),
                "bc": rng.choice(["fill", "exchange"])}
    if kind == "batch":
        return {"kind": kind, "domains": rng.randint(4, 16), "sizes": rng.randint(0, 10**6),
                "prec": rng.choice(["f64", "mixed"])}
    if kind == "tracers":
        return {"kind": kind, "ni": log(32, 256), "nj": log(32, 256), "nk": rng.randint(40, 80),
                "members": rng.randint(2, 40), "prec": prec}
    return {"kind": kind, "ni": log(24, 512), "nj": log(24, 512), "nk": rng.randint(20, 137),
            "prec": rng.choice(["f64", "f32"])}


# ---------------------------------------------------------------------------------------------------- inputs
# value ranges of the fields: winds and tendencies U(-1, 1), diffusion coefficient U(0, 0.25); the vertical wind keeps
# the implicit system diagonally dominant (|a| + |c| <= 0.025 < dtr), as a stable timestep does
RANGES = {"in": (-1.0, 1.0), "coeff": (0.0, 0.25), "u_stage": (-1.0, 1.0), "u_pos": (-1.0, 1.0),
          "utens": (-1.0, 1.0), "utens_stage": (-1.0, 1.0), "wcon": (-0.05, 0.05), "rho": (0.5, 1.5),
          "tracer": (0.0, 1.0), "field": (-1.0, 1.0)}
IDS = {n: i for i, n in enumerate(RANGES)}


def _np_dtype(case):
    return np.float64 if case.get("prec", "mixed") == "f64" else np.float32


def _t_dtype(case):
    return torch.float64 if case.get("prec", "mixed") == "f64" else torch.float32


def _precision(case):
    return stencils.WIDEN if case.get("prec", "mixed") == "mixed" else stencils.NATIVE


def _values(name, seed, member, shape, dtype):
    """Seeded uniform values of a field, indexed [k, j, i]."""
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1009 + member) * 64 + IDS[name])
    lo, hi = RANGES[name]
    return torch.rand(shape, generator=g, device=DEV, dtype=dtype) * (hi - lo) + lo


class _Device:
    """The array interface of a field's memory; it holds the store, whose memory lives as long as the store does."""

    def __init__(self, ds):
        self.store = ds
        s = ds.dtype.itemsize
        self.__cuda_array_interface__ = {
            "shape": tuple(reversed(ds.lengths)), "strides": tuple(s * x for x in reversed(ds.strides)),
            "typestr": ds.dtype.str, "data": (ds.base, False), "version": 2}


def _view(ds):
    """The field's device memory as a tensor indexed [k, j, i], halo included, which keeps the store alive."""
    t = torch.as_tensor(_Device(ds), device=DEV)
    t.store = ds
    return t


def _inner(t, ni, nj):
    return t[:, HALO:HALO + nj, HALO:HALO + ni]


def _result(ds, ni, nj):
    """The field's interior as a tensor, which keeps the store alive."""
    t = _inner(_view(ds), ni, nj)
    t.store = ds
    return t


def _store(case, values):
    nk, nj, ni = values.shape
    ds = DataStore(_np_dtype(case), (ni, nj, nk), (HALO, HALO, 0))
    _view(ds).copy_(values)
    return ds


def _empty(case, ni, nj, nk):
    return DataStore(_np_dtype(case), (ni + 2 * HALO, nj + 2 * HALO, nk), (HALO, HALO, 0))


def _grid(ni, nj, nk):
    return make_grid(halo_descriptor.symmetric(HALO, ni + 2 * HALO), halo_descriptor.symmetric(HALO, nj + 2 * HALO), nk)


def _field(case, name, seed, member=0, size=None):
    ni, nj, nk = size or (case["ni"], case["nj"], case["nk"])
    extra = 1 if name == "wcon" else 0  # wcon lies on level interfaces
    return _values(name, seed, member, (nk + extra, nj + 2 * HALO, ni + 2 * HALO), _t_dtype(case))


def _bc_index(n, periodic):
    """Interior index (0-based in the padded field) that each point of a dimension with a halo takes its value from."""
    p = torch.arange(-HALO, n + HALO, device=DEV)
    return HALO + (p % n if periodic else p.clamp(0, n - 1))


def _with_bc(t, ni, nj):
    """t [k, j, i] with its halos filled: periodic in i, zero-gradient in j."""
    return t[:, _bc_index(nj, False)][:, :, _bc_index(ni, True)]


def _batch_sizes(case):
    """The domain sizes (ni, nj, nk) of a batched case: ni, nj in 48..384, nk in 40..137."""
    rng = np.random.default_rng(case["sizes"])
    n = case["domains"]
    ni, nj, nk = (rng.integers(lo, hi + 1, size=n) for lo, hi in ((48, 384), (48, 384), (40, 137)))
    return [(int(a), int(b), int(c)) for a, b, c in zip(ni, nj, nk)]


VADV = ("utens_stage", "u_stage", "wcon", "u_pos", "utens")


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "batch":
        members, outs = [], []
        for d, (ni, nj, nk) in enumerate(_batch_sizes(case)):
            m = {n: _store(case, _field(case, n, seed, d, (ni, nj, nk)))
                 for n in ("coeff", "utens_stage", "wcon", "u_pos", "utens")}
            m["in_"] = _store(case, _field(case, "in", seed, d, (ni, nj, nk)))
            m["lap"], m["u_stage"] = _empty(case, ni, nj, nk), _empty(case, ni, nj, nk)
            m["grid"] = _grid(ni, nj, nk)
            members.append(m)
            outs.append([_result(m[n], ni, nj) for n in ("lap", "u_stage", "utens_stage")])
        return dict(st, batch=Batch(members, precision=_precision(case)), outs=outs)
    ni, nj, nk = case["ni"], case["nj"], case["nk"]
    grid = _grid(ni, nj, nk)
    if kind == "hdiff":
        f = [_store(case, _field(case, n, seed)) for n in ("in", "coeff")]
        out = _empty(case, ni, nj, nk)
        return dict(st, grid=grid, f=f, out=out, precision=_precision(case), outs=_result(out, ni, nj))
    if kind == "vadv":
        f = [_store(case, _field(case, n, seed)) for n in VADV]
        return dict(st, grid=grid, f=f, precision=_precision(case), outs=_result(f[0], ni, nj))
    if kind == "compose":
        f = [_store(case, _field(case, n, seed)) for n in ("in", "coeff")]
        f.append(_empty(case, ni, nj, nk))
        f += [_store(case, _field(case, n, seed)) for n in ("utens_stage", "wcon", "u_pos", "utens")]
        return dict(st, grid=grid, f=f, precision=_precision(case),
                    outs=[_result(f[2], ni, nj), _result(f[3], ni, nj)])
    if kind == "timestep":
        ts = HdiffVadvTimestepper(ni, nj, nk, dtype=np.float32, halo=HALO, dtr=DTR, bc=case["bc"])
        _view(ts.u).copy_(_with_bc(_field(case, "in", seed), ni, nj))
        for n in ("coeff", "utens_stage", "wcon", "u_pos", "utens"):
            _view(getattr(ts, n)).copy_(_field(case, n, seed))
        return dict(st, ts=ts, views={id(s): _view(s) for s in (ts.u, ts.u_stage, ts.utens_stage)})
    if kind == "tracers":
        now = [_store(case, _field(case, "tracer", seed, m)) for m in range(case["members"])]
        data = [_empty(case, ni, nj, nk) for _ in now]
        return dict(st, grid=grid, data=data, now=now, rho=_store(case, _field(case, "rho", seed)),
                    precision=_precision(case), outs=[_result(d, ni, nj) for d in data])
    src, back = _store(case, _field(case, "field", seed)), _empty(case, ni, nj, nk)
    dense = torch.empty((ni, nj, nk), dtype=_t_dtype(case), device=DEV)
    return dict(st, src=src, back=back, dense=dense, dims=(ni, nj, nk), dstr=(nj * nk, nk, 1),
                outs=[dense, _result(back, ni, nj)])


def run(st):
    kind = st["case"]["kind"]
    if kind == "hdiff":
        stencils.hdiff(st["out"], *st["f"], st["grid"], precision=st["precision"])
    elif kind == "vadv":
        stencils.vadv(*st["f"], DTR, st["grid"], precision=st["precision"])
    elif kind == "compose":
        stencils.hdiff_vadv(*st["f"], DTR, st["grid"], precision=st["precision"])
    elif kind == "timestep":
        ts = st["ts"]
        ts.step()
        return [st["views"][id(ts.u)], st["views"][id(ts.utens_stage)]]
    elif kind == "batch":
        st["batch"].run(DTR)
    elif kind == "tracers":
        stencils.prepare_tracers(st["data"], st["now"], st["rho"], st["grid"], precision=st["precision"])
    else:
        src, back, dense, size = st["src"], st["back"], st["dense"], st["dense"].element_size()
        transform_layout(dense.data_ptr(), src.address(HALO, HALO, 0), st["dims"], st["dstr"], src.strides, size)
        transform_layout(back.address(HALO, HALO, 0), dense.data_ptr(), st["dims"], back.strides, st["dstr"], size)
    return st["outs"]


def work(case):
    kind, s = case["kind"], 8 if case.get("prec", "mixed") == "f64" else 4

    def hdiff(ni, nj, nk):  # reads in with its rim and coeff, writes the result
        return ((ni + 4) * (nj + 4) + 2 * ni * nj) * nk * s, 33 * ni * nj * nk

    def vadv(ni, nj, nk):  # reads five fields (wcon with one more column), rewrites utens_stage
        return (6 * ni + 1) * nj * nk * s, 40 * ni * nj * nk

    def total(sizes, parts):
        b = sum(p(*z)[0] for z in sizes for p in parts)
        f = sum(p(*z)[1] for z in sizes for p in parts)
        return {"bytes": b, "flops": f}

    if kind == "batch":  # one more output (the laplacian), one input less (the diffused field is made on the way)
        return total(_batch_sizes(case), (hdiff, vadv))
    ni, nj, nk = case["ni"], case["nj"], case["nk"]
    pts = ni * nj * nk
    if kind == "hdiff":
        return total([(ni, nj, nk)], (hdiff,))
    if kind == "vadv":
        return total([(ni, nj, nk)], (vadv,))
    if kind in ("compose", "timestep"):
        w = total([(ni, nj, nk)], (hdiff, vadv))
        w["bytes"] -= pts * s  # u_stage is written once; the solve need not read it from memory
        if kind == "timestep":  # the halos of two fields are written
            w["bytes"] += 2 * ((ni + 2 * HALO) * (nj + 2 * HALO) - ni * nj) * nk * s
        return w
    if kind == "tracers":
        return {"bytes": (2 * case["members"] + 1) * pts * s, "flops": case["members"] * pts}
    return {"bytes": 4 * pts * s, "flops": 0}


# ---------------------------------------------------------------------------------------------------- exact values
def _hdiff64(u, co, ni, nj):
    """Horizontal diffusion of u [k, j, i] (halo HALO) with coefficient co: (result, laplacian) on the interior."""
    def at(t, di, dj, r=0):  # the interior grown by r points, shifted
        j0, i0 = HALO - r + dj, HALO - r + di
        return t[:, j0:j0 + nj + 2 * r, i0:i0 + ni + 2 * r]

    lap = 4.0 * at(u, 0, 0, 1) - (at(u, 1, 0, 1) + at(u, 0, 1, 1) + at(u, -1, 0, 1) + at(u, 0, -1, 1))
    lc = lap[:, 1:-1, 1:-1]

    def flux(lp, l0, up, u0):
        r = lp - l0
        return torch.where(r * (up - u0) > 0, torch.zeros_like(r), r)

    c = at(u, 0, 0)
    flx, flx_m = flux(lap[:, 1:-1, 2:], lc, at(u, 1, 0), c), flux(lc, lap[:, 1:-1, :-2], c, at(u, -1, 0))
    fly, fly_m = flux(lap[:, 2:, 1:-1], lc, at(u, 0, 1), c), flux(lc, lap[:, :-2, 1:-1], c, at(u, 0, -1))
    return c - at(co, 0, 0) * (flx - flx_m + fly - fly_m), lc


def _vadv64(uts, us, wcon, up, ut, ni, nj, dtr):
    """Vertical advection on interior arrays [k, j, i]; wcon with its halo."""
    nk = us.shape[0]
    w = wcon[:, HALO:HALO + nj, HALO:HALO + ni + 1]
    w = 0.25 * (w[:, :, 1:] + w[:, :, :-1])  # wind at the column, per interface
    c, d = [], []
    for k in range(nk):
        rhs = dtr * up[k] + ut[k] + uts[k]
        diag = torch.full_like(rhs, dtr)
        if k > 0:
            a = -0.5 * w[k]
            rhs = rhs - a * (us[k - 1] - us[k])
            diag = diag - a
        if k < nk - 1:
            cc = 0.5 * w[k + 1]
            rhs = rhs - cc * (us[k + 1] - us[k])
            diag = diag - cc
        if k > 0:
            diag = diag - c[-1] * a
            rhs = rhs - d[-1] * a
        c.append(cc / diag)
        d.append(rhs / diag)
    out = torch.empty_like(us)
    x = d[-1]
    out[nk - 1] = dtr * (x - up[nk - 1])
    for k in range(nk - 2, -1, -1):
        x = d[k] - c[k] * x
        out[k] = dtr * (x - up[k])
    return out


def exact(case, seed):
    kind = case["kind"]
    dtr = DTR if case.get("prec", "mixed") == "f64" else float(np.float32(DTR))

    def f64(name, member=0, size=None):
        return _field(case, name, seed, member, size).double()

    def composed(member=0, size=None):
        ni, nj, nk = size or (case["ni"], case["nj"], case["nk"])
        u = f64("in", member, size)
        if kind == "timestep":
            u = _with_bc(u, ni, nj)
        us, lap = _hdiff64(u, f64("coeff", member, size), ni, nj)
        v = [_inner(f64(n, member, size), ni, nj) for n in ("utens_stage", "u_pos", "utens")]
        return us, _vadv64(v[0], us, f64("wcon", member, size), v[1], v[2], ni, nj, dtr), lap

    if kind == "batch":
        outs = []
        for d, size in enumerate(_batch_sizes(case)):
            us, uts, lap = composed(d, size)
            outs.append([lap, us, uts])
        return outs
    ni, nj, nk = case["ni"], case["nj"], case["nk"]
    if kind == "hdiff":
        return _hdiff64(f64("in"), f64("coeff"), ni, nj)[0]
    if kind == "vadv":
        v = {n: _inner(f64(n), ni, nj) for n in VADV if n != "wcon"}
        return _vadv64(v["utens_stage"], v["u_stage"], f64("wcon"), v["u_pos"], v["utens"], ni, nj, dtr)
    if kind == "compose":
        return list(composed()[:2])
    if kind == "timestep":
        i, j = _bc_index(ni, True) - HALO, _bc_index(nj, False) - HALO
        return [t[:, j][:, :, i] for t in composed()[:2]]
    if kind == "tracers":
        rho = _inner(f64("rho"), ni, nj)
        return [rho * _inner(f64("tracer", m), ni, nj) for m in range(case["members"])]
    v = _inner(_field(case, "field", seed), ni, nj)
    return [v.permute(2, 1, 0).contiguous(), v]
