"""Fused forms that must return the same bits as the forms they replace.

* fv3_fvtp2d_corner_fill: CopyCornersXY(q, q_x = q, q_y) + fv_tp_2d in one
  call (the y corner fill applied as the transport reads q) against the two
  calls, on domains with all four and with two cube corners.
* fv_tp_2d segment height: the rows of a segment follow from the launch's size;
  output rows are computed the same way in any, so one call on 64 C48 tiles must
  equal eight calls on 8 tiles each, which take segments of another height, bit
  for bit, FP64 and FP32.
* map_single: the launcher chooses between one thread per column (four sweeps,
  or fused) and layers spread over a workgroup by layer count and columns.
  Columns are independent, so one call on six 128 x 128 tiles must equal four
  calls on its quadrants, which take another form, bit for bit; and the value
  of the tangent-linear call, which runs one thread per column, must be that of
  the spread form at the edges of its layer counts.
* The Riemann solvers: one thread per column and both level counts a thread
  holds must return the same bits, on one call and on calls of its parts.
"""
import ctypes

import numpy as np
import pytest
import torch

from fv3core_amd import _lib
from fv3core_amd.stencils.map_single import MapSingle
from fv3core_amd.utils import gt4py_utils as utils
from fv3core_amd.utils.grid import to_storage
from fv3core_amd.utils.stencil import GridIndexing, StencilConfig, StencilFactory
from fv3core_amd.workloads import remap_inputs, transport_inputs

pytestmark = pytest.mark.gpu


def _like(x):
    y = utils.empty(tuple(x.shape), batch_dims=x.dim() - 3 if x.dim() > 3 else 0)
    y.copy_(x)
    return y


@pytest.mark.parametrize("hord", [5, 6, 7, 8])
@pytest.mark.parametrize("edges", [(True, True, True, True), (True, False, True, False)])
def test_corner_fill_transport_equals_copy_then_transport(hord, edges):
    n, nz = 24, 8
    d = transport_inputs(n, nz, workload=5)
    gi = GridIndexing((n, n, nz), 3, *edges)
    dev = {k: to_storage(v) for k, v in d.items()}
    q_a, q_b = _like(dev["q"]), _like(dev["q"])
    qy, scratch = torch.zeros_like(q_a), torch.zeros_like(q_a)
    fx_a, fy_a = torch.zeros_like(q_a), torch.zeros_like(q_a)
    fx_b, fy_b = torch.zeros_like(q_a), torch.zeros_like(q_a)
    aux = (dev["crx"], dev["cry"], dev["x_area_flux"], dev["y_area_flux"])
    dd = _lib.make_domain(gi, q_a, nz + 1, dev["area"],
                          others3=(q_b, qy, scratch, fx_a, fy_a, fx_b, fy_b) + aux)
    lib = _lib.lib()
    s = ctypes.c_void_p(_lib.stream_handle())
    metr = (_lib.ptr(dev["area"]), _lib.ptr(dev["dxa"]), _lib.ptr(dev["dya"]))
    _lib.check(lib.fv3_copy_corners_xy_f64(ctypes.byref(dd), _lib.ptr(q_a), _lib.ptr(q_a),
                                           _lib.ptr(qy), s))
    _lib.check(lib.fv3_fvtp2d_f64(ctypes.byref(dd), hord, _lib.ptr(q_a), _lib.ptr(qy),
                                  *[_lib.ptr(a) for a in aux], None, None, *metr,
                                  _lib.ptr(fx_a), _lib.ptr(fy_a), s))
    _lib.check(lib.fv3_fvtp2d_corner_fill_f64(ctypes.byref(dd), hord, _lib.ptr(q_b),
                                              _lib.ptr(scratch), *[_lib.ptr(a) for a in aux],
                                              None, None, *metr, _lib.ptr(fx_b),
                                              _lib.ptr(fy_b), s))
    torch.cuda.synchronize()
    assert torch.equal(q_a, q_b), "the x corner fill of q differs"
    assert torch.equal(fx_a, fx_b) and torch.equal(fy_a, fy_b), "fluxes differ"
    assert float(fx_b.abs().max()) > 0.0


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("hord", [6, 8])
def test_fvtp2d_tall_segments_equal_regular_segments(dtype, hord):
    n, nz, nt, chunk = 48, 79, 64, 8
    gi = GridIndexing((n, n, nz), 3, True, True, True, True)
    g = torch.Generator(device="cuda").manual_seed(4800 + hord)
    shape = (nt, n + 7, n + 7, nz + 1)

    def rand(lo, hi, shp=shape):
        t = utils.empty(shp, dtype=dtype, batch_dims=1)
        t.copy_(lo + (hi - lo) * torch.rand(shp, generator=g, device="cuda", dtype=torch.float64))
        return t

    q = rand(0.0, 1.0)
    crx, cry = rand(-0.45, 0.45), rand(-0.45, 0.45)
    xfx, yfx = rand(-2e9, 2e9), rand(-2e9, 2e9)
    area = rand(4e10, 6e10, (nt, n + 7, n + 7))
    dxa, dya = rand(1.8e5, 2.2e5, (nt, n + 7, n + 7)), rand(1.8e5, 2.2e5, (nt, n + 7, n + 7))
    name = "fv3_fvtp2d_f64" if dtype == torch.float64 else "fv3_fvtp2d_f32"
    fn = getattr(_lib.lib(), name)
    s = ctypes.c_void_p(_lib.stream_handle())

    def run(sl):
        fx, fy = torch.zeros_like(q[sl]), torch.zeros_like(q[sl])
        f3 = (q[sl], crx[sl], cry[sl], xfx[sl], yfx[sl], fx, fy)
        dd = _lib.make_domain(gi, q[sl], nz, area[sl], others3=f3,
                              others2=(dxa[sl], dya[sl]))
        _lib.check(fn(ctypes.byref(dd), hord, _lib.ptr(q[sl]), _lib.ptr(q[sl]),
                      _lib.ptr(crx[sl]), _lib.ptr(cry[sl]), _lib.ptr(xfx[sl]), _lib.ptr(yfx[sl]),
                      None, None, _lib.ptr(area[sl]), _lib.ptr(dxa[sl]), _lib.ptr(dya[sl]),
                      _lib.ptr(fx), _lib.ptr(fy), s))
        return fx, fy

    # the heights of the one call and of a part's, 49 rows of one strip a level
    rows = [_lib.lib().fv3_plan_fvtp2d_rows(n + 1, ctypes.c_int64(t * nz),
                                            int(dtype == torch.float32)) for t in (nt, chunk)]
    assert rows[0] != rows[1], rows
    fx_all, fy_all = run(slice(0, nt))
    for c in range(0, nt, chunk):
        fx_c, fy_c = run(slice(c, c + chunk))
        assert torch.equal(fx_all[c:c + chunk], fx_c), f"x fluxes of tiles {c}..{c + chunk - 1}"
        assert torch.equal(fy_all[c:c + chunk], fy_c), f"y fluxes of tiles {c}..{c + chunk - 1}"
    assert float(fx_all.abs().max()) > 0.0


SWEEPS, FUSED, LAYERS = 0, 1, 2


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("nz,whole_form,part_form", [(10, SWEEPS, LAYERS), (81, FUSED, LAYERS),
                                                     (137, FUSED, SWEEPS)])
@pytest.mark.parametrize("kord,mode", [(9, 1), (10, 0), (10, -2), (9, -1)])
def test_map_single_forms_equal(kord, mode, nz, whole_form, part_form, dtype):
    n, nt, h = 128, 6, 64
    gi = GridIndexing((n, n, nz), 3, True, True, True, True)
    factory = StencilFactory(StencilConfig(), gi)

    def plan(columns):
        waves = (columns + 63) // 64 * nt
        return _lib.lib().fv3_plan_map_single(nz, ctypes.c_int64(waves),
                                              int(dtype == torch.float32))

    assert (plan(n * n), plan(h * h)) == (whole_form, part_form)
    g = torch.Generator(device="cuda").manual_seed(nz)
    shape = (nt,) + gi.max_shape

    def field(t):
        b = utils.empty(shape, dtype=dtype, batch_dims=1)
        b.copy_(t)
        return b

    def interfaces():
        dp = 500.0 + 1000.0 * torch.rand(shape, generator=g, device="cuda", dtype=torch.float64)
        return field(100.0 + 1e5 * dp.cumsum(-1) / dp.sum(-1, keepdim=True))

    pe1, pe2 = interfaces(), interfaces()
    pe2[..., 0], pe2[..., nz] = pe1[..., 0], pe1[..., nz]
    src = field(torch.rand(shape, generator=g, device="cuda", dtype=torch.float64))
    qs = field(torch.rand(shape, generator=g, device="cuda"))[..., 0] if mode == -2 else None
    whole, parts = _like(src).to(dtype), _like(src).to(dtype)
    MapSingle(factory, kord, mode, gi.isc, gi.iec, gi.jsc, gi.jec)(whole, pe1, pe2, qs=qs)
    for i1 in (gi.isc, gi.isc + h):
        for j1 in (gi.jsc, gi.jsc + h):
            MapSingle(factory, kord, mode, i1, i1 + h - 1, j1, j1 + h - 1)(parts, pe1, pe2,
                                                                        qs=qs)
    torch.cuda.synchronize()
    assert torch.equal(whole, parts)
    assert not torch.equal(whole, src)


@pytest.mark.parametrize("nz", [79, 80, 81, 127, 128])
@pytest.mark.parametrize("mode", [-2, -1, 0, 1, 2])
def test_map_single_spread_layers_equal_the_tangent_linear_value(mode, nz, monkeypatch):
    from fv3core_amd import workloads
    from fv3core_amd.adjoint import RemapLinearization

    monkeypatch.setattr(workloads, "hybrid_coefficients", workloads.synthetic_hybrid)
    n = 7
    d = remap_inputs(n, nz, workload=91)
    gi = GridIndexing((n, n, nz), 3, True, True, True, True)
    box = (gi.isc, gi.iec, gi.jsc, gi.jec)
    assert _lib.lib().fv3_plan_map_single(nz, ctypes.c_int64(1), 0) == LAYERS
    src = to_storage(d["q"] if mode == 0 else d["w"] if mode in (-2, -1) else d["pt"])
    pe1, pe2 = to_storage(d["pe1"]), to_storage(d["pe2"])
    qs = to_storage(d["qs"]) if mode == -2 else None
    spread = _like(src)
    MapSingle(StencilFactory(StencilConfig(), gi), 9, mode, *box)(spread, pe1, pe2, qs=qs)
    value, _ = RemapLinearization(gi, mode).tlm(src, _like(src), pe1, pe2, qs)
    torch.cuda.synchronize()
    assert torch.equal(spread[..., :nz], value[..., :nz])
    assert not torch.equal(spread, src)


COLUMN = 0  # the other forms of the Riemann solvers go by the levels a thread holds


# Every pair of forms: few layers, 16 layers (one wave of 8 levels a thread), a
# full round of columns, above the reach of 5 levels a thread.
@pytest.mark.parametrize("solver_c,nz,tiles,whole_form,part_form", [
    (True, 4, 8, COLUMN, 5), (True, 16, 16, 8, 5), (True, 50, 56, COLUMN, 5),
    (True, 90, 40, COLUMN, 8), (False, 4, 8, COLUMN, 5), (False, 16, 16, 8, 5),
    (False, 64, 16, 8, 5), (False, 90, 40, COLUMN, 8)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_riemann_forms_equal(solver_c, nz, tiles, whole_form, part_form, dtype, monkeypatch):
    from fv3core_amd import workloads
    from fv3core_amd._config import RiemannConfig
    from fv3core_amd.stencils.riem_solver3 import RiemannSolver3
    from fv3core_amd.stencils.riem_solver_c import RiemannSolverC

    monkeypatch.setattr(workloads, "hybrid_coefficients", workloads.synthetic_hybrid)
    n = 30 if solver_c else 32  # 1024 columns a tile
    for waves, form in ((16 * tiles, whole_form), (16, part_form)):
        assert _lib.lib().fv3_plan_riem(nz, ctypes.c_int64(waves), int(solver_c),
                                        int(dtype == torch.float32)) == form
    r = workloads.riemann_inputs(n, nz, workload=7)
    gi = GridIndexing((n, n, nz), 3, True, True, True, True)
    factory = StencilFactory(StencilConfig(), gi)
    bulk = ("cappa", "pt", "q_con", "delp", "w")

    def batch(name):
        a = torch.as_tensor(np.ascontiguousarray(r[name]), device="cuda")
        b = utils.empty((tiles,) + tuple(a.shape), batch_dims=1,
                        dtype=dtype if name in bulk else torch.float64)
        b.copy_(a.expand(b.shape))
        if name == "pt":  # tiles that differ
            b.mul_(1.0 + 1e-3 * torch.arange(tiles, device="cuda").view(-1, 1, 1, 1))
        return b

    out = []
    for parts in (False, True):
        t = {k: batch(k) for k in bulk + ("gz", "zh", "delz", "pe", "hs", "ws", "zs")}
        o = [batch("pe").zero_() for _ in range(4)]
        for sl in ([slice(k, k + 1) for k in range(tiles)] if parts else [slice(0, tiles)]):
            f = {k: v[sl] for k, v in t.items()}
            p = [v[sl] for v in o]
            if solver_c:
                RiemannSolverC(factory, 0.05)(18.75, f["cappa"], r["ptop"], f["hs"], f["ws"],
                                              f["pt"], f["q_con"], f["delp"], f["gz"], p[0],
                                              f["w"])
            else:
                RiemannSolver3(factory, RiemannConfig(p_fac=0.05, a_imp=1.0, use_logp=False,
                                                      beta=0.0))(
                    True, 37.5, f["cappa"], r["ptop"], f["zs"], f["ws"], f["delz"], f["q_con"],
                    f["delp"], f["pt"], f["zh"], f["pe"], *p, f["w"])
        out.append(list(t.values()) + o)
    torch.cuda.synchronize()
    for a, b in zip(*out):
        assert torch.equal(a, b)
    changed = out[0][5 if solver_c else 6]
    assert not torch.equal(changed, batch("gz" if solver_c else "zh"))
    assert bool(torch.isfinite(changed).all())
