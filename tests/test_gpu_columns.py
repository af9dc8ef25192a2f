"""GPU parity of the column kernels (remap, Riemann solvers) against the oracle."""
import numpy as np
import pytest
import torch

from fv3core_amd._config import RiemannConfig
from fv3core_amd.stencils.map_single import MapSingle
from fv3core_amd.stencils.riem_solver3 import RiemannSolver3
from fv3core_amd.stencils.riem_solver_c import RiemannSolverC
from fv3core_amd.utils import gt4py_utils as utils
from fv3core_amd.utils.grid import to_storage
from fv3core_amd.utils.stencil import GridIndexing, StencilConfig, StencilFactory
from fv3core_amd.workloads import remap_inputs, riemann_inputs
from oracle import remap as orm
from oracle import riemann as ori
from tests.helpers import assert_close, to_np

pytestmark = pytest.mark.gpu

NZ = 79


def _factory(n, nz=NZ):
    gi = GridIndexing((n, n, nz), 3, True, True, True, True)
    return StencilFactory(StencilConfig(), gi), gi


@pytest.mark.parametrize("kord,mode", [(9, 1), (10, 1), (10, 0), (9, -1), (10, -2), (9, 2),
                                       (5, 1), (-10, 1)])
def test_map_single_parity(kord, mode):
    n = 12
    d = remap_inputs(n, NZ, workload=51)
    factory, gi = _factory(n)
    i1, i2, j1, j2 = gi.isc, gi.iec, gi.jsc, gi.jec
    src = d["q"] if mode == 0 else (d["w"] if mode in (-2, -1) else d["pt"])
    ms = MapSingle(factory, kord, mode, i1, i2, j1, j2)
    q1 = to_storage(src)
    qs = to_storage(d["qs"]) if mode == -2 else None
    ms(q1, to_storage(d["pe1"]), to_storage(d["pe2"]), qs=qs, qmin=0.0)
    torch.cuda.synchronize()
    ref = orm.map_single(src, d["pe1"], d["pe2"], kord, mode, i1, i2, j1, j2,
                         qs=d["qs"] if mode == -2 else None)
    assert_close(to_np(q1)[..., :NZ], ref[..., :NZ], 1e-12, near_zero=1e-18, what="q1")


def test_map_single_batched_and_qmin():
    n, nt = 10, 3
    factory, gi = _factory(n)
    ins = [remap_inputs(n, NZ, workload=60 + t) for t in range(nt)]
    shape = gi.max_shape

    def batch(name):
        b = utils.empty((nt,) + shape)
        for t in range(nt):
            b[t].copy_(torch.as_tensor(ins[t][name]))
        return b

    q1, pe1, pe2 = batch("pt"), batch("pe1"), batch("pe2")
    ms = MapSingle(factory, 9, 1, gi.isc, gi.iec, gi.jsc, gi.jec)
    ms(q1, pe1, pe2, qmin=221.0)
    torch.cuda.synchronize()
    for t in range(nt):
        ref = orm.map_single(ins[t]["pt"], ins[t]["pe1"], ins[t]["pe2"], 9, 1, gi.isc, gi.iec,
                             gi.jsc, gi.jec, qmin=221.0)
        assert_close(to_np(q1[t])[..., :NZ], ref[..., :NZ], 1e-12, what=f"tile {t}")


@pytest.mark.parametrize("seed", [0, 1])
def test_riem_solver_c_parity(seed):
    n = 12
    r = riemann_inputs(n, NZ, workload=70 + seed)
    factory, gi = _factory(n)
    rs = RiemannSolverC(factory, 0.05)
    dev = {k: to_storage(v) for k, v in r.items() if isinstance(v, np.ndarray) and v.ndim >= 2}
    gz = dev["gz"].clone()
    pef = utils.zeros(gi.max_shape)
    rs(r["dt"] / 2, dev["cappa"], r["ptop"], dev["hs"], dev["ws"], dev["pt"], dev["q_con"],
       dev["delp"], gz, pef, dev["w"])
    torch.cuda.synchronize()
    sl = (slice(gi.isc - 1, gi.iec + 2), slice(gi.jsc - 1, gi.jec + 2))
    rgz, rpef = ori.riem_solver_c(r["dt"] / 2, r["cappa"][sl], r["ptop"], r["hs"][sl],
                                  r["ws"][sl], r["pt"][sl], r["q_con"][sl], r["delp"][sl],
                                  r["gz"][sl], r["w"][sl], 0.05)
    assert_close(to_np(gz)[sl], rgz, 1e-12, what="gz")
    assert_close(to_np(pef)[sl], rpef, 1e-12, what="pef")


@pytest.mark.parametrize("last_call,use_logp,beta", [(True, False, 0.0), (False, False, 0.0),
                                                     (True, True, -0.2)])
def test_riem_solver3_parity(last_call, use_logp, beta):
    n = 12
    r = riemann_inputs(n, NZ, workload=80)
    factory, gi = _factory(n)
    cfg = RiemannConfig(p_fac=0.05, a_imp=1.0, use_logp=use_logp, beta=beta)
    rs = RiemannSolver3(factory, cfg)
    rng = np.random.default_rng(3)
    pk3_0 = rng.uniform(size=r["pe"].shape)
    pk_0 = rng.uniform(size=r["pe"].shape)
    peln_0 = rng.uniform(size=r["pe"].shape)
    ppe_0 = np.zeros(r["pe"].shape)
    t = {k: to_storage(v) for k, v in r.items() if isinstance(v, np.ndarray) and v.ndim >= 2}
    delz, zh, pe, w = t["delz"].clone(), t["zh"].clone(), t["pe"].clone(), t["w"].clone()
    ppe, pk3, pk, peln = (to_storage(a) for a in (ppe_0, pk3_0, pk_0, peln_0))
    wsd = to_storage(np.full(r["zs"].shape, 0.01))
    rs(last_call, r["dt"], t["cappa"], r["ptop"], t["zs"], wsd, delz, t["q_con"], t["delp"],
       t["pt"], zh, pe, ppe, pk3, pk, peln, w)
    torch.cuda.synchronize()
    sl = (slice(gi.isc, gi.iec + 1), slice(gi.jsc, gi.jec + 1))
    ref = ori.riem_solver3(last_call, r["dt"], r["cappa"][sl], r["ptop"], r["zs"][sl],
                           np.full(r["zs"].shape, 0.01)[sl], r["delz"][sl], r["q_con"][sl],
                           r["delp"][sl], r["pt"][sl], r["zh"][sl], r["pe"][sl], ppe_0[sl],
                           pk3_0[sl], pk_0[sl], peln_0[sl], r["w"][sl], 0.05, use_logp=use_logp,
                           beta=beta)
    names = ["zh", "pe", "ppe", "pk3", "pk", "peln", "w", "delz"]
    got = [zh, pe, ppe, pk3, pk, peln, w, delz]
    # ppe and w come out of small differences (w - w1 summed into ppe): their
    # error is measured against the field's largest magnitude, so that
    # last-bit exp/log differences amplified by the cancellation do not count
    floors = {"ppe": 0.5, "w": 0.5}
    for name, g, rr in zip(names, got, ref):
        assert_close(to_np(g)[sl], rr, 1e-12, near_zero=1e-12, what=name,
                     scale_floor=floors.get(name, 0.0))


class _OneUlp:
    """numpy with every exp and log result moved by one ulp, up or down."""

    def __init__(self, seed):
        self._rng = np.random.default_rng(seed)

    def __getattr__(self, name):
        return getattr(np, name)

    def _moved(self, a):
        return np.nextafter(a, self._rng.choice([-np.inf, np.inf], size=np.shape(a)))

    def exp(self, a):
        return self._moved(np.exp(a))

    def log(self, a):
        return self._moved(np.log(a))


# Columns of 3 layers up to the most a workgroup holds: one thread's levels,
# one more than whole sets, the last layer alone in its set, and both sides
# of the change from 5 to 8 levels a thread (80 / 81).
@pytest.mark.parametrize("nz", [3, 5, 6, 10, 11, 41, 80, 81, 127])
@pytest.mark.parametrize("n", [5, 9])
def test_riem_solvers_level_counts(nz, n, monkeypatch):
    from fv3core_amd import workloads

    monkeypatch.setattr(workloads, "hybrid_coefficients", workloads.synthetic_hybrid)
    r = riemann_inputs(n, nz, workload=90 + nz)
    factory, gi = _factory(n, nz)
    t = {k: to_storage(v) for k, v in r.items() if isinstance(v, np.ndarray) and v.ndim >= 2}
    gz, pef = t["gz"].clone(), utils.zeros(gi.max_shape)
    RiemannSolverC(factory, 0.05)(r["dt"] / 2, t["cappa"], r["ptop"], t["hs"], t["ws"], t["pt"],
                                  t["q_con"], t["delp"], gz, pef, t["w"])
    wsd = np.full(r["zs"].shape, 0.01)
    delz, zh, pe, w = (t[k].clone() for k in ("delz", "zh", "pe", "w"))
    ppe, pk3, pk, peln = (utils.zeros(gi.max_shape) for _ in range(4))
    RiemannSolver3(factory, RiemannConfig(p_fac=0.05, a_imp=1.0, use_logp=False, beta=0.0))(
        True, r["dt"], t["cappa"], r["ptop"], t["zs"], to_storage(wsd), delz, t["q_con"],
        t["delp"], t["pt"], zh, pe, ppe, pk3, pk, peln, w)
    torch.cuda.synchronize()
    sl = (slice(gi.isc - 1, gi.iec + 2), slice(gi.jsc - 1, gi.jec + 2))
    rgz, rpef = ori.riem_solver_c(r["dt"] / 2, r["cappa"][sl], r["ptop"], r["hs"][sl],
                                  r["ws"][sl], r["pt"][sl], r["q_con"][sl], r["delp"][sl],
                                  r["gz"][sl], r["w"][sl], 0.05)
    assert_close(to_np(gz)[sl], rgz, 1e-12, what="gz")
    assert_close(to_np(pef)[sl], rpef, 1e-12, what="pef")
    sl = (slice(gi.isc, gi.iec + 1), slice(gi.jsc, gi.jec + 1))
    z = np.zeros(r["pe"].shape)

    def oracle():
        return ori.riem_solver3(True, r["dt"], r["cappa"][sl], r["ptop"], r["zs"][sl], wsd[sl],
                                r["delz"][sl], r["q_con"][sl], r["delp"][sl], r["pt"][sl],
                                r["zh"][sl], r["pe"][sl], z[sl], z[sl], z[sl], z[sl],
                                r["w"][sl], 0.05)

    ref = oracle()
    monkeypatch.setattr(ori, "np", _OneUlp(nz))
    moved = oracle()
    for name, g, rr, mm in zip(["zh", "pe", "ppe", "pk3", "pk", "peln", "w", "delz"],
                               [zh, pe, ppe, pk3, pk, peln, w, delz], ref, moved):
        # ppe and w come out of cancelling terms: they are measured against
        # the field's scale, within four times what a last-bit difference in
        # exp and log does there (log enters pm as the difference of
        # neighbouring levels' logs)
        tol, floor = 1e-12, 0.0
        if name in ("ppe", "w"):
            floor = 0.5
            tol = max(tol, 4.0 * np.abs(mm - rr).max() / (0.5 * np.abs(rr).max()))
        assert_close(to_np(g)[sl], rr, tol, near_zero=1e-12, what=name, scale_floor=floor)
    # outside its box a solver writes nothing
    for got, was in ((zh, r["zh"]), (delz, r["delz"]), (w, r["w"])):
        a = to_np(got)
        a[sl] = was[sl]
        assert np.array_equal(a, was)


# Layer counts with and without layers past the bottom in the last set of 5 or 8.
@pytest.mark.parametrize("nz", [3, 5, 10, 12, 79, 81, 127])
def test_riem_solver3_infinite_wind_in_the_lowest_layer(nz, monkeypatch):
    """An infinite w in the lowest layer, under a layer hot enough for its
    change of w to be infinite and not NaN: pe is -inf there, the pressure
    limit p_fac takes over and the layer keeps a finite height, as in the oracle."""
    from fv3core_amd import workloads

    monkeypatch.setattr(workloads, "hybrid_coefficients", workloads.synthetic_hybrid)
    r = riemann_inputs(5, nz, workload=1)
    factory, gi = _factory(5, nz)
    c = gi.isc
    for j, wind in ((c, np.inf), (c + 1, -np.inf)):
        r["w"][c + 1, j, nz - 1] = wind
        r["pt"][c + 1, j, nz - 2] = 3e38
    t = {k: to_storage(v) for k, v in r.items() if isinstance(v, np.ndarray) and v.ndim >= 2}
    wsd = np.full(r["zs"].shape, 0.01)
    ppe, pk3, pk, peln = (utils.zeros(gi.max_shape) for _ in range(4))
    RiemannSolver3(factory, RiemannConfig(p_fac=0.05, a_imp=1.0, use_logp=False, beta=0.0))(
        True, r["dt"], t["cappa"], r["ptop"], t["zs"], to_storage(wsd), t["delz"], t["q_con"],
        t["delp"], t["pt"], t["zh"], t["pe"], ppe, pk3, pk, peln, t["w"])
    torch.cuda.synchronize()
    sl = (slice(gi.isc, gi.iec + 1), slice(gi.jsc, gi.jec + 1))
    z = np.zeros(r["pe"].shape)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = ori.riem_solver3(True, r["dt"], r["cappa"][sl], r["ptop"], r["zs"][sl], wsd[sl],
                               r["delz"][sl], r["q_con"][sl], r["delp"][sl], r["pt"][sl],
                               r["zh"][sl], r["pe"][sl], z[sl], z[sl], z[sl], z[sl],
                               r["w"][sl], 0.05)
    assert np.isfinite(ref[7][1, 0, nz - 1]) and not np.isfinite(ref[7][1, 0, 0])
    for name, got, want in zip(["zh", "pe", "ppe", "pk3", "pk", "peln", "w", "delz"],
                               [t["zh"], t["pe"], ppe, pk3, pk, peln, t["w"], t["delz"]], ref):
        g = to_np(got)[sl]
        np.testing.assert_array_equal(np.isfinite(g), np.isfinite(want), err_msg=name)
        if name in ("zh", "delz"):
            fin = np.isfinite(want)
            assert_close(np.where(fin, g, 0.0), np.where(fin, want, 0.0), 1e-11, near_zero=1e-12,
                         what=name)


# 10^e m: where the factor of w's lowest layer overflows while the terms it sums
# and every output stay finite.
@pytest.mark.parametrize("nz,e", [(6, -299.05), (12, -299.45), (41, -300.15), (79, -300.55),
                                  (127, -300.82)])
def test_riem_solver3_overflowing_divisor(nz, e, monkeypatch):
    """A quotient by an infinite divisor is 0, as IEEE division has it: three
    layers so thin that the lowest one's divisor overflows leave a finite
    column, as in the oracle."""
    from fv3core_amd import workloads

    monkeypatch.setattr(workloads, "hybrid_coefficients", workloads.synthetic_hybrid)
    r = riemann_inputs(5, nz, workload=1)
    factory, gi = _factory(5, nz)
    sl = (slice(gi.isc, gi.iec + 1), slice(gi.jsc, gi.jec + 1))
    for l, height in enumerate((2.0, 3.0, 4.0)):
        r["zh"][..., nz - 1 - l] = height * 10.0 ** e
        r["pt"][..., nz - 1 - l] = 0.02 * (r["zh"][..., nz - 1 - l] - r["zh"][..., nz - l])
    t = {k: to_storage(v) for k, v in r.items() if isinstance(v, np.ndarray) and v.ndim >= 2}
    wsd = np.full(r["zs"].shape, 0.01)
    ppe, pk3, pk, peln = (utils.zeros(gi.max_shape) for _ in range(4))
    RiemannSolver3(factory, RiemannConfig(p_fac=0.05, a_imp=1.0, use_logp=False, beta=0.0))(
        True, r["dt"], t["cappa"], r["ptop"], t["zs"], to_storage(wsd), t["delz"], t["q_con"],
        t["delp"], t["pt"], t["zh"], t["pe"], ppe, pk3, pk, peln, t["w"])
    torch.cuda.synchronize()
    z = np.zeros(r["pe"].shape)
    with np.errstate(over="ignore"):
        ref = ori.riem_solver3(True, r["dt"], r["cappa"][sl], r["ptop"], r["zs"][sl], wsd[sl],
                               r["delz"][sl], r["q_con"][sl], r["delp"][sl], r["pt"][sl],
                               r["zh"][sl], r["pe"][sl], z[sl], z[sl], z[sl], z[sl],
                               r["w"][sl], 0.05)
    for name, got, want in zip(["zh", "pe", "ppe", "pk3", "pk", "peln", "w", "delz"],
                               [t["zh"], t["pe"], ppe, pk3, pk, peln, t["w"], t["delz"]], ref):
        g = to_np(got)[sl]
        assert np.isfinite(want).all() and np.isfinite(g).all(), name
        assert_close(g, want, 1e-9, what=name, scale_floor=1.0)


def test_riem_solver_c_wide_offsets():
    """Storages whose levels lie more than 4 GiB apart: 64-bit offsets, the
    same results as on dense storages."""
    n, nz = 5, 3
    ni, nk = n + 7, nz + 1
    factory, gi = _factory(n, nz)
    rng = np.random.default_rng(5)
    dp = rng.uniform(2.0e4, 3.0e4, size=(ni, ni, nk))
    ins = dict(cappa=np.full(dp.shape, 0.2857), pt=rng.uniform(5.0, 12.0, size=dp.shape),
               q_con=np.zeros(dp.shape), delp=dp, w=rng.normal(size=dp.shape),
               gz=np.cumsum(rng.uniform(2e3, 3e3, size=dp.shape)[..., ::-1], axis=2)[..., ::-1])
    zero = to_storage(np.zeros((ni, ni)))
    out = []
    for wide in (False, True):
        rows = -(-(1 << 27) // ni) + 1 if wide else ni  # (nk - 1) sk 8 B is past 4 GiB

        def store(a):
            t = torch.empty((nk, rows, ni), dtype=torch.float64, device="cuda")[:, :ni]
            t = t.permute(2, 1, 0)
            t.copy_(torch.as_tensor(np.ascontiguousarray(a)))
            return t

        f = {k: store(a) for k, a in ins.items()}
        pef = store(np.zeros(dp.shape))
        RiemannSolverC(factory, 0.05)(18.75, f["cappa"], 300.0, zero, zero, f["pt"], f["q_con"],
                                      f["delp"], f["gz"], pef, f["w"])
        out.append((to_np(f["gz"].clone()), to_np(pef.clone())))
        del f, pef
        torch.cuda.empty_cache()
    assert np.isfinite(out[0][0]).all()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


# Column heights at the edges of a set, a wave and a workgroup of each set size
# and past the kernel that spreads layers; a box that does not fill a workgroup.
@pytest.mark.parametrize("nz", [6, 7, 20, 21, 80, 81, 128, 129])
@pytest.mark.parametrize("kord,mode", [(9, 1), (10, 0), (10, -2), (8, -1), (9, 2)])
def test_map_single_layer_sets(nz, kord, mode):
    n = 5
    factory, gi = _factory(n, nz)
    box = (gi.isc, gi.iec, gi.jsc, gi.jec - 1)
    rng = np.random.default_rng(nz)
    shape = gi.max_shape[:2] + (nz + 1,)
    pe1 = 100.0 + np.cumsum(rng.uniform(500.0, 1500.0, shape), axis=2)
    pe2 = pe1.copy()
    # target interfaces up to two layers away, in order, ends in common
    pe2[..., 1:-1] = np.sort(pe1[..., 1:-1] + rng.uniform(-1500.0, 1500.0, shape)[..., 1:-1])
    pe2 = np.clip(pe2, pe1[..., :1] + np.arange(nz + 1), pe1[..., -1:] - np.arange(nz, -1, -1))
    src = rng.normal(0.0, 1.0, shape) + np.sin(0.4 * np.arange(nz + 1))
    if mode == 0:
        src = np.abs(src)
    qs = rng.normal(0.0, 1.0, shape[:2]) if mode == -2 else None
    q1 = to_storage(src)
    MapSingle(factory, kord, mode, *box)(q1, to_storage(pe1), to_storage(pe2),
                                         qs=None if qs is None else to_storage(qs))
    torch.cuda.synchronize()
    ref = orm.map_single(src, pe1, pe2, kord, mode, *box, qs=qs)
    # a target layer's integral is a difference of parabola terms of the
    # field's size over at least a thousandth of a layer, so values near zero
    # are compared on the field's scale
    err = np.abs(to_np(q1)[..., :nz] - ref[..., :nz]).max()
    assert err <= 1e-12 * np.abs(src).max(), err


def test_map_single_unordered_and_special_columns():
    """Columns whose target interfaces are out of order, and columns with an
    infinity, a NaN or zeros in the field: as the oracle's walk from the top."""
    n = 4
    d = remap_inputs(n, NZ, workload=53)
    factory, gi = _factory(n)
    src, pe1, pe2 = d["pt"].copy(), d["pe1"].copy(), d["pe2"].copy()
    c = gi.isc
    pe2[c, c, 30], pe2[c, c, 33] = pe2[c, c, 33], pe2[c, c, 30]
    pe2[c + 1, c, 5] = 0.5 * (pe1[c + 1, c, 40] + pe1[c + 1, c, 41])
    src[c + 2, c, 20] = np.inf
    src[c + 3, c, 50] = np.nan
    src[c, c + 1, :] = 0.0
    q1 = to_storage(src)
    box = (gi.isc, gi.iec, gi.jsc, gi.jec)
    MapSingle(factory, 9, 1, *box)(q1, to_storage(pe1), to_storage(pe2))
    torch.cuda.synchronize()
    with np.errstate(invalid="ignore"):
        ref = orm.map_single(src, pe1, pe2, 9, 1, *box)
    got = to_np(q1)[..., :NZ]
    finite = np.isfinite(ref[..., :NZ])
    assert (np.isfinite(got) == finite).all()
    assert_close(np.where(finite, got, 0.0), np.where(finite, ref[..., :NZ], 0.0), 1e-12,
                 what="q1")
