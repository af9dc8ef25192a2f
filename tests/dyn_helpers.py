"""Inputs shared by the acoustic-step tests: smooth seeded fields on one
periodic plane tile or on the six tiles of the cube, and device copies."""
import numpy as np
import torch

from fv3core_amd import cube
from fv3core_amd.utils import gt4py_utils as utils
from fv3core_amd.utils.grid import GridData
from fv3core_amd.utils.stencil import GridIndexing, StencilConfig, StencilFactory
from fv3core_amd.workloads import fill_periodic, plane_metric
from oracle.fvtp2d import Tile


def smooth(rng, shape, mean, amp, modes=(1, 2, 3)):
    """Sum of random-phase sinusoids over the (i, j, k) index space."""
    ni, nj, nk = shape[-3:]
    x = np.arange(ni)[:, None, None] / ni
    y = np.arange(nj)[None, :, None] / nj
    z = np.arange(nk)[None, None, :] / max(nk, 1)
    f = np.zeros((ni, nj, nk))
    for m in modes:
        a = rng.uniform(0.3, 1.0) / m
        p = rng.uniform(0, 2 * np.pi, size=3)
        f += a * np.sin(2 * np.pi * m * x + p[0]) * np.cos(2 * np.pi * m * y + p[1]) * \
            np.cos(np.pi * z + p[2])
    return mean + amp * f / np.abs(f).max()


class Case:
    """A single periodic plane tile (edges off) or the six cube tiles (edges on:
    all of them, or those of a tuple of south, north, west and east)."""

    def __init__(self, n, nz, cube_tiles, seed=0, f=1.0e-4):
        self.n, self.nz, self.cube = n, nz, cube_tiles
        self.ntiles = 6 if cube_tiles else 1
        self.rng = np.random.default_rng(seed)
        edges = cube_tiles if isinstance(cube_tiles, tuple) else (bool(cube_tiles),) * 4
        self.tile = Tile(n, n, 3, *edges)
        self.gi = GridIndexing((n, n, nz), 3, *edges)
        self.factory = StencilFactory(StencilConfig(), self.gi)
        if cube_tiles:
            m = cube.tile_metrics(n)
            self.metric = [{k: v[t] for k, v in m.items() if isinstance(v, np.ndarray)}
                           for t in range(6)]
        else:
            m = plane_metric(n, f=f)
            self.metric = [{k: v for k, v in m.items() if isinstance(v, np.ndarray)}]
        # scalar terms (da_min, da_min_c ...), the same for every tile
        self.scalars = {k: float(v) for k, v in m.items() if not isinstance(v, np.ndarray)}
        self.shape = (n + 7, n + 7, nz + 1)

    def field(self, mean, amp):
        out = []
        for _ in range(self.ntiles):
            a = smooth(self.rng, self.shape, mean, amp)
            if not self.cube:
                a = fill_periodic(a, self.n)
            out.append(a)
        return out

    def dev(self, arrs):
        """Device storage of one field: (I, J, K) for one tile, (6, I, J, K) for six."""
        if self.ntiles == 1:
            t = utils.empty(arrs[0].shape)
            t.copy_(torch.as_tensor(arrs[0]))
            return t
        t = utils.empty((6,) + arrs[0].shape)
        t.copy_(torch.as_tensor(np.stack(arrs)))
        return t

    def host(self, t):
        a = t.detach().cpu().numpy()
        return [a] if self.ntiles == 1 else [a[i] for i in range(6)]

    def grid_data(self, names=None):
        fields = {}
        keys = names or self.metric[0].keys()
        for k in keys:
            if self.ntiles == 1:
                t = utils.empty(self.metric[0][k].shape)
                t.copy_(torch.as_tensor(self.metric[0][k]))
            else:
                t = utils.empty((6,) + self.metric[0][k].shape, batch_dims=1)
                t.copy_(torch.as_tensor(np.stack([m[k] for m in self.metric])))
            fields[k] = t
        return GridData(fields)


def to_fp32(case, fields):
    """fields, and the case's metric terms, with every value rounded to FP32."""
    r = lambda a: a.astype(np.float32).astype(np.float64)  # noqa: E731
    case.metric = [{k: r(v) for k, v in m.items()} for m in case.metric]
    return {k: [r(a) for a in v] for k, v in fields.items()}


def oracle_acoustic_call(init, cfg, n, nz, pfull):
    """The oracle's AcousticDynamics call on the six tiles of one cube state
    (what workloads.cube_state returns), with the host restatement of the
    halo map between its components; returns the updated state dict."""
    from fv3core_amd.halo import CENTER, CORNER, X_FACE, Y_FACE, apply_map_numpy, build_map, \
        build_sync_map
    from fv3core_amd.stencils.d_sw import get_column_namelist
    from oracle import dyncore as odc

    st0, m = init["state"], init["metric"]
    S = {k: v.copy() for k, v in st0.items()}
    S["phis"] = init["phis"].copy()
    S["wsd"] = init["wsd"].copy()
    S["ws3"] = np.zeros_like(init["wsd"])
    shape = st0["delp"].shape
    for k in ("ut", "vt", "gz", "pem", "pkc", "pk3", "heat_source", "divgd", "crx", "xfx",
              "cry", "yfx", "delpc", "ptc"):
        S[k] = np.zeros(shape)
    S["gz"][:] = 1.0e40
    S["pk3"][:] = 1.0e40
    maps = {}

    def halo(kind, names, n_halo=3):
        key = (kind, n_halo)
        if key not in maps:
            stg = {"scalar": (CENTER,), "vector_d": (Y_FACE, X_FACE),
                   "vector_c": (X_FACE, Y_FACE), "corner": (CORNER,)}[kind]
            maps[key] = build_map(n, stg, n_halo, 3)
        mp = maps[key]
        if kind.startswith("vector"):
            for a in range(0, len(names), 2):
                u, v = apply_map_numpy([S[names[a]], S[names[a + 1]]], mp)
                S[names[a]][...] = u
                S[names[a + 1]][...] = v
        else:
            for name in names:
                S[name][...] = apply_map_numpy([S[name]], mp)[0]

    def sync():
        mp = build_sync_map(n, 3)
        u, v = apply_map_numpy([S["u"], S["v"]], mp)
        S["u"][...] = u
        S["v"][...] = v

    col = get_column_namelist(cfg.d_grid_shallow_water, nz)
    ocfg = dict(mdt=float(cfg.dt_atmos), n_split=cfg.n_split, k_split=cfg.k_split, n_map=1,
                ptop=init["ptop"], hord_dp=cfg.hord_dp, hord_tm=cfg.hord_tm,
                hord_mt=cfg.hord_mt, hord_vt=cfg.hord_vt, dddmp=cfg.dddmp, d4_bg=cfg.d4_bg,
                nord=cfg.nord, d_con=cfg.d_con, convert_ke=cfg.convert_ke, vtdm4=cfg.vtdm4,
                p_fac=cfg.p_fac, rf_cutoff=cfg.rf_cutoff, tau=cfg.tau, delt_max=cfg.delt_max)
    metrics = [{k: v[t] for k, v in m.items() if isinstance(v, np.ndarray) and v.ndim == 3}
               for t in range(6)]
    odc.acoustic_dynamics(S, ocfg, metrics, dict(da_min=m["da_min"], da_min_c=m["da_min_c"]),
                          init["ak"], init["bk"], pfull, halo, sync, col, nz)
    return S
