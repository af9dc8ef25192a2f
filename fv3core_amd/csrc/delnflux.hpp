// Del-n diffusive fluxes (DelnFlux / DelnFluxNoSG) with what uses them.
//
// Reference: fv3core/stencils/delnflux.py:901-1207 runs, per call, 5 + 5*nmax
// stencils (d2 preamble, x/y corner copies, fx/fy, and per extra order a
// divergence d2 plus corner copies and fluxes) on full-size temporaries.
// Here one wave marches up a strip of 64 columns of one level: every pass of
// a row follows its predecessor by one row, in registers, with lane shifts
// across i, no LDS and no barrier.  What the passes produce, the flux pair of
// an interface row and the four fluxes around each cell of the row below,
// goes to an epilogue that adds it to the caller's fluxes, or straight on to
// the stencil that would read them back.  Levels whose band has nord == 0
// take the del-2 flux alone, as the reference's regions do.
//
// The corner copies turn columns into rows at the cube corners, which a march
// cannot follow; the few interfaces they reach (two cells in each direction
// for up to two extra passes) are left to a window of 8 x 8 cells in LDS, one
// wave per corner and level, in the same launch.  Along a direction in which a
// tile is narrower than four cells, where the corners' reaches meet, one window
// spans it (at most 9 cells, halo included).
//
// What bounds it: the passes' memory traffic for large calls, the latency of a
// march step for small ones.  Measured in the acoustic call, FP64, against LDS
// blocks that ran every pass with barriers: six C96 tiles, 79 levels (added to
// the caller's fluxes) 84 -> 64 us.  With the readers as epilogues the d_sw call
// there loses five launches of 60 to 150 us and 14 passes over full-size
// fields; the acoustic call goes 26.3 -> 25.2 ms, and 6.0 -> 5.2 ms on six C12
// tiles.  Two rows per loop pass with the load buffers in turn and branch-free
// stores, as other marches here have, measured 2 to 9 % slower at C96 (more
// registers in flight, stores issued for rows without owned interfaces).
#pragma once

#include "strip.hpp"
#include "tile_config.hpp"
#include "timing.hpp"

namespace fv3 {

constexpr int DN_W = 64;            // lanes = strip columns
constexpr int DN_TI = DN_W - 6;     // interfaces per strip in i
constexpr int DN_NY = FV3_DN_NY;    // strips (waves) per workgroup
constexpr int DN_WIN = 81;          // cells of a corner window (at most 9 x 9)

// The march's cost.  FP64 (two extra passes) measured in the acoustic call, FP32
// on the launch alone: [1, 1, 1, 1] on six C48 tiles, 79 levels, 19.4 us by the
// FP64 figures, 17.4 by its own (17.7 in LDS blocks); six C128 72.2 and 60.7; in
// the mixed acoustic call on 96 C48 tiles the same.  Segments of more than 33
// rows where there are more than three waves measured slower (96 C48 tiles in
// FP32: one 49-row segment 266 us, two of 25 rows 230 us).
inline StripCost deln_cost(bool fp32) {
  return fp32 ? StripCost{0.62, 0.18, 0.62, 0.18, true, 6, 4.0, 3, FV3_DN_TJ}
              : StripCost{0.65, 0.28, 0.75, 0.37, false, 6, 4.0, 3, FV3_DN_TJ};
}

// Launch-wide arguments of the passes.
template <typename T>
struct DelnArgs {
  const T *q, *damp, *del6_u, *del6_v, *rarea;
  int nord4[4];
  int nmax;
  int use_damp;       // d2 starts as damp q (else q)
  int nbi, nbj, seg;  // strips, segments, rows per segment
  // corner windows of a plane: wi along i times wj along j (0 without corners;
  // 1 along a direction in which the tile is narrower than four cells)
  int wi, wj;
};

// The interfaces and cells at (i, j) that the corner windows own.
struct DelnOwned {
  bool fx, fy, cell;
};

template <typename T>
__device__ __forceinline__ DelnOwned deln_owned(const Dom& d, const DelnArgs<T>& a, int i, int j) {
  if (a.wi == 0) return {false, false, false};
  const bool xw = a.wi == 1 || i == d.is || i == d.is + 1;
  const bool yw = a.wj == 1 || j == d.js || j == d.js + 1;
  const bool xf = xw || i == d.ie || i == d.ie + 1, xc = xw || i == d.ie - 1 || i == d.ie;
  const bool yf = yw || j == d.je || j == d.je + 1, yc = yw || j == d.je - 1 || j == d.je;
  return {xf && yc, xc && yf, xc && yc};
}

// One wave's strip: P extra passes (0 .. 2).  EPI::In is what the epilogue
// reads for the cell row below, loaded a step ahead.
template <typename T, int P, typename EPI>
__device__ __forceinline__ void deln_strip(const Dom& d, const DelnArgs<T>& a, EPI& epi, T dk,
                                           int i0, int j0, int rows, const T* __restrict__ q,
                                           const T* __restrict__ u6, const T* __restrict__ v6,
                                           const T* __restrict__ ra) {
  const int lane = threadIdx.x;
  const int i = i0 - 3 + lane;
  const StripColumn<T> col(d, i);
  const bool out = lane >= 3 && lane < 3 + DN_TI;
  const bool cell_i = out && i <= d.iec, fx_i = out && i <= d.iec + 1;
  struct Row {
    T q, v, u, ra;
  };
  auto load = [&](int r) {
    Row w;
    w.q = col.f(q, r);
    w.v = col.m(v6, r);
    w.u = col.m(u6, r);
    w.ra = P > 0 ? col.m(ra, r) : T(0);
    return w;
  };
  const int r0 = j0 - 1 - P, r1 = j0 + rows + P;
  Row nx = load(r0);
  typename EPI::In en = epi.load(col, j0);
  T v1 = 0, v2 = 0, u1 = 0, u2 = 0, a1 = 0, a2 = 0;      // metric terms of rows r-1, r-2
  T d0 = 0, x0 = 0, y0 = 0, d1 = 0, x1 = 0, y1 = 0, d2 = 0;  // the passes' last rows
  T fp = 0, gp = 0;                                      // the fluxes of the row before
  for (int r = r0; r <= r1; ++r) {
    const Row w = nx;
    nx = load(r + 1);
    const int g = r - P - 1;  // cell row with all four fluxes
    const typename EPI::In ec = en;
    if (g + 1 > j0) en = epi.load(col, g + 1);
    T fc, gc;
    {
      const T dn = a.use_damp ? dk * w.q : w.q;
      const T xn = w.v * (lane_up(dn, 1) - dn);
      const T yn = w.u * (d0 - dn);
      if constexpr (P == 0) {
        fc = xn;
        gc = yn;
      } else {
        // d2_highorder (delnflux.py:178-181) of row r - 1
        const T e1 = (x0 - lane_dn(x0, 1) + y0 - yn) * a1;
        const T xe = -v1 * (lane_up(e1, 1) - e1);
        const T ye = -u1 * (d1 - e1);
        if constexpr (P == 1) {
          fc = xe;
          gc = ye;
        } else {
          const T e2 = (x1 - lane_dn(x1, 1) + y1 - ye) * a2;
          fc = -v2 * (lane_up(e2, 1) - e2);
          gc = -u2 * (d2 - e2);
          d2 = e2;
          x1 = xe;
          y1 = ye;
        }
        d1 = e1;
        x0 = xn;
        y0 = yn;
      }
      d0 = dn;
      v2 = v1;
      v1 = w.v;
      u2 = u1;
      u1 = w.u;
      a2 = a1;
      a1 = w.ra;
    }
    const T fe = lane_dn(fp, 1);
    if (g >= j0) {
      const DelnOwned own = deln_owned(d, a, i, g);
      epi.apply(ec, i, g, fp, fe, gp, gc, fx_i && g <= d.jec && !own.fx,
                cell_i && g <= d.jec + 1 && !own.fy, cell_i && g <= d.jec && !own.cell);
    }
    fp = fc;
    gp = gc;
  }
}

// Loads of one window cell (i, j), clamped as a strip's.
template <typename T>
struct DelnCell {
  int i, j, ni, nj;
  int64_t sj, sj2;
  __device__ __forceinline__ T at(const T* p, int64_t stride, int jj, int di) const {
    return p[(int64_t)min(max(jj, 0), nj - 1) * stride + min(max(i + di, 0), ni - 1)];
  }
  __device__ __forceinline__ T f(const T* p, int jj, int di = 0) const { return at(p, sj, jj, di); }
  __device__ __forceinline__ T m(const T* p, int jj, int di = 0) const { return at(p, sj2, jj, di); }
};

// One wave's corner window: the passes on a small box in LDS with the corner
// copies, for the interfaces deln_owned gives to the windows.
template <typename T, typename EPI>
__device__ __forceinline__ void deln_window(const Dom& d, const DelnArgs<T>& a,
                                            const CornerTable& tab, EPI& epi, T dk, int passes,
                                            bool corners, int win, T* lds,
                                            const T* __restrict__ q, const T* __restrict__ u6,
                                            const T* __restrict__ v6,
                                            const T* __restrict__ ra) {
  // the window: cells bi .. bi + nw - 1 by bj .. bj + nh - 1
  const bool east = a.wi == 2 && win % a.wi == 1, north = a.wj == 2 && win / a.wi == 1;
  const int bi = east ? d.ie - 4 : d.is - 3, nw = a.wi == 1 ? d.ie - d.is + 7 : 8;
  const int bj = north ? d.je - 4 : d.js - 3, nh = a.wj == 1 ? d.je - d.js + 7 : 8;
  const int nc = nw * nh, lane = threadIdx.x;
  T* const sd = lds;
  T* const sx = lds + DN_WIN;
  T* const sy = lds + 2 * DN_WIN;
  short* const src = (short*)(lds + 3 * DN_WIN);  // [2][DN_WIN]: a cell's x and y source
  // this lane's cells lane and lane + 64: their values after the x and y
  // copies, sources, and metric terms
  T dx[2], dy[2], mu[2], mv[2], ma[2];
  int srcx[2], srcy[2];
  auto each = [&](auto f) {
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int c = lane + 64 * m;
      if (c < nc) f(m, c, bi + c % nw, bj + c / nw);
    }
  };
  // one wave owns the window: in-order LDS, the fence only orders the compiler
  auto sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup", "local");
    __builtin_amdgcn_wave_barrier();
  };
  each([&](int m, int c, int i, int j) {
    const DelnCell<T> cell{i, j, d.ni, d.nj, d.sj, d.sj2};
    const T qv = cell.f(q, j);
    mv[m] = cell.m(v6, j);
    mu[m] = cell.m(u6, j);
    ma[m] = cell.m(ra, j);
    src[c] = src[DN_WIN + c] = (short)c;
    sd[c] = a.use_damp ? dk * qv : qv;
  });
  sync();
  if (corners) {
    for (int e = lane; e < tab.n; e += 64) {
      const int di = tab.dst_i[e] - bi, dj = tab.dst_j[e] - bj;
      const int si = tab.src_i[e] - bi, sj = tab.src_j[e] - bj;
      if (di >= 0 && di < nw && dj >= 0 && dj < nh && si >= 0 && si < nw && sj >= 0 && sj < nh)
        src[(tab.dir[e] ? DN_WIN : 0) + dj * nw + di] = (short)(sj * nw + si);
    }
    sync();
  }
  each([&](int m, int c, int, int) {
    srcx[m] = src[c];
    srcy[m] = src[DN_WIN + c];
  });
  for (int p = 0; p <= passes; ++p) {
    const T sgnv = p == 0 ? T(1) : T(-1);
    sync();
    // the x- and y-copied values (a y destination that is no x destination
    // keeps its own; sources are never corner cells)
    each([&](int m, int c, int, int) {
      dx[m] = sd[srcx[m]];
      dy[m] = srcy[m] != c ? sd[srcy[m]] : dx[m];
    });
    sync();
    each([&](int m, int c, int, int) { sd[c] = dx[m]; });
    sync();
    each([&](int m, int c, int, int) {
      sx[c] = c % nw > 0 ? sgnv * mv[m] * (sd[c - 1] - dx[m]) : T(0);
    });
    sync();
    each([&](int m, int c, int, int) { sd[c] = dy[m]; });
    sync();
    each([&](int m, int c, int, int) {
      sy[c] = c >= nw ? sgnv * mu[m] * (sd[c - nw] - dy[m]) : T(0);
    });
    sync();
    if (p < passes) {
      T nd[2];
      each([&](int m, int c, int, int) {
        nd[m] = c % nw + 1 < nw && c + nw < nc
                    ? (sx[c] - sx[c + 1] + sy[c] - sy[c + nw]) * ma[m]
                    : T(0);
      });
      sync();
      each([&](int m, int c, int, int) { sd[c] = nd[m]; });
    }
  }
  each([&](int, int c, int i, int j) {
    if (c % nw + 1 >= nw || c + nw >= nc) return;
    // each window emits what lies at its own end of the tile
    if ((a.wi == 2 && (east ? i < d.ie - 1 : i > d.is + 1)) ||
        (a.wj == 2 && (north ? j < d.je - 1 : j > d.js + 1)))
      return;
    const DelnOwned own = deln_owned(d, a, i, j);
    const bool ii = i >= d.isc && i <= d.iec, jj = j >= d.jsc && j <= d.jec;
    const bool fx = own.fx && i >= d.isc && i <= d.iec + 1 && jj;
    const bool fy = own.fy && j >= d.jsc && j <= d.jec + 1 && ii;
    const bool cl = own.cell && ii && jj;
    if (!(fx || fy || cl)) return;
    const DelnCell<T> cell{i, j, d.ni, d.nj, d.sj, d.sj2};
    epi.apply(epi.load(cell, j), i, j, sx[c], sx[c + 1], sy[c], sy[c + nw], fx, fy, cl);
  });
}

template <typename T, typename EPI>
__global__ void __launch_bounds__(DN_W * DN_NY)
    delnflux_kernel(Dom d, DelnArgs<T> a, CornerTable tab, EPI epi) {
  __shared__ T lds[DN_NY][4 * DN_WIN];  // three planes of values, one of sources
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int strips = a.nbi * a.nbj, per_plane = strips + a.wi * a.wj;
  const int total = per_plane * d.nk * d.ntiles;
  const int unit = xcd_logical_block(blockIdx.x, (total + DN_NY - 1) / DN_NY) * DN_NY + wave;
  if (unit >= total) return;
  const int plane = unit / per_plane, within = unit % per_plane;
  const int k = plane % d.nk, t = plane / d.nk;
  const int64_t off3 = (int64_t)t * d.st + (int64_t)k * d.sk;
  const int64_t off2 = (int64_t)t * d.st2;
  const int band = k < 3 ? k : 3;
  const int nord = band == 0   ? a.nord4[0]
                   : band == 1 ? a.nord4[1]
                   : band == 2 ? a.nord4[2]
                               : a.nord4[3];
  const T dk = a.damp[k];
  const int passes = nord > 0 ? a.nmax : 0;
  const T* q = a.q + off3;
  const T *u6 = a.del6_u + off2, *v6 = a.del6_v + off2, *ra = a.rarea + off2;
  epi.plane(d, k, dk, off3, off2);
  if (within >= strips) {
    deln_window<T>(d, a, tab, epi, dk, passes, nord > 0, within - strips, lds[wave], q, u6, v6, ra);
    return;
  }
  const int i0 = d.isc + within % a.nbi * DN_TI, j0 = d.jsc + within / a.nbi * a.seg;
  const int rows = min(a.seg, d.jec + 2 - j0);
  if (passes == 2)
    deln_strip<T, 2>(d, a, epi, dk, i0, j0, rows, q, u6, v6, ra);
  else if (passes == 1)
    deln_strip<T, 1>(d, a, epi, dk, i0, j0, rows, q, u6, v6, ra);
  else
    deln_strip<T, 0>(d, a, epi, dk, i0, j0, rows, q, u6, v6, ra);
}

// Runs the passes on every level of the domain with epilogue epi; `bytes` is
// the call's algorithmic traffic.
template <typename T, typename EPI>
int deln_launch(const fv3_domain* dom, const int32_t* nord4, int use_damp, const T* q,
                const T* damp, const T* del6_u, const T* del6_v, const T* rarea, const EPI& epi,
                double bytes, void* stream, const char* who) {
  int nmax = 0;
  for (int b = 0; b < 4; ++b) {
    // The reference states nord in {0, 2, 3} but its check accepts any value
    // up to 3 (delnflux.py:1024-1029), so 1 is accepted here too.
    FV3_REQUIRE(nord4[b] >= 0 && nord4[b] <= 3, FV3_E_UNSUPPORTED,
                "%s: nord must be in [0, 3] (got %d)", who, nord4[b]);
    nmax = nord4[b] > nmax ? nord4[b] : nmax;
  }
  // nmax = 3 puts the reference's d2 origin at isc - 4, outside the 3-cell
  // halo storage (delnflux.py:1031-1036), so it cannot run there either.
  FV3_REQUIRE(nmax <= 2, FV3_E_UNSUPPORTED, "%s: nord = 3 needs a 4-cell halo", who);
  if (dom->nk == 0 || dom->ntiles == 0) return FV3_OK;
  FV3_REQUIRE(dom->nk <= 65535 && dom->ntiles <= 65535, FV3_E_ARG, "%s: grid too large", who);
  Dom d = to_dom(dom);
  CornerTable tab;
  build_corner_table(dom, 3, &tab);
  DelnArgs<T> a;
  a.q = q;
  a.damp = damp;
  a.del6_u = del6_u;
  a.del6_v = del6_v;
  a.rarea = rarea;
  for (int b = 0; b < 4; ++b) a.nord4[b] = nord4[b];
  a.nmax = nmax;
  a.use_damp = use_damp;
  const int nfi = d.iec + 2 - d.isc, nfj = d.jec + 2 - d.jsc;
  a.nbi = (nfi + DN_TI - 1) / DN_TI;
  // corners the copies can reach (nord > 0 somewhere)
  a.wi = a.wj = 0;
  if (tab.n > 0 && nmax > 0) {
    a.wi = d.ie - d.is + 1 < 4 ? 1 : 2;
    a.wj = d.je - d.js + 1 < 4 ? 1 : 2;
  }
  a.seg = strip_segment_rows(nfj, (int64_t)a.nbi * d.nk * d.ntiles, deln_cost(sizeof(T) == 4));
  a.nbj = (nfj + a.seg - 1) / a.seg;
  const int64_t total = (int64_t)(a.nbi * a.nbj + a.wi * a.wj) * d.nk * d.ntiles;
  FV3_REQUIRE(total < (int64_t)1 << 30, FV3_E_ARG, "%s: grid too large", who);
  const int64_t blocks = (total + DN_NY - 1) / DN_NY;
  const int64_t launched = (blocks + kNumXcd - 1) / kNumXcd * kNumXcd;
  TimedLaunch timed("delnflux_kernel", as_stream(stream), bytes);
  hipLaunchKernelGGL((delnflux_kernel<T, EPI>), dim3((unsigned)launched), dim3(DN_W, DN_NY), 0,
                     as_stream(stream), d, a, tab, epi);
  FV3_HIP_CHECK_LAUNCH(who);
  return FV3_OK;
}

}  // namespace fv3
