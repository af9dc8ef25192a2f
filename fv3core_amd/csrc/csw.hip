// C-grid half step: DGrid2AGrid2CGridVectors (d2a2c_vect) and
// CGridShallowWaterDynamics (c_sw).
//
// Reference: fv3core/stencils/d2a2c_vect.py:1-651, fv3core/stencils/c_sw.py:
// 1-659.  Three marches up the rows of each level, 64 columns to a wave, the
// neighbours across i by lane shifts and those across j in registers, so that
// only what a later march needs goes through memory.  Region statements become
// index tests against the tile-edge anchors, with the reference's statement
// order deciding which formula a point gets.
//
// Launch sequence of fv3_c_sw (workspace slabs in brackets):
//   1 fill:      x, then y corner fills of delp, pt, w
//   2 d2a2c:     ua, va, ut, vt; uc, vc before the update [W0, W1]
//   3 transport: delpc, ptc, omga, ke [W2]; divergence_corner -> divgd (nord > 0)
//   4 update:    vorticity; update_y_velocity (vc), update_x_velocity (uc)
//
// What bounds it: memory, at about half the rate of a large copy (a wave streams
// up to 16 fields in pieces of 512 bytes; rows per segment from 9 to 35, 1 to 16
// waves a workgroup, tiles spread over the XCDs or kept on one and non-temporal
// stores all measure within 10 %).  31 passes over full-size fields against 54
// of one pointwise pass per stencil.  Measured, FP64, 79 levels: six C97 tiles
// 593 -> 423 us (d2a2c 169 -> 126, transport with the divergence 301 -> 195,
// update with the vorticity 112 -> 97); 96 C48 tiles in FP32 1510 -> 975 us;
// six C12 tiles, where a launch is its latency, 52 -> 47 us.
#include "strip.hpp"
#include "stencil.hpp"

namespace fv3 {

namespace {

// Lagrange weights of a2b_ord4 (a2b_ord4.py:26-34) and the volume-conserving
// cubic weights of d2a2c_vect.py:12-15.
constexpr double kA1 = 9.0 / 16.0;
constexpr double kA2 = -1.0 / 16.0;
constexpr double kC1 = -2.0 / 14.0;
constexpr double kC2 = 11.0 / 14.0;
constexpr double kC3 = 5.0 / 14.0;
constexpr double kBigNumber = 1e30;

// Index bounds of DGrid2AGrid2CGridVectors.__init__ (d2a2c_vect.py:374-470).
struct D2A2CBounds {
  int is1, ie1, js1, je1, is2, ie2, js2, je2;
  int ifirst, ilast, jfirst, jlast;
  int avg_offset;
};

D2A2CBounds d2a2c_bounds(const fv3_domain* d) {
  const int nxc = d->iec - d->isc + 1, nyc = d->jec - d->jsc + 1;
  const int nx = d->iec + 1, ny = d->jec + 1;
  const int h = d->isc;  // n_halo
  const bool w = has_edge(d->i_start), e = has_edge(d->i_end);
  const bool s = has_edge(d->j_start), n = has_edge(d->j_end);
  int npt = 4;  // not nested
  if (npt > nxc - 1 || npt > nyc - 1) npt = 0;
  const int off = 2;
  D2A2CBounds b;
  b.js1 = s ? npt + off : d->jsc - 1;
  b.je1 = n ? ny - npt : d->jec + 1;
  b.is1 = w ? npt + off : d->isc - h;
  b.ie1 = e ? nx - npt : d->iec + h;
  b.is2 = w ? npt + off : d->isc - 1;
  b.ie2 = e ? nx - npt : d->iec + 1;
  b.js2 = s ? npt + off : d->jsc - h;
  b.je2 = n ? ny - npt : d->jec + h;
  b.ifirst = w ? d->isc + 2 : d->isc - 1;
  b.ilast = e ? d->iec - 1 : d->iec + 2;
  b.jfirst = s ? d->jsc + 2 : d->jsc - 1;
  b.jlast = n ? d->jec - 1 : d->jec + 2;
  b.avg_offset = npt == 0 ? -1 : 3;
  return b;
}

template <typename T>
__device__ __forceinline__ T contravariant(T v1, T v2, T cosa, T rsin2) {
  return (v1 - v2 * cosa) * rsin2;
}

// The marches' cost, measured on the launches alone: rows per segment of c_sw and
// of d2a2c_vect on 12 to 128 cells a side, one to 96 tiles.  By the del-n march's
// figures six C12 tiles, 79 levels, took 53.2 us in FP64 and 39.6 in FP32, six
// C24 71.8 and 50.9; by these 46.8 and 36.9, 65.5 and 48.5.  Above three waves
// the heights differ little.
inline StripCost csw_cost(bool fp32) {
  return fp32 ? StripCost{0.62, 0.27, 0.75, 0.37, true, 2, 3.5, 2, 33}
              : StripCost{0.7, 0.53, 1.2, 0.52, true, 2, 3.5, 2, 33};
}
inline StripCost d2a2c_cost(bool fp32) {
  return fp32 ? StripCost{0.62, 0.27, 0.75, 0.37, true, 3, 3.5, 2, 33}
              : StripCost{0.78, 0.39, 1.0, 0.44, true, 3, 3.5, 2, 33};
}

// ---------------------------------------------------------------- d2a2c_vect
// set_tmps, lagrange_interpolation_y_p1/x_p1, avg_box, contravariant_components,
// ut_main + east_west_edges, north_south_edges + vt_main and, when geo != 0,
// geoadjust_ut / geoadjust_vt, as one march: at row r the strip forms the A-grid
// winds of row r, uc of row r and vc of row r - 1.
//
// The corner fills turn the interpolated covariant winds (and the A-grid winds)
// by a quarter: a cell (is - 1 - a, js - 1) takes -+ the other component of
// (is - 1, js + a) before uc is formed, a cell (is - 1, js - 1 - a) that of
// (is + a, js - 1) before vc is formed, and so at the other corners.  The few
// lanes and rows they reach form the other component from u and v again.
template <typename T>
struct D2A2C {
  D2A2CBounds b;
  Met<T> m;
  int geo;
  T dt2;
  const T *u, *v;
  T *ua, *va, *uc, *vc, *utc, *vtc;

  // utmp / vtmp of any cell from u rows j - 1 .. j + 2 / v columns i - 1 .. i + 2
  __device__ __forceinline__ T ut_of(bool band, int i, int j, T um, T u0, T u1, T u2) const {
    if (band) return T(0.5) * (u0 + u1);
    return i >= b.is1 && i <= b.ie1 && j >= b.js1 && j <= b.je1
               ? T(kA2) * (um + u2) + T(kA1) * (u0 + u1)
               : T(kBigNumber);
  }
  __device__ __forceinline__ T vt_of(bool band, int i, int j, T vm, T v0, T v1, T v2) const {
    if (band) return T(0.5) * (v0 + v1);
    return i >= b.is2 && i <= b.ie2 && j >= b.js2 && j <= b.je2
               ? T(kA2) * (vm + v2) + T(kA1) * (v0 + v1)
               : T(kBigNumber);
  }
  __device__ __forceinline__ bool band(const Dom& d, int i, int j) const {
    const int off = b.avg_offset;
    return j < d.js + off || j > d.je - off || i < d.is + off || i > d.ie - off;
  }

  // what a corner fill reads: both components at cell (i, j), which lies in the
  // band beside the tile edges
  __device__ __forceinline__ void cell(const Dom& d, int64_t o3, int64_t o2, int i, int j, T& ut,
                                       T& vt, T& uaa, T& vaa) const {
    const T *pu = u + o3 + (int64_t)j * d.sj + i, *pv = v + o3 + (int64_t)j * d.sj + i;
    const int64_t om = o2 + (int64_t)j * d.sj2 + i;
    ut = T(0.5) * (pu[0] + pu[d.sj]);
    vt = T(0.5) * (pv[0] + pv[1]);
    uaa = contravariant(ut, vt, m.cosa_s[om], m.rsin2[om]);
    vaa = contravariant(vt, ut, m.cosa_s[om], m.rsin2[om]);
  }

  __device__ __forceinline__ void operator()(const Dom& d, int i0, int r0, int rows, int k,
                                             int t) const {
    const int lane = threadIdx.x, i = i0 - 2 + lane;
    const StripColumn<T> col(d, i);
    const int64_t o3 = (int64_t)t * d.st + (int64_t)k * d.sk, o2 = (int64_t)t * d.st2;
    const bool out = lane >= 2 && lane < 62;
    const bool a_i = out && i <= d.iec + 2, uc_i = a_i && i >= d.isc - 1,
               vc_i = uc_i && i <= d.iec + 1;
    const bool cl = i < d.is || i > d.ie;  // a corner's columns
    // x's edge formulas (east_west_edges)
    const bool xe = i == d.is || i == d.ie + 1, xl = i == d.is - 1 || i == d.ie,
               xr = !xl && (i == d.is + 1 || i == d.ie + 2);
    struct Row {
      T v, u3, cs, r2, cu, ru, dy, s3, s1, dxa, cv, rv, dx, s4, s2;
    };
    auto load = [&](int r) {
      Row w;
      w.v = col.f(v + o3, r);
      w.u3 = col.f(u + o3, r + 2);
      w.cs = col.m(m.cosa_s + o2, r);
      w.r2 = col.m(m.rsin2 + o2, r);
      w.cu = col.m(m.cosa_u + o2, r);
      w.ru = col.m(m.rsin_u + o2, r);
      w.s3 = col.m(m.sin_sg3 + o2, r, -1);
      w.s1 = col.m(m.sin_sg1 + o2, r);
      w.dxa = col.m(m.dxa + o2, r);
      w.cv = col.m(m.cosa_v + o2, r - 1);
      w.rv = col.m(m.rsin_v + o2, r - 1);
      w.s4 = col.m(m.sin_sg4 + o2, r - 2);
      w.s2 = col.m(m.sin_sg2 + o2, r - 1);
      w.dy = geo ? col.m(m.dy + o2, r) : T(0);
      w.dx = geo ? col.m(m.dx + o2, r - 1) : T(0);
      return w;
    };
    const int ra = r0 - 3;
    T um = 0, u0 = col.f(u + o3, ra - 1), u1 = col.f(u + o3, ra), u2 = col.f(u + o3, ra + 1);
    T vt1 = 0, vt2 = 0, vt3 = 0, va1 = 0, va2 = 0, va3 = 0;  // rows r - 1 .. r - 3
    strip_march(ra, r0 + rows - 1, load(ra), [&](int r, const Row& w, Row& nx) {
      nx = load(r + 1);
      um = u0;
      u0 = u1;
      u1 = u2;
      u2 = w.u3;
      const bool bd = band(d, i, r);
      const T v1 = lane_dn(w.v, 1);
      const T ut = ut_of(bd, i, r, um, u0, u1, u2);
      const T vt = vt_of(bd, i, r, lane_up(w.v, 1), w.v, v1, lane_dn(v1, 1));
      T utx = ut, vty = vt;
      T uax = contravariant(ut, vt, w.cs, w.r2), vay = contravariant(vt, ut, w.cs, w.r2);
      if (r < d.js || r > d.je) {
        if (cl) {
          const bool south = r < d.js, west = i < d.is;
          const int ax = west ? d.is - 1 - i : i - d.ie - 1, ay = south ? d.js - 1 - r : r - d.je - 1;
          const T mult = west == south ? T(-1) : T(1);
          T cut, cvt, cua, cva;
          if (ay == 0 && ax < 3) {
            cell(d, o3, o2, west ? d.is - 1 : d.ie + 1, south ? d.js + ax : d.je - ax, cut, cvt,
                 cua, cva);
            utx = mult * cvt;
            if (ax < 2) uax = mult * cva;
          }
          if (ax == 0 && ay < 3) {
            cell(d, o3, o2, west ? d.is + ay : d.ie - ay, south ? d.js - 1 : d.je + 1, cut, cvt,
                 cua, cva);
            vty = mult * cut;
            if (ay < 2) vay = mult * cua;
          }
        }
      }
      // uc of row r
      T ucv, utv;
      {
        const T tm2 = lane_up(utx, 2), tm1 = lane_up(utx, 1), tp1 = lane_dn(utx, 1);
        const T am2 = lane_up(uax, 2), am1 = lane_up(uax, 1), ap1 = lane_dn(uax, 1);
        const T dm2 = lane_up(w.dxa, 2), dm1 = lane_up(w.dxa, 1), dp1 = lane_dn(w.dxa, 1);
        if (xl || xr)
          ucv = T(kC1) * (xl ? tm2 : tp1) + T(kC2) * (xl ? tm1 : utx) + T(kC3) * (xl ? utx : tm1);
        else
          ucv = T(kA2) * (tm2 + tp1) + T(kA1) * (tm1 + utx);
        utv = contravariant(ucv, w.v, w.cu, w.ru);
        if (xe) {
          // edge_interpolate4_x (d2a2c_vect.py:254-260; n2 uses t1 as there)
          const T t1 = dm2 + dm1, t2 = w.dxa + dp1;
          const T n1 = (t1 + dm1) * am1 - dm1 * am2;
          const T n2 = (t1 + w.dxa) * uax - w.dxa * ap1;
          utv = T(0.5) * (n1 / t1 + n2 / t2);
          ucv = utv > T(0) ? utv * w.s3 : utv * w.s1;
        }
        if (geo) utv = utv > T(0) ? dt2 * utv * w.dy * w.s3 : dt2 * utv * w.dy * w.s1;
      }
      // vc of row j = r - 1
      const int j = r - 1;
      T vcv, vtv;
      const bool jm = j >= b.jfirst && j <= b.jlast;
      if (!jm && (j == d.js || j == d.je + 1) && j != d.js - 1 && j != d.je) {
        const T dm2 = col.m(m.dya + o2, j - 2), dm1 = col.m(m.dya + o2, j - 1),
                d0 = col.m(m.dya + o2, j), dp1 = col.m(m.dya + o2, j + 1);
        const T t1 = dm2 + dm1, t2 = d0 + dp1;
        const T n1 = (t1 + dm1) * va2 - dm1 * va3;
        const T n2 = (t1 + d0) * va1 - d0 * vay;
        vtv = T(0.5) * (n1 / t1 + n2 / t2);
        vcv = vtv > T(0) ? vtv * w.s4 : vtv * w.s2;
      } else {
        if (!jm && (j == d.js - 1 || j == d.je))
          vcv = T(kC1) * vt3 + T(kC2) * vt2 + T(kC3) * vt1;
        else if (!jm && (j == d.js + 1 || j == d.je + 2))
          vcv = T(kC1) * vty + T(kC2) * vt1 + T(kC3) * vt2;
        else
          vcv = T(kA2) * (vt3 + vty) + T(kA1) * (vt2 + vt1);
        vtv = contravariant(vcv, um, w.cv, w.rv);
      }
      if (geo) vtv = vtv > T(0) ? dt2 * vtv * w.dx * w.s4 : dt2 * vtv * w.dx * w.s2;
      const bool sa = a_i && r >= r0 && r <= d.jec + 2;
      const bool su = uc_i && r >= r0 && r >= d.jsc - 1 && r <= d.jec + 1;
      const bool sv = vc_i && r >= r0 && j >= d.jsc - 1;
      col.store(ua + o3, r, uax, sa);
      col.store(va + o3, r, vay, sa);
      col.store(uc + o3, r, ucv, su);
      col.store(utc + o3, r, utv, su);
      col.store(vc + o3, j, vcv, sv);
      col.store(vtc + o3, j, vtv, sv);
      vt3 = vt2;
      vt2 = vt1;
      vt1 = vty;
      va3 = va2;
      va2 = va1;
      va1 = vay;
    });
  }
};

// The d2a2c part shared by fv3_d2a2c_vect and fv3_c_sw.
template <typename T>
int run_d2a2c(hipStream_t s, const fv3_domain* dom, const Met<T>& m, int geo, T dt2, T* uc,
              T* vc, const T* u, const T* v, T* ua, T* va, T* utc, T* vtc, const char* who) {
  const Dom d = to_dom(dom);
  const D2A2C<T> f{d2a2c_bounds(dom), m, geo, dt2, u, v, ua, va, uc, vc, utc, vtc};
  return launch_strips(s, d, d.isc - 2, d.iec + 2, d.jsc - 2, d.jec + 3, 60,
                       d2a2c_cost(sizeof(T) == 4), f, who);
}

// ----------------------------------------------------------------------- c_sw
// compute_nonhydro_fluxes_x, transportdelp_update_vorticity_and_kineticenergy
// on [isc-1, iec+1]^2 with initialize_delpc_ptc (zero) on the rest of the full
// domain and, when divg is given, divergence_corner on [isc, iec+1] x
// [jsc, jec+1]: at row r the strip forms the x fluxes and the divergence of row
// r and finishes the cells of row r - 1.
//
// delp, pt and w hold the x corner fills with the y fills over them; only the
// cell next to a corner, (is - 1, js - 1), differs between the two, and the x
// fluxes take it from (is - 1, js), where the x fill reads.
template <typename T>
struct CswTransport {
  Met<T> m;
  T dt2;
  const T *delp, *pt, *w, *utc, *vtc, *ua, *va, *uc, *vc, *u, *v;
  T *delpc, *ptc, *wc, *ke, *divg;

  __device__ __forceinline__ void operator()(const Dom& d, int i0, int j0, int rows, int k,
                                             int t) const {
    const int lane = threadIdx.x, i = i0 - 1 + lane;
    const StripColumn<T> col(d, i);
    const int64_t o3 = (int64_t)t * d.st + (int64_t)k * d.sk, o2 = (int64_t)t * d.st2;
    const bool out = lane >= 1 && lane < 63 && i <= d.iec + 3;
    const bool cell_i = out && i >= d.isc - 1 && i <= d.iec + 1;
    const bool div_i = out && i >= d.isc && i <= d.iec + 1;
    const bool west = i == d.is || i == d.ie + 1;  // beside a tile edge
    const bool kl = i == d.ie || i == d.is - 1, kr = !kl && west;
    const bool corner = i == d.is - 1 || i == d.ie + 1;
    // rows that only hold zeros
    for (int j = j0; j < j0 + rows; ++j) {
      if (j >= d.jsc - 1 && j <= d.jec + 1) continue;
      if (out) {
        (delpc + o3 + (int64_t)j * d.sj)[i] = T(0);
        (ptc + o3 + (int64_t)j * d.sj)[i] = T(0);
      }
    }
    const int jb = max(j0, d.jsc - 1), je = min(j0 + rows - 1, d.jec + 1);
    if (jb > je) return;
    struct Row {
      T dp, pt, w, ut, vt, ua, va, uc, vc, u, v, ra;
    };
    struct Div {
      T s1, s2, s3, s4, c1, c2, c3, c4, dxc, dyc, rac;
    };
    auto load = [&](int r) {
      Row x;
      x.dp = col.f(delp + o3, r);
      x.pt = col.f(pt + o3, r);
      x.w = col.f(w + o3, r);
      x.ut = col.f(utc + o3, r);
      x.vt = col.f(vtc + o3, r);
      x.ua = col.f(ua + o3, r);
      x.va = col.f(va + o3, r);
      x.uc = col.f(uc + o3, r);
      x.vc = col.f(vc + o3, r);
      x.u = col.f(u + o3, r);
      x.v = col.f(v + o3, r);
      x.ra = col.m(m.rarea + o2, r);
      return x;
    };
    auto load_div = [&](int r) {
      Div y{};
      y.s1 = col.m(m.sin_sg1 + o2, r);
      y.c1 = col.m(m.cos_sg1 + o2, r);
      y.s3 = col.m(m.sin_sg3 + o2, r);
      y.c3 = col.m(m.cos_sg3 + o2, r);
      if (divg) {
        y.s2 = col.m(m.sin_sg2 + o2, r);
        y.c2 = col.m(m.cos_sg2 + o2, r);
        y.s4 = col.m(m.sin_sg4 + o2, r - 1);
        y.c4 = col.m(m.cos_sg4 + o2, r - 1);
        y.dxc = col.m(m.dxc + o2, r);
        y.dyc = col.m(m.dyc + o2, r);
        y.rac = col.m(m.rarea_c + o2, r);
      }
      return y;
    };
    const T half = T(0.5), quarter = T(0.25);
    T dp1 = 0, pt1 = 0, w1 = 0, va1 = 0, vc1 = 0, ra1 = 0, u1 = 0;  // row r - 1
    T gx = 0, gx1 = 0, gx2 = 0;                                     // its x flux differences
    T fy = 0, fy1 = 0, fy2 = 0, kx = 0, vf1 = 0;  // its lower y fluxes, ua kev, vf
    struct Both {
      Row x;
      Div y;
    };
    const Both first{load(jb - 1), load_div(jb - 1)};
    strip_march(jb - 1, je + 1, first, [&](int r, const Both& cur, Both& nx) {
      nx.x = load(r + 1);
      nx.y = load_div(r + 1);
      const Row& x = cur.x;
      const Div& y = cur.y;
      // y fluxes at interface r
      const bool dn = x.vt > T(0);
      const T hy1 = x.vt * (dn ? dp1 : x.dp);
      const T hy = hy1 * (dn ? pt1 : x.pt), hy2 = hy1 * (dn ? w1 : x.w);
      // the cells of row j = r - 1
      const int j = r - 1;
      const T dpc = dp1 + (gx1 + fy1 - hy1) * ra1;
      const T ptv = (pt1 * dp1 + (gx + fy - hy) * ra1) / dpc;
      const T wv = (w1 * dp1 + (gx2 + fy2 - hy2) * ra1) / dpc;
      T vort = va1 > T(0) ? vc1 : x.vc;
      if (j == d.js - 1 || j == d.je) {
        if (va1 <= T(0)) vort = vort * col.m(m.sin_sg4 + o2, j) + x.u * col.m(m.cos_sg4 + o2, j);
      } else if (j == d.js || j == d.je + 1) {
        if (va1 > T(0)) vort = vort * col.m(m.sin_sg2 + o2, j) + u1 * col.m(m.cos_sg2 + o2, j);
      }
      col.store(delpc + o3, j, cell_i ? dpc : T(0), out && j >= jb);
      col.store(ptc + o3, j, cell_i ? ptv : T(0), out && j >= jb);
      col.store(wc + o3, j, wv, cell_i && j >= jb);
      col.store(ke + o3, j, half * dt2 * (kx + va1 * vort), cell_i && j >= jb);
      // x fluxes of row r
      {
        T xd = x.dp, xp = x.pt, xw = x.w;
        if ((r == d.js - 1 || r == d.je + 1) && corner) {
          const int rs = r < d.js ? r + 1 : r - 1;
          xd = col.f(delp + o3, rs);
          xp = col.f(pt + o3, rs);
          xw = col.f(w + o3, rs);
        }
        const T ld = lane_up(xd, 1), lp = lane_up(xp, 1), lw = lane_up(xw, 1);
        const bool rt = x.ut > T(0);
        const T f1 = x.ut * (rt ? ld : xd);
        const T f = f1 * (rt ? lp : xp), f2 = f1 * (rt ? lw : xw);
        gx1 = f1 - lane_dn(f1, 1);
        gx = f - lane_dn(f, 1);
        gx2 = f2 - lane_dn(f2, 1);
      }
      // the x part of the kinetic energy of row r
      {
        const T ucp = lane_dn(x.uc, 1), vp = lane_dn(x.v, 1);
        T kev = x.ua > T(0) ? x.uc : ucp;
        if (kl) {
          if (x.ua <= T(0)) kev = kev * y.s3 + vp * y.c3;
        } else if (kr) {
          if (x.ua > T(0)) kev = kev * y.s1 + x.v * y.c1;
        }
        kx = x.ua * kev;
      }
      if (divg) {
        // divergence_corner (c_sw.py:172-289): next to a tile edge the flux
        // along it leaves the other wind out, and at a tile corner one of the
        // two vf is missing
        const bool south = r == d.js || r == d.je + 1;
        const T s3m = lane_up(y.s3, 1), c3m = lane_up(y.c3, 1), uam = lane_up(x.ua, 1);
        const T uw = south ? x.u : x.u - quarter * (va1 + x.va) * (y.c4 + y.c2);
        const T uf = uw * y.dyc * half * (y.s4 + y.s2);
        const T vw = west ? x.v : x.v - quarter * (uam + x.ua) * (c3m + y.c1);
        const T vf = vw * y.dxc * half * (s3m + y.s1);
        const T uf1 = lane_up(uf, 1);
        T sum = vf1 - vf;
        if (south && west) sum = r == d.js ? -vf : vf1;
        col.store(divg + o3, r, (sum + uf1 - uf) * y.rac,
                  div_i && r >= jb && r >= d.jsc && r <= je);
        vf1 = vf;
      }
      dp1 = x.dp;
      pt1 = x.pt;
      w1 = x.w;
      va1 = x.va;
      vc1 = x.vc;
      ra1 = x.ra;
      u1 = x.u;
      fy = hy;
      fy1 = hy1;
      fy2 = hy2;
    });
  }
};

// circulation_cgrid + absolute_vorticity on [isc, iec+1]^2, update_y_velocity
// (vc on [isc, iec] x [jsc, jec+1]) and update_x_velocity (uc on [isc, iec+1] x
// [jsc, jec]); c and e are the winds of D2A2C, copied to uc and vc around those
// boxes.  At row r the strip forms the vorticity and vc of row r and uc of row
// r - 1.
template <typename T>
struct CswUpdate {
  Met<T> m;
  T dt2;
  const T *c, *e, *ke, *u, *v;
  T *uc, *vc;

  __device__ __forceinline__ void operator()(const Dom& d, int i0, int j0, int rows, int k,
                                             int t) const {
    const int lane = threadIdx.x, i = i0 - 1 + lane;
    const StripColumn<T> col(d, i);
    const int64_t o3 = (int64_t)t * d.st + (int64_t)k * d.sk, o2 = (int64_t)t * d.st2;
    const bool uc_i = lane >= 1 && lane < 63 && i <= d.iec + 2, vc_i = uc_i && i <= d.iec + 1;
    const bool uu = i >= d.isc && i <= d.iec + 1, vu = i >= d.isc && i <= d.iec;
    const bool west = i == d.is || i == d.ie + 1;
    struct Row {
      T c, e, ke, u, v, dxc, dyc, f, rac, cv, sv, cu, su, rdx, rdy;
    };
    auto load = [&](int r) {
      Row x;
      x.c = col.f(c + o3, r);
      x.e = col.f(e + o3, r);
      x.ke = col.f(ke + o3, r);
      x.u = col.f(u + o3, r);
      x.v = col.f(v + o3, r);
      x.dxc = col.m(m.dxc + o2, r);
      x.dyc = col.m(m.dyc + o2, r);
      x.f = col.m(m.fC + o2, r);
      x.rac = col.m(m.rarea_c + o2, r);
      x.cv = col.m(m.cosa_v + o2, r);
      x.sv = col.m(m.sina_v + o2, r);
      x.cu = col.m(m.cosa_u + o2, r);
      x.su = col.m(m.sina_u + o2, r);
      x.rdx = col.m(m.rdxc + o2, r);
      x.rdy = col.m(m.rdyc + o2, r);
      return x;
    };
    T fx1 = 0, ke1 = 0;                     // row r - 1
    T c1 = 0, tmp1 = 0, vort1 = 0, g1 = 0;  // its uc and what updates it
    strip_march(j0 - 1, j0 + rows, load(j0 - 1), [&](int r, const Row& x, Row& nx) {
      nx = load(r + 1);
      const T fx = x.dxc * x.c, fy = x.dyc * x.e;
      const T fy1 = lane_up(fy, 1);
      T cir = fx1 - fx - fy1 + fy;
      if (r == d.js || r == d.je + 1) {
        if (i == d.is)
          cir = fx1 - fx + fy;
        else if (i == d.ie + 1)
          cir = fx1 - fx - fy1;
      }
      const T vort = x.f + x.rac * cir;
      const T vortp = lane_dn(vort, 1), kem = lane_up(x.ke, 1);
      const int j = r - 1;
      const T uflux = tmp1 > T(0) ? vort1 : vort;
      col.store(uc + o3, j, uu && j >= d.jsc && j <= d.jec ? c1 + tmp1 * uflux + g1 : c1,
                uc_i && j >= j0 && j <= d.jec + 1);
      T vcv = x.e;
      if (r >= d.jsc && r <= d.jec + 1) {
        const T tmp =
            (r == d.js || r == d.je + 1) ? dt2 * x.u : dt2 * (x.u - vcv * x.cv) / x.sv;
        const T flux = tmp > T(0) ? vort : vortp;
        const T up = vcv - tmp * flux + x.rdy * (ke1 - x.ke);
        vcv = vu ? up : vcv;
      }
      col.store(vc + o3, r, vcv, vc_i && r >= j0 && r < j0 + rows);
      c1 = x.c;
      tmp1 = west ? dt2 * x.v : dt2 * (x.v - x.c * x.cu) / x.su;
      g1 = x.rdx * (kem - x.ke);
      vort1 = vort;
      fx1 = fx;
      ke1 = x.ke;
    });
  }
};

const int kUnitMult[4] = {1, 1, 1, 1};

int check_csw_domain(const fv3_domain* dom, const char* who) {
  int rc = check_domain(dom, who);
  if (rc) return rc;
  FV3_REQUIRE(dom->isc >= 3 && dom->jsc >= 3, FV3_E_ARG, "%s: the stencils need a 3-cell halo",
              who);
  FV3_REQUIRE(dom->iec - dom->isc + 1 >= 5 && dom->jec - dom->jsc + 1 >= 5, FV3_E_ARG,
              "%s: compute domain must be at least 5 x 5", who);
  return FV3_OK;
}

#define FV3_REQ_MET(g, name, who) \
  FV3_REQUIRE((g)->name != nullptr, FV3_E_ARG, "%s: metric " #name " is NULL", who)

int check_d2a2c_metrics(const fv3_metrics* g, const char* who) {
  FV3_REQUIRE(g != nullptr, FV3_E_ARG, "%s: NULL metrics", who);
  FV3_REQ_MET(g, cosa_s, who);
  FV3_REQ_MET(g, rsin2, who);
  FV3_REQ_MET(g, cosa_u, who);
  FV3_REQ_MET(g, cosa_v, who);
  FV3_REQ_MET(g, rsin_u, who);
  FV3_REQ_MET(g, rsin_v, who);
  FV3_REQ_MET(g, dxa, who);
  FV3_REQ_MET(g, dya, who);
  FV3_REQ_MET(g, sin_sg1, who);
  FV3_REQ_MET(g, sin_sg2, who);
  FV3_REQ_MET(g, sin_sg3, who);
  FV3_REQ_MET(g, sin_sg4, who);
  return FV3_OK;
}

int check_csw_metrics(const fv3_metrics* g, int nord, const char* who) {
  int rc = check_d2a2c_metrics(g, who);
  if (rc) return rc;
  FV3_REQ_MET(g, dx, who);
  FV3_REQ_MET(g, dy, who);
  FV3_REQ_MET(g, dxc, who);
  FV3_REQ_MET(g, dyc, who);
  FV3_REQ_MET(g, rdxc, who);
  FV3_REQ_MET(g, rdyc, who);
  FV3_REQ_MET(g, rarea, who);
  FV3_REQ_MET(g, rarea_c, who);
  FV3_REQ_MET(g, cos_sg1, who);
  FV3_REQ_MET(g, cos_sg2, who);
  FV3_REQ_MET(g, cos_sg3, who);
  FV3_REQ_MET(g, cos_sg4, who);
  FV3_REQ_MET(g, sina_u, who);
  FV3_REQ_MET(g, sina_v, who);
  FV3_REQ_MET(g, fC, who);
  (void)nord;
  return FV3_OK;
}

template <typename T>
int run_c_sw(const fv3_domain* dom, const fv3_metrics* g, int32_t nord, T dt2, T* delp, T* pt,
             const T* u, const T* v, T* w, T* uc, T* vc, T* ua, T* va, T* ut, T* vt, T* divgd,
             T* omga, T* delpc, T* ptc, T* work, int64_t work_slab, void* stream) {
  const char* who = "fv3_c_sw";
  int rc = check_csw_domain(dom, who);
  if (rc) return rc;
  rc = check_csw_metrics(g, nord, who);
  if (rc) return rc;
  FV3_REQUIRE(delp && pt && u && v && w && uc && vc && ua && va && ut && vt && omga && delpc &&
                  ptc && work && (nord <= 0 || divgd),
              FV3_E_ARG, "%s: NULL pointer", who);
  if (dom->nk == 0 || dom->ntiles == 0) return FV3_OK;
  FV3_REQUIRE(work_slab >= (int64_t)(dom->ntiles - 1) * dom->st + (int64_t)dom->nk * dom->sk,
              FV3_E_ARG, "%s: work_slab too small", who);
  const Met<T> m = to_met<T>(g);
  hipStream_t s = as_stream(stream);
  T* uc0 = work;
  T* vc0 = work + work_slab;
  T* ke = work + 2 * work_slab;
  const Dom d = to_dom(dom);
  const Box edges{dom->isc - 3, dom->iec + 3, dom->jsc - 3, dom->jec + 3};
  FillTable fill;
  fill.n = 0;
  FillFields<T> ff{};
  ff.f[0] = delp;
  ff.f[1] = pt;
  ff.f[2] = w;
  for (int f = 0; f < 3; ++f) append_fill(&fill, dom, kFill2X, f, f, kUnitMult, edges);
  for (int f = 0; f < 3; ++f) append_fill(&fill, dom, kFill2Y, f, f, kUnitMult, edges);
  launch_fill(s, d, fill, ff);
  FV3_HIP_CHECK_LAUNCH(who);
  rc = run_d2a2c<T>(s, dom, m, 1, dt2, uc0, vc0, u, v, ua, va, ut, vt, who);
  if (rc) return rc;
  const CswTransport<T> transport{m,  dt2, delp, pt, w,     ut,  vt, ua, va,
                                  uc0, vc0, u,   v,  delpc, ptc, omga, ke,
                                  nord > 0 ? divgd : nullptr};
  const StripCost cost = csw_cost(sizeof(T) == 4);
  rc = launch_strips(s, d, d.isc - 3, d.iec + 3, d.jsc - 3, d.jec + 3, 62, cost, transport, who);
  if (rc) return rc;
  const CswUpdate<T> update{m, dt2, uc0, vc0, ke, u, v, uc, vc};
  return launch_strips(s, d, d.isc - 1, d.iec + 2, d.jsc - 1, d.jec + 2, 62, cost, update, who);
}

}  // namespace

}  // namespace fv3

extern "C" {

int32_t fv3_plan_c_sw_rows(int32_t rows, int64_t planes, int32_t fp32) {
  return fv3::strip_segment_rows(rows, planes, fv3::csw_cost(fp32 != 0));
}

int32_t fv3_plan_d2a2c_rows(int32_t rows, int64_t planes, int32_t fp32) {
  return fv3::strip_segment_rows(rows, planes, fv3::d2a2c_cost(fp32 != 0));
}

int32_t fv3_d2a2c_vect_f64(const fv3_domain* dom, const fv3_metrics* g, double* uc, double* vc,
                           const double* u, const double* v, double* ua, double* va,
                           double* utc, double* vtc, double* work, int64_t work_slab,
                           void* stream) {
  using namespace fv3;
  const char* who = "fv3_d2a2c_vect";
  int rc = check_csw_domain(dom, who);
  if (rc) return rc;
  rc = check_d2a2c_metrics(g, who);
  if (rc) return rc;
  FV3_REQUIRE(uc && vc && u && v && ua && va && utc && vtc && work, FV3_E_ARG,
              "%s: NULL pointer", who);
  if (dom->nk == 0 || dom->ntiles == 0) return FV3_OK;
  FV3_REQUIRE(work_slab >= (int64_t)(dom->ntiles - 1) * dom->st + (int64_t)dom->nk * dom->sk,
              FV3_E_ARG, "%s: work_slab too small", who);
  const Met<double> m = to_met<double>(g);
  return run_d2a2c<double>(as_stream(stream), dom, m, 0, 0.0, uc, vc, u, v, ua, va, utc, vtc,
                           who);
}

int32_t fv3_c_sw_f64(const fv3_domain* dom, const fv3_metrics* g, int32_t nord, double dt2,
                     double* delp, double* pt, const double* u, const double* v, double* w,
                     double* uc, double* vc, double* ua, double* va, double* ut, double* vt,
                     double* divgd, double* omga, double* delpc, double* ptc, double* work,
                     int64_t work_slab, void* stream) {
  return fv3::run_c_sw<double>(dom, g, nord, dt2, delp, pt, u, v, w, uc, vc, ua, va, ut, vt,
                               divgd, omga, delpc, ptc, work, work_slab, stream);
}

int32_t fv3_c_sw_f32(const fv3_domain* dom, const fv3_metrics* g, int32_t nord, float dt2,
                     float* delp, float* pt, const float* u, const float* v, float* w, float* uc,
                     float* vc, float* ua, float* va, float* ut, float* vt, float* divgd,
                     float* omga, float* delpc, float* ptc, float* work, int64_t work_slab,
                     void* stream) {
  return fv3::run_c_sw<float>(dom, g, nord, dt2, delp, pt, u, v, w, uc, vc, ua, va, ut, vt,
                              divgd, omga, delpc, ptc, work, work_slab, stream);
}
}
