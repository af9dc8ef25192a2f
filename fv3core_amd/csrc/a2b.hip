// AGrid2BGridFourthOrder (a2b_ord4): cell-centre values to cell corners.
//
// Reference: fv3core/stencils/a2b_ord4.py:1-695.  Three launches for up to four
// fields on one grid:
//   0 weights: the corner extrapolation weights from great-circle
//             distances on the A/B-grid longitudes and latitudes (12 per
//             tile, grid only);
//   1 edges:  the four corner extrapolations and the tile-edge lines
//             qout_x_edge / qout_y_edge, into qout;
//   2 interp: ppm_volume_mean_x and ppm_volume_mean_y, formed in registers as
//             a strip marches up the rows, and a2b_interpolation on the corners
//             off the tile-edge lines;
// and the optional copy back into qin.
#include "divide.hpp"
#include "kernels.hpp"
#include "strip.hpp"
#include "tile_config.hpp"
#include "timing.hpp"

namespace fv3 {

namespace {

constexpr double kA1 = 9.0 / 16.0;
constexpr double kA2 = -1.0 / 16.0;
constexpr double kB1 = 7.0 / 12.0;
constexpr double kB2 = -1.0 / 12.0;
constexpr double kCc1 = 2.0 / 3.0;
constexpr double kCc2 = -1.0 / 6.0;

// Runs f(i, j, k, t) on the perimeter of box b only (its first and last
// rows and columns), for levels [k0, k0 + nk) of every tile.
template <typename F>
__global__ void __launch_bounds__(256) perimeter_kernel(Box b, int k0, F f) {
  const int nbi = b.i1 - b.i0 + 1, nbj = b.j1 - b.j0 + 1;
  const int per = 2 * nbi + 2 * (nbj - 2);
  const int n = (int)(blockIdx.x * 256 + threadIdx.x);
  if (n >= per) return;
  int i, j;
  if (n < nbi) {
    i = b.i0 + n;
    j = b.j0;
  } else if (n < 2 * nbi) {
    i = b.i0 + n - nbi;
    j = b.j1;
  } else {
    const int m = n - 2 * nbi;
    i = m < nbj - 2 ? b.i0 : b.i1;
    j = b.j0 + 1 + (m < nbj - 2 ? m : m - (nbj - 2));
  }
  f(i, j, k0 + (int)blockIdx.y, (int)blockIdx.z);
}

template <typename F>
inline void launch_perimeter(hipStream_t s, const Dom& d, Box b, int k0, int nk, F f) {
  const int nbi = b.i1 - b.i0 + 1, nbj = b.j1 - b.j0 + 1;
  if (nbi <= 0 || nbj < 3 || nk <= 0 || d.ntiles <= 0) return;
  const int per = 2 * nbi + 2 * (nbj - 2);
  dim3 grid((unsigned)((per + 255) / 256), (unsigned)nk, (unsigned)d.ntiles);
  hipLaunchKernelGGL((perimeter_kernel<F>), grid, dim3(256), 0, s, b, k0, f);
}

// great_circle_dist (a2b_ord4.py:37-41)
template <typename T>
__device__ __forceinline__ T gc_dist(T p1a, T p1b, T p2a, T p2b) {
  const T sb = sin((p1b - p2b) / T(2));
  const T sa = sin((p1a - p2a) / T(2));
  const T tb = sb * sb;
  const T ta = sa * sa;
  return asin(sqrt(tb + cos(p1b) * cos(p2b) * ta)) * T(2);
}

// The three extrapolations of each cube corner (a2b_ord4.py:617-658), as
// centre offsets (di1, dj1, di2, dj2) from the corner point; corners in the
// order (isc, jsc), (iec+1, jsc), (iec+1, jec+1), (isc, jec+1).
__constant__ int kCornerTaps[4][3][4] = {
    {{0, 0, 1, 1}, {-1, 0, -2, 1}, {0, -1, 1, -2}},
    {{-1, 0, -2, 1}, {-1, -1, -2, -2}, {0, 0, 1, 1}},
    {{-1, -1, -2, -2}, {0, -1, 1, -2}, {-1, 0, -2, 1}},
    {{0, -1, 1, -2}, {-1, -1, -2, -2}, {0, 0, 1, 1}},
};

// Weight x1 / (x2 - x1) of extrapolation e (corner e / 3, tap e % 3) of
// tile blockIdx.x: extrap_corner is qa + x1 / (x2 - x1) (qa - qb) with
// great-circle distances that depend on the grid only, so they are formed
// once per call here instead of once per level in the perimeter launch.
//
// The same launch forms, per tile and row j in [jsc-2, jec+2], the cell-length
// ratios of the one-sided x volume means (qx_edge_west's g_in = dxa(p+1) /
// dxa(p) and g_ou = dxa(p-2) / dxa(p-1) at p = is, then at p = ie+1), which
// depend on the grid only; the means read them instead of dividing again on
// every level (the same divisions, so the same bits).
template <typename T>
__global__ void __launch_bounds__(64) corner_weights_kernel(Met<T> m, Dom d, T* w, T* xr,
                                                            int nrow) {
  const int e = threadIdx.x;
  const int t = blockIdx.x;
  for (int r = e; r < nrow; r += 64) {
    const T* dx = m.dxa + (int64_t)t * d.st2 + (int64_t)(d.jsc - 2 + r) * d.sj2;
    T* out = xr + ((int64_t)t * nrow + r) * 4;
    if (d.is >= 2 && d.is + 1 < d.ni) {
      out[0] = dx[d.is + 1] / dx[d.is];
      out[1] = dx[d.is - 2] / dx[d.is - 1];
    }
    if (d.ie >= 1 && d.ie + 2 < d.ni) {
      out[2] = dx[d.ie + 2] / dx[d.ie + 1];
      out[3] = dx[d.ie - 1] / dx[d.ie];
    }
  }
  if (e >= 12) return;
  const int corner = e / 3, tap = e % 3;
  const int ic = (corner == 1 || corner == 2) ? d.iec + 1 : d.isc;
  const int jc = (corner >= 2) ? d.jec + 1 : d.jsc;
  const int64_t o2 = at2(d, ic, jc, t);
  const int* tp = kCornerTaps[corner][tap];
  const int64_t a1 = o2 + tp[0] + (int64_t)tp[1] * d.sj2, a2 = o2 + tp[2] + (int64_t)tp[3] * d.sj2;
  const T p0a = m.bgrid1[o2], p0b = m.bgrid2[o2];
  const T x1 = gc_dist(m.agrid1[a1], m.agrid2[a1], p0a, p0b);
  const T x2 = gc_dist(m.agrid1[a2], m.agrid2[a2], p0a, p0b);
  w[t * 12 + e] = x1 / (x2 - x1);
}

template <typename T>
__device__ __forceinline__ T qx_edge_west(const T* q, const T* dx) {
  // q[], dx[] centred at the point (index 0 = the point)
  const T g_in = dx[1] / dx[0];
  const T g_ou = dx[-2] / dx[-1];
  return T(0.5) * (((T(2) + g_in) * q[0] - q[1]) / (T(1) + g_in) +
                   ((T(2) + g_ou) * q[-1] - q[-2]) / (T(1) + g_ou));
}

template <typename T>
__device__ __forceinline__ T qx_edge_west2(const T* q, const T* dx) {
  const T g_in = dx[0] / dx[-1];
  const T g_ou = dx[-3] / dx[-2];
  const T left = T(0.5) * (((T(2) + g_in) * q[-1] - q[0]) / (T(1) + g_in) +
                           ((T(2) + g_ou) * q[-2] - q[-3]) / (T(1) + g_ou));
  const T right = T(kB2) * (q[-1] + q[2]) + T(kB1) * (q[0] + q[1]);
  return (T(3) * (g_in * q[-1] + q[0]) - (g_in * left + right)) / (T(2) + T(2) * g_in);
}

template <typename T>
__device__ __forceinline__ T qx_edge_east(const T* q, const T* dx) {
  const T g_in = dx[-2] / dx[-1];
  const T g_ou = dx[1] / dx[0];
  return T(0.5) * (((T(2) + g_in) * q[-1] - q[-2]) / (T(1) + g_in) +
                   ((T(2) + g_ou) * q[0] - q[1]) / (T(1) + g_ou));
}

template <typename T>
__device__ __forceinline__ T qx_edge_east2(const T* q, const T* dx) {
  const T g_in = dx[-1] / dx[0];
  const T g_ou = dx[2] / dx[1];
  const T right = T(0.5) * (((T(2) + g_in) * q[0] - q[-1]) / (T(1) + g_in) +
                            ((T(2) + g_ou) * q[1] - q[2]) / (T(1) + g_ou));
  const T left = T(kB2) * (q[-3] + q[0]) + T(kB1) * (q[-2] + q[-1]);
  return (T(3) * (q[-1] + g_in * q[0]) - (g_in * right + left)) / (T(2) + T(2) * g_in);
}

// ppm_volume_mean_x / _y at a point: q7/dx7 hold cells p-3..p+3 along the
// direction; a = absolute index of the point along it, s/e the anchors.
template <typename T>
__device__ __forceinline__ T volume_mean(const T (&q7)[7], const T (&dx7)[7], int a, int s,
                                         int e) {
  const T* q = q7 + 3;
  const T* dx = dx7 + 3;
  // regions in the reference's order: start, start+1, end+1, end (last wins)
  if (a == e) return qx_edge_east2(q, dx);
  if (a == e + 1) return qx_edge_east(q, dx);
  if (a == s + 1) return qx_edge_west2(q, dx);
  if (a == s) return qx_edge_west(q, dx);
  return T(kB2) * (q[-2] + q[1]) + T(kB1) * (q[-1] + q[0]);
}

// The field and level of level kk of a set.
template <typename T>
__device__ __forceinline__ int a2b_field(const A2BFields<T>& f, int& k) {
  int n = 0;
  while (n + 1 < f.n && k >= f.nk[n]) {
    k -= f.nk[n];
    ++n;
  }
  k += f.k0[n];
  return n;
}

// Volume means and interpolation on the corners [ci0, ci1] x [cj0, cj1] off the
// tile-edge lines: at row r of q a strip forms the x means of row r and the
// corners of row r - 2, whose means and rows lie in windows of registers.
//
// What bounds it: memory, one row of q in and one of corners out per step of
// about 130 instructions.  The LDS blocks of 58 x 16 corners it replaces read
// six more rows per block and passed both means through LDS behind two
// barriers.  KR rows are loaded at a time, one block ahead (two measured 2 %
// faster than three and 15 % faster than four, which leave fewer waves).
// Measured in the acoustic call with its five fields in two sets instead of
// five, means, weights and edge lines together: six C96 tiles 374 -> 262 us, 96
// C48 tiles mixed 1330 -> 960 us, six C128 tiles 650 -> 435 us, six C12 tiles
// 93 -> 60 us.
template <typename T>
struct A2BInterp {
  Met<T> m;
  A2BFields<T> f;
  const T* xr;
  int nrow;  // rows of the edge ratios (jsc-2 .. jec+2)
  int ci0, ci1, cj0, cj1;

  static constexpr int KR = 2;  // rows loaded at a time
  struct Rows {
    T q[KR], e[KR], gi[KR], go[KR];
  };

  __device__ __forceinline__ void operator()(const Dom& d, int i0, int j0, int rows, int k,
                                             int t) const {
    const int n = a2b_field(f, k);
    const int64_t o3 = (int64_t)t * d.st + (int64_t)k * d.sk, o2 = (int64_t)t * d.st2;
    const T* const q = f.qin[n] + o3;
    T* const qout = f.qout[n] + o3;
    const int lane = threadIdx.x, i = i0 - 3 + lane;
    const StripColumn<T> col(d, i);
    const bool out = lane >= 3 && lane < 61 && i <= ci1;
    // x means: form 0 interior, 1 outer (at is or ie + 1), 2 inner west, 3 inner
    // east, in volume_mean's order of precedence.  The outer form at is equals
    // the one at ie + 1 (the same two halves, added in the other order), and the
    // inner form at is + 1 or ie is the outer form of its neighbour combined
    // with interior means, mirrored for the east side; its ratio is the outer
    // form's g_in or g_ou.
    int form = 0;
    if (i == d.ie)
      form = 3;
    else if (i == d.ie + 1)
      form = 1;
    else if (i == d.is + 1)
      form = 2;
    else if (i == d.is)
      form = 1;
    const bool west = form == 2;
    // the corner on the tile-edge line beside i == is + 1 or ie, if any
    const int ce = i == d.ie ? i + 1 : i == d.is + 1 ? i - 1 : min(max(i, ci0), ci1);
    const StripColumn<T> edge(d, ce);
    const T* const gr = xr + (int64_t)t * nrow * 4 + (i <= d.is + 1 ? 0 : 2);
    auto load = [&](int r) {
      Rows w;
#pragma unroll
      for (int u = 0; u < KR; ++u) {
        w.q[u] = col.f(q, r + u);
        w.e[u] = edge.f(qout, r + u - 2);
        const T* g = gr + min(max(r + u - (d.jsc - 2), 0), nrow - 1) * 4;
        w.gi[u] = g[0];
        w.go[u] = g[1];
      }
      return w;
    };
    T q1 = 0, q2 = 0, q3 = 0, q4 = 0, q5 = 0;  // rows r - 1 .. r - 5
    T s1 = 0, s2 = 0, s3 = 0, s4 = 0, s5 = 0;  // their x means
    const int last = j0 + rows - 1;
    auto row = [&](int r, T q0, T ev, T g_in, T g_ou) {
      const T qm1 = lane_up(q0, 1), qm2 = lane_up(qm1, 1), qm3 = lane_up(qm2, 1);
      const T qp1 = lane_dn(q0, 1), qp2 = lane_dn(qp1, 1);
      T s0 = T(kB2) * (qm2 + qp1) + T(kB1) * (qm1 + q0);
      if (form != 0) {
        // the outer form at point p = i, i - 1 (inner west) or i + 1 (inner east)
        const T b0 = form == 1 ? q0 : west ? qm1 : qp1, b1 = form == 1 ? qp1 : west ? q0 : qp2;
        const T a1 = form == 1 ? qm1 : west ? qm2 : q0, a2 = form == 1 ? qm2 : west ? qm3 : qm1;
        const T outer = T(0.5) * (Divisor<T>(T(1) + g_in).quot((T(2) + g_in) * b0 - b1) +
                                  Divisor<T>(T(1) + g_ou).quot((T(2) + g_ou) * a1 - a2));
        if (form == 1) {
          s0 = outer;
        } else {
          // qx_edge_west2, or qx_edge_east2 with q[k] -> q[-1-k]
          const T g = west ? g_in : g_ou;
          const T w0 = west ? q0 : qm1, w1 = west ? qp1 : qm2, wm = west ? qm1 : q0,
                  w2 = west ? qp2 : qm3;
          const T inner = T(kB2) * (wm + w2) + T(kB1) * (w0 + w1);
          s0 = Divisor<T>(T(2) + T(2) * g).quot(T(3) * (g * wm + w0) - (g * outer + inner));
        }
      }
      // corners of row j
      const int j = r - 2;
      T y = T(kB2) * (q4 + q1) + T(kB1) * (q3 + q2);
      if (j == d.js || j == d.js + 1 || j == d.je || j == d.je + 1) {
        const T q7[7] = {q5, q4, q3, q2, q1, q0, T(0)};
        T dy7[7];
#pragma unroll
        for (int u = 0; u < 6; ++u) dy7[u] = col.m(m.dya + o2, j + u - 3);
        dy7[6] = T(1);
        y = volume_mean(q7, dy7, j, d.js, d.je);
      }
      const T ym1 = lane_up(y, 1), ym2 = lane_up(ym1, 1), ym3 = lane_up(ym2, 1);
      const T yp1 = lane_dn(y, 1), yp2 = lane_dn(yp1, 1);
      T qxx = T(kA2) * (s4 + s1) + T(kA1) * (s3 + s2);
      if (j == d.js + 1) {
        const T up = T(kA2) * (s3 + s0) + T(kA1) * (s2 + s1);
        qxx = T(kCc1) * (s3 + s2) + T(kCc2) * (col.f(qout, j - 1) + up);
      }
      if (j == d.je) {
        const T lo = T(kA2) * (s5 + s2) + T(kA1) * (s4 + s3);
        qxx = T(kCc1) * (s3 + s2) + T(kCc2) * (col.f(qout, j + 1) + lo);
      }
      T qyy = T(kA2) * (ym2 + yp1) + T(kA1) * (ym1 + y);
      if (i == d.is + 1) {
        const T rr = T(kA2) * (ym1 + yp2) + T(kA1) * (y + yp1);
        qyy = T(kCc1) * (ym1 + y) + T(kCc2) * (ev + rr);
      }
      if (i == d.ie) {
        const T l = T(kA2) * (ym3 + y) + T(kA1) * (ym2 + ym1);
        qyy = T(kCc1) * (ym1 + y) + T(kCc2) * (ev + l);
      }
      col.store(qout, j, T(0.5) * (qxx + qyy), out && j >= j0 && j <= last);
      q5 = q4;
      q4 = q3;
      q3 = q2;
      q2 = q1;
      q1 = q0;
      s5 = s4;
      s4 = s3;
      s3 = s2;
      s2 = s1;
      s1 = s0;
    };
    // rows r0 .. last + 2 in blocks of KR
    const int r0 = j0 - 3, blocks = (rows + 5 + KR - 1) / KR;
    strip_march(0, blocks - 1, load(r0), [&](int b, const Rows& w, Rows& nx) {
      const int r = r0 + b * KR;
      nx = load(r + KR);
#pragma unroll
      for (int u = 0; u < KR; ++u) row(r + u, w.q[u], w.e[u], w.gi[u], w.go[u]);
    });
  }
};

// The same means and interpolation in LDS blocks, for small launches: one
// workgroup owns AB_TI x AB_TJ corners of one level.  It stages q over the block
// plus a 3-cell halo, forms the x means on the rows j - 3 .. j + 2 and the y
// means on the columns i - 3 .. i + 2 of its corners there, and interpolates.
// Lane x of every wave owns LDS column x; wave y owns rows y, y + AB_NY, ...
// Six more rows are read per block and both means pass through LDS behind two
// barriers, but a block's rows run side by side where the march runs them one
// after the other.  Measured on 12 to 192 cells a side, 4 to 127 levels, one to
// 96 tiles, one field or the pressure gradient's four, the march overtakes it
// between 3000 and 4500 blocks.  One field of 79 levels, block and march: one
// C12 tile 13.7 and 16.3 us, six 15.2 and 21.0, six C48 29.4 and 32.3, six C96
// 64.0 and 61.3, 96 C48 274 and 208 us.
constexpr int64_t kA2BMarchBlocks = 3500;
// The march's cost is the del-n march's (delnflux.hpp), with five rows beside a
// segment's own and the cap on every launch (six C128 tiles, 79 levels, 1.4 waves
// a SIMD: 64 rows 99.5 us, 32 rows 94.8).
constexpr StripCost kA2BCost{0.65, 0.28, 0.75, 0.37, false, 5, 4.0, 3, FV3_AB_TJ, 0.0};
constexpr int AB_W = 64;         // LDS columns = TI + 6
constexpr int AB_TI = AB_W - 6;  // corners per block in i
constexpr int AB_TJ = 16;        // corners per block in j
constexpr int AB_H = AB_TJ + 6;  // q rows: j0-3 .. j0+TJ+2
constexpr int AB_NY = 8;         // waves per block

template <typename T>
__global__ void __launch_bounds__(AB_W * AB_NY)
    a2b_block_kernel(Dom d, A2BInterp<T> p, int nbi) {
  __shared__ T sq[AB_H][AB_W];
  __shared__ T sx[AB_H - 1][AB_W];  // x means on rows j0-3 .. j0+TJ+1
  __shared__ T sy[AB_TJ][AB_W];     // y means on rows j0 .. j0+TJ-1
  const int li = threadIdx.x, ty = threadIdx.y;
  const int bi = blockIdx.x % nbi, bj = blockIdx.x / nbi;
  int k = (int)blockIdx.y;
  const int n = a2b_field(p.f, k), t = blockIdx.z;
  const int i0 = p.ci0 + bi * AB_TI, j0 = p.cj0 + bj * AB_TJ;
  const int i = i0 - 3 + li;  // absolute column of this lane
  const int jb = j0 - 3;      // absolute row of LDS row 0
  const bool col_ok = i >= 0 && i < d.ni;
  const int64_t off3 = (int64_t)t * d.st + (int64_t)k * d.sk;
  const int64_t off2 = (int64_t)t * d.st2;
  const T* const qin = p.f.qin[n] + off3;
  T* const qout = p.f.qout[n] + off3;  // holds the tile-edge lines
  for (int r = ty; r < AB_H; r += AB_NY) {
    const int j = jb + r;
    sq[r][li] = (col_ok && j >= 0 && j < d.nj) ? qin[(int64_t)j * d.sj + i] : T(0);
  }
  __syncthreads();
  // x means, i in [isc, iec+1], j in [jsc-2, jec+2], in the march's forms
  if (li >= 3 && li < AB_W - 3 && i >= d.isc && i <= d.iec + 1) {
    int form = 0, sh = 0;  // sh: the outer form's point, relative to i
    if (i == d.ie) {
      form = 3;
      sh = 1;
    } else if (i == d.ie + 1) {
      form = 1;
    } else if (i == d.is + 1) {
      form = 2;
      sh = -1;
    } else if (i == d.is) {
      form = 1;
    }
    const bool west = form == 2;
    for (int r = ty; r < AB_H - 1; r += AB_NY) {
      const int j = jb + r;
      if (j < d.jsc - 2 || j > d.jec + 2) continue;
      const T* q = &sq[r][li];
      T v = T(kB2) * (q[-2] + q[1]) + T(kB1) * (q[-1] + q[0]);
      if (form != 0) {
        const T* gr = p.xr + ((int64_t)t * p.nrow + (j - (d.jsc - 2))) * 4;
        const bool wside = i <= d.is + 1;
        const T g_in = wside ? gr[0] : gr[2], g_ou = wside ? gr[1] : gr[3];
        const T* qb = q + sh;
        const T outer = T(0.5) * (((T(2) + g_in) * qb[0] - qb[1]) / (T(1) + g_in) +
                                  ((T(2) + g_ou) * qb[-1] - qb[-2]) / (T(1) + g_ou));
        if (form == 1) {
          v = outer;
        } else {
          auto qm = [&](int m) { return west ? q[m] : q[-1 - m]; };
          const T g = west ? g_in : g_ou;
          const T inner = T(kB2) * (qm(-1) + qm(2)) + T(kB1) * (qm(0) + qm(1));
          v = (T(3) * (g * qm(-1) + qm(0)) - (g * outer + inner)) / (T(2) + T(2) * g);
        }
      }
      sx[r][li] = v;
    }
  }
  // y means, i in [isc-2, iec+2], j in [jsc, jec+1]; only the rows on the
  // tile-edge interfaces read the cell lengths
  if (li < AB_W - 1 && i >= d.isc - 2 && i <= d.iec + 2) {
    for (int r = ty; r < AB_TJ; r += AB_NY) {
      const int j = j0 + r;
      if (j >= d.jsc && j <= d.jec + 1) {
        T v = T(kB2) * (sq[r + 1][li] + sq[r + 4][li]) + T(kB1) * (sq[r + 2][li] + sq[r + 3][li]);
        if (j == d.js || j == d.js + 1 || j == d.je || j == d.je + 1) {
          const int64_t o2 = off2 + (int64_t)j * d.sj2 + i;
          T q7[7], dy7[7];
#pragma unroll
          for (int u = 0; u < 7; ++u) {
            q7[u] = sq[r + u][li];
            dy7[u] = p.m.dya[o2 + (int64_t)(u - 3) * d.sj2];
          }
          v = volume_mean(q7, dy7, j, d.js, d.je);
        }
        sy[r][li] = v;
      }
    }
  }
  __syncthreads();
  // a2b_interpolation on the block's corners (qx rows and qy columns -3 .. +2)
  if (li < 3 || li >= 3 + AB_TI || i > p.ci1) return;
  const int64_t sj = d.sj;
  for (int r = ty; r < AB_TJ; r += AB_NY) {
    const int j = j0 + r;
    if (j > p.cj1) break;
    const int x = r + 3;  // sx row of j
    T* const o = qout + (int64_t)j * sj + i;
    T qxx = T(kA2) * (sx[x - 2][li] + sx[x + 1][li]) + T(kA1) * (sx[x - 1][li] + sx[x][li]);
    T qyy = T(kA2) * (sy[r][li - 2] + sy[r][li + 1]) + T(kA1) * (sy[r][li - 1] + sy[r][li]);
    if (j == d.js + 1) {
      const T up = T(kA2) * (sx[x - 1][li] + sx[x + 2][li]) + T(kA1) * (sx[x][li] + sx[x + 1][li]);
      qxx = T(kCc1) * (sx[x - 1][li] + sx[x][li]) + T(kCc2) * (o[-sj] + up);
    }
    if (j == d.je) {
      const T lo = T(kA2) * (sx[x - 3][li] + sx[x][li]) + T(kA1) * (sx[x - 2][li] + sx[x - 1][li]);
      qxx = T(kCc1) * (sx[x - 1][li] + sx[x][li]) + T(kCc2) * (o[sj] + lo);
    }
    if (i == d.is + 1) {
      const T rr = T(kA2) * (sy[r][li - 1] + sy[r][li + 2]) + T(kA1) * (sy[r][li] + sy[r][li + 1]);
      qyy = T(kCc1) * (sy[r][li - 1] + sy[r][li]) + T(kCc2) * (o[-1] + rr);
    }
    if (i == d.ie) {
      const T l = T(kA2) * (sy[r][li - 3] + sy[r][li]) + T(kA1) * (sy[r][li - 2] + sy[r][li - 1]);
      qyy = T(kCc1) * (sy[r][li - 1] + sy[r][li]) + T(kCc2) * (o[1] + l);
    }
    *o = T(0.5) * (qxx + qyy);
  }
}

}  // namespace

template <typename T>
int launch_a2b_ord4(hipStream_t s, const fv3_domain* dom, const Met<T>& m,
                    const A2BFields<T>& f, T* weights, const char* who) {
  int nk = 0;
  for (int n = 0; n < f.n; ++n) nk += f.nk[n];
  if (nk <= 0) return FV3_OK;
  Dom d = to_dom(dom);
  const bool w = has_edge(dom->i_start), e = has_edge(dom->i_end);
  const bool so = has_edge(dom->j_start), no = has_edge(dom->j_end);
  const int js2 = so ? d.jsc + 1 : d.jsc, je1 = no ? d.jec : d.jec + 1;
  const int is2 = w ? d.isc + 1 : d.isc, ie1 = e ? d.iec : d.iec + 1;
  // 0: corner extrapolation weights, 12 per tile, into the head of the slab,
  // and the x volume means' edge ratios after them
  T* const cw = weights;
  T* const xr = weights + 12 * (int64_t)d.ntiles;
  const int nrow = d.jec - d.jsc + 5;
  hipLaunchKernelGGL((corner_weights_kernel<T>), dim3((unsigned)d.ntiles), dim3(64), 0, s, m, d,
                     cw, xr, nrow);
  FV3_HIP_CHECK_LAUNCH(who);
  // 1: corners and edge lines: only the perimeter of [isc, iec+1]^2 can hold them
  const Box bx{d.isc, d.iec + 1, d.jsc, d.jec + 1};
  launch_perimeter(s, d, bx, 0, nk, [=] __device__(int i, int j, int k, int t) {
    const int n = a2b_field(f, k);
    const T* const qin = f.qin[n];
    const int64_t o = at3(d, i, j, k, t);
    const int64_t o2 = at2(d, i, j, t);
    T val;
    const bool ci = i == d.isc || i == d.iec + 1, cj = j == d.jsc || j == d.jec + 1;
    // a corner where the tile has one edge only lies on that edge's line
    if (ci && ((i == d.isc && w) || (i == d.iec + 1 && e)) && j >= js2 && j <= je1) {
      // qout_x_edge (a2b_ord4.py:313-323): q2 at j and j - 1
      const T* dxa = m.dxa;
      const T q2 = (qin[o - 1] * dxa[o2] + qin[o] * dxa[o2 - 1]) / (dxa[o2 - 1] + dxa[o2]);
      const int64_t om = o - d.sj, om2 = o2 - d.sj2;
      const T q2m = (qin[om - 1] * dxa[om2] + qin[om] * dxa[om2 - 1]) / (dxa[om2 - 1] + dxa[om2]);
      const T wgt = (i == d.isc ? m.edge_w : m.edge_e)[o2];
      val = wgt * q2m + (T(1) - wgt) * q2;
    } else if (cj && ((j == d.jsc && so) || (j == d.jec + 1 && no)) && i >= is2 && i <= ie1) {
      const T* dya = m.dya;
      const int64_t sj = d.sj, sj2 = d.sj2;
      const T q1 = (qin[o - sj] * dya[o2] + qin[o] * dya[o2 - sj2]) / (dya[o2 - sj2] + dya[o2]);
      const T q1m = (qin[o - 1 - sj] * dya[o2 - 1] + qin[o - 1] * dya[o2 - 1 - sj2]) /
                    (dya[o2 - 1 - sj2] + dya[o2 - 1]);
      const T wgt = (j == d.jsc ? m.edge_s : m.edge_n)[o2];
      val = wgt * q1m + (T(1) - wgt) * q1;
    } else if (ci && cj) {
      // _sw_corner at (isc, jsc), _nw_corner at (iec+1, jsc), _ne_corner at
      // (iec+1, jec+1), _se_corner at (isc, jec+1) (a2b_ord4.py:617-658)
      const int corner = j == d.jsc ? (i == d.isc ? 0 : 1) : (i == d.iec + 1 ? 2 : 3);
      T ex[3];
#pragma unroll
      for (int tap = 0; tap < 3; ++tap) {
        const int* tp = kCornerTaps[corner][tap];
        const T qa = qin[o + tp[0] + (int64_t)tp[1] * d.sj];
        const T qb = qin[o + tp[2] + (int64_t)tp[3] * d.sj];
        ex[tap] = qa + cw[t * 12 + corner * 3 + tap] * (qa - qb);
      }
      val = (ex[0] + ex[1] + ex[2]) * (T(1) / T(3));
    } else {
      return;
    }
    f.qout[n][o] = val;
  });
  FV3_HIP_CHECK_LAUNCH(who);
  // 2: volume means and interpolation off the tile-edge lines
  const A2BInterp<T> interp{m, f, xr, nrow, is2, ie1, js2, je1};
  if (is2 > ie1 || js2 > je1) return FV3_OK;
  Dom dk = d;
  dk.nk = nk;
  // q read, qout written (per corner-level)
  TimedLaunch timed("a2b_interp_kernel", s,
                    2.0 * sizeof(T) * (double)(ie1 - is2 + 1) * (je1 - js2 + 1) * nk * d.ntiles);
  const int nbi = (ie1 - is2 + AB_TI) / AB_TI, nbj = (je1 - js2 + AB_TJ) / AB_TJ;
  if ((int64_t)nbi * nbj * nk * d.ntiles < kA2BMarchBlocks) {
    hipLaunchKernelGGL((a2b_block_kernel<T>),
                       dim3((unsigned)(nbi * nbj), (unsigned)nk, (unsigned)d.ntiles),
                       dim3(AB_W, AB_NY), 0, s, d, interp, nbi);
    FV3_HIP_CHECK_LAUNCH(who);
    return FV3_OK;
  }
  return launch_strips<FV3_AB_NY>(s, dk, is2, ie1, js2, je1, 58, kA2BCost, interp, who);
}

template int launch_a2b_ord4<double>(hipStream_t, const fv3_domain*, const Met<double>&,
                                     const A2BFields<double>&, double*, const char*);
template int launch_a2b_ord4<float>(hipStream_t, const fv3_domain*, const Met<float>&,
                                    const A2BFields<float>&, float*, const char*);

int check_a2b_metrics(const fv3_metrics* g, const char* who) {
  FV3_REQUIRE(g && g->dxa && g->dya && g->agrid1 && g->agrid2 && g->bgrid1 && g->bgrid2 &&
                  g->edge_w && g->edge_e && g->edge_s && g->edge_n,
              FV3_E_ARG, "%s: a2b_ord4 needs dxa, dya, agrid1/2, bgrid1/2 and edge_w/e/s/n",
              who);
  return FV3_OK;
}

}  // namespace fv3

extern "C" int32_t fv3_plan_a2b_rows(int32_t rows, int64_t planes, int32_t most) {
  fv3::StripCost cost = fv3::kA2BCost;
  if (most > 0) cost.most = most;
  return fv3::strip_segment_rows(rows, planes, cost);
}

extern "C" int32_t fv3_a2b_ord4_f64(const fv3_domain* dom, const fv3_metrics* g, int32_t replace,
                                    double* qin, double* qout, double* work, int64_t work_slab,
                                    void* stream) {
  using namespace fv3;
  const char* who = "fv3_a2b_ord4";
  int rc = check_domain(dom, who);
  if (rc) return rc;
  rc = check_a2b_metrics(g, who);
  if (rc) return rc;
  FV3_REQUIRE(qin && qout && work, FV3_E_ARG, "%s: NULL pointer", who);
  if (dom->nk == 0 || dom->ntiles == 0) return FV3_OK;
  FV3_REQUIRE(work_slab >= (int64_t)(dom->ntiles - 1) * dom->st + (int64_t)dom->nk * dom->sk,
              FV3_E_ARG, "%s: work_slab too small", who);
  const Met<double> m = to_met<double>(g);
  const hipStream_t s = as_stream(stream);
  rc = launch_a2b_ord4<double>(s, dom, m, A2BFields<double>{1, {qin}, {qout}, {0}, {dom->nk}}, work,
                               who);
  if (rc || !replace) return rc;
  const Dom d = to_dom(dom);
  launch_box(s, d, Box{d.isc, d.iec + 1, d.jsc, d.jec + 1}, 0, d.nk,
             [=] __device__(int i, int j, int k, int t) {
               const int64_t o = at3(d, i, j, k, t);
               qin[o] = qout[o];
             });
  FV3_HIP_CHECK_LAUNCH(who);
  return FV3_OK;
}
