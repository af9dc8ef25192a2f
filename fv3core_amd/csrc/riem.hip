// Semi-implicit vertical sound-wave solvers: sim1_solver, RiemannSolverC,
// RiemannSolver3.
//
// Reference: fv3core/stencils/sim1_solver.py:11-101 (two tridiagonal
// solves, for the pressure perturbation and for w, plus the dz update),
// riem_solver_c.py:13-165 and riem_solver3.py:24-242 (precompute / sim1 /
// finalize stencils).  Each solver is one kernel, always in FP64.  Two are
// here for each: this file's, which spreads a column's levels over a workgroup
// and reads every input level once (pt, cappa and w a second time at the end,
// which frees their registers in between), and riem_column.hpp's, which runs a
// column in one thread, where that is the faster one (riem_form).
//
// What bounds it: nearly all of the ~1000 instructions a column-level takes
// are the logs, exps and divisions of pressures and coefficients, which
// depend on their own level only; what one level hands to the next is two
// division chains and a few sums.  One thread per column runs everything in
// sequence, at less than one wave per SIMD on a C96 cube, and reads the inputs
// again in each of six sweeps.  Here a column's levels are spread over a
// workgroup: RC columns by sets of LV levels, two sets to a wave.  Every thread
// forms the independent part of its levels in registers, and the recurrences
// run as eight chains (A to H): the waves take turns, each carrying the running
// values through its levels and handing them on through LDS.  Sums and
// recurrences keep the order of the stencils' sweeps, so the results are those
// of the one-thread form bit for bit.  Intermediates stay on chip but for what
// five levels a thread spill: 28 to 68 bytes a lane.
//
// Measured (RiemannSolver3, last call, 79 levels, one MI355X; one thread per
// column -> levels spread): six C12 tiles 224 -> 46 us, six C51 193 -> 66 us,
// six C96 311 -> 242 us, six C128 628 -> 406 us, 96 C48 tiles with FP32
// inputs 1242 -> 1014 us.  One workgroup takes about 104 k cycles, of which
// the chains take 60 k; with two to a CU one's chains run beside the other's
// independent parts.  64 columns by 10 levels (a whole wave per set, one
// workgroup per CU) measured 342 us on six C96 tiles.
#include <algorithm>
#include <cmath>

#include "common.hpp"
#include "divide.hpp"
#include "riem_column.hpp"
#include "timing.hpp"

namespace fv3 {

constexpr int RC = 32;      // columns per workgroup (half a wave)

// The low (hi = false) or high half-wave's value in both halves.
__device__ __forceinline__ double half_bcast(double v, bool hi) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)u, up = (unsigned)(u >> 32);
  const auto a = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(up, up, false, false);
  return __builtin_bit_cast(double, hi ? ((unsigned long long)b[1] << 32) | a[1]
                                       : ((unsigned long long)b[0] << 32) | a[0]);
}

constexpr int kRiemMaxLevels = 128;

// C = true: RiemannSolverC (riem_solver_c.py:13-64); false: RiemannSolver3
// (riem_solver3.py:24-103).  The sim1 arithmetic (sim1_solver.py:11-101) is
// shared and evaluated in the stencils' order.
//
// Thread (x, y) holds column x & 31 and, as set 2 y + (x >> 5), the layers
// k0 .. k0 + LV - 1 of it (k0 = set LV); layers at and past nz compute on
// clamped loads and reach no store.  slot[] passes a chain's carried values
// from one wave to the next; xch[] a set's first or last level to its
// neighbours.  At most five column arrays are alive at a time (2 LV registers
// each), so that two workgroups fit a CU: gm, gr and w are formed or loaded a
// second time instead of kept.
template <bool C, typename S, int LV, int NW>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(LV <= 5 ? 4 : 2)))
    riem_kernel(Dom d, Box2 bx, Riem3Opts o, double dt, double p_fac, RiemFields<S> f) {
  extern __shared__ double lds[];
  const int col = threadIdx.x & (RC - 1), half = threadIdx.x >> 5, nwave = blockDim.y;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int set = 2 * wave + half;
  double* const slot = lds;                 // 2 x 2 x RC
  double* const bot = slot + 4 * RC;        // pp at the surface
  double* const xch = bot + RC;             // 2 x (2 nwave + 2) x RC
  // pm waits in LDS until the end (each thread its own entries)
  double* const pm = xch + 2 * (2 * nwave + 2) * RC + set * LV * RC + col;
  auto sl = [&](int v, int w) -> double& { return slot[(v * 2 + (w & 1)) * RC + col]; };
  auto xc = [&](int v, int w) -> double& { return xch[(v * (2 * nwave + 2) + w + 1) * RC + col]; };

  const int ncol = bx.nib * bx.njb;
  const int n0 = (int)blockIdx.x * RC + col;
  const bool keep = n0 < ncol;  // columns past the box: clamped loads, no stores
  const int n = keep ? n0 : ncol - 1;
  const int i = bx.i1 + n % bx.nib, j = bx.j1 + n / bx.nib;
  const int t = blockIdx.y;
  const int64_t c2 = (int64_t)t * d.st2 + (int64_t)j * d.sj2 + i;
  const int nz = d.nk - 1;
  const int k0 = set * LV;
  // fields are addressed as a tile's uniform base plus the lane's offset in
  // elements, layers past the bottom clamped to it
  const int64_t tb = (int64_t)t * d.st;
  typedef uint32_t OFF;
  const OFF sk = (OFF)d.sk;
  const OFF c = (OFF)j * (OFF)d.sj + (OFF)i;
  auto ptr = [tb](auto* base, OFF e) {
    typedef decltype(base) P;
    return (P)((const char*)(base + tb) + (size_t)(OFF)(e * (OFF)sizeof(*base)));
  };
  auto lay = [&](int u) -> OFF { return c + (OFF)min(k0 + u, nz - 1) * sk; };
  auto itf = [&](int u) -> OFF { return c + (OFF)min(k0 + u, nz) * sk; };
  const double ptop = o.ptop;
  const double t1g = 2.0 * dt * dt;
  const double rdt = 1.0 / dt;
  const double rgrav = o.rgrav;
  auto dm_of = [rgrav](double dpk) -> double {
    if constexpr (C)
      return dpk / kGrav;
    else
      return dpk * rgrav;
  };
  // The waves exchange through LDS only, so a barrier waits for LDS alone
  // (__syncthreads would also wait for every load and store in flight).
  auto barrier = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  // A chain up (down) the column: the waves take turns, each its lower (upper)
  // set first, on the values v0, v1 the one before left.  Every wave passes
  // nwave barriers.
  auto chain = [&](bool up, double v0, double v1, auto body) {
    const int turn = up ? wave : nwave - 1 - wave;
    for (int w = 0; w < turn; ++w) barrier();
    if (turn > 0) {
      v0 = sl(0, turn);
      v1 = sl(1, turn);
    }
    if (half == (up ? 0 : 1)) body(v0, v1);
    v0 = half_bcast(v0, !up);
    v1 = half_bcast(v1, !up);
    if (half == (up ? 1 : 0)) {
      body(v0, v1);
      sl(0, turn + 1) = v0;
      sl(1, turn + 1) = v1;
    }
    for (int w = turn; w < nwave; ++w) barrier();
  };

  // ---- inputs, then chain A (up): the interface sums pem (of dp) and peg
  // (of the dry part); entry u holds the interface below layer k0 + u
  double dm[LV], pem[LV], dz[LV], g[LV], p[LV];
  double pem0 = ptop, peg0 = ptop;  // the set's top interface
#pragma unroll
  for (int u = 0; u < LV; ++u) {
    const double dp = *ptr(f.dp, lay(u)), qc = *ptr(f.qc, lay(u));
    const bool in = k0 + u < nz;  // layers past the bottom add nothing
    pem[u] = in ? dp : 0.0;
    g[u] = in ? dp * (1.0 - qc) : 0.0;
    dm[u] = dm_of(dp);
  }
  {
    double z = *ptr(f.z, itf(0));
#pragma unroll
    for (int u = 0; u < LV; ++u) {
      const double zn = *ptr(f.z, itf(u + 1));
      dz[u] = zn - z;
      z = zn;
    }
  }
  chain(true, ptop, ptop, [&](double& a, double& b) {
    pem0 = a;
    peg0 = b;
#pragma unroll
    for (int u = 0; u < LV; ++u) {
      a = a + pem[u];
      b = b + g[u];
      pem[u] = a;
      g[u] = b;
    }
  });
  // ---- precompute: pm and pe = exp(gm log(-dm/dz Rd pt)) - pm (into p)
  {
    double pg = peg0, lg = 0.0;
    if constexpr (!C) lg = k0 == 0 ? o.peln1 : log(pg);
#pragma unroll
    for (int u = 0; u < LV; ++u) {
      double pmk;
      if constexpr (C) {
        pmk = (g[u] - pg) / log(g[u] / pg);
      } else {
        const double ln = log(g[u]);
        pmk = (g[u] - pg) / (ln - lg);
        lg = ln;
      }
      pg = g[u];
      pm[u * RC] = pmk;
      const double pt = *ptr(f.pt, lay(u)), cp = *ptr(f.cappa, lay(u));
      p[u] = exp(gm_of(cp) * log(-dm[u] / dz[u] * kRdgas * pt)) - pmk;
    }
  }
  xc(0, set) = dm[0];
  xc(1, set) = p[0];
  barrier();
  // ---- chain B (up): pp forward elimination (sim1_solver.py:42-56) of
  // bb = 2 (1 + gr), dd = 3 (pe_k + gr pe_k+1); gr (in g) becomes gam, dd (in
  // p) pp of the layer's top interface
  double ppn = 0.0;  // pp at the set's bottom interface
  {
    const double dmn = xc(0, set + 1), pen = xc(1, set + 1);
#pragma unroll
    for (int u = 0; u < LV; ++u) {
      const bool last = k0 + u >= nz - 1;
      const double dm1 = u + 1 < LV ? dm[u + 1 < LV ? u + 1 : u] : dmn;
      const double pe1 = u + 1 < LV ? p[u + 1 < LV ? u + 1 : u] : pen;
      g[u] = last ? 0.0 : dm[u] / dm1;
      p[u] = last ? 3.0 * p[u] : 3.0 * (p[u] + g[u] * pe1);
    }
    chain(true, 0.0, 0.0, [&](double& pk, double& gk) {
#pragma unroll
      for (int u = 0; u < LV; ++u) {
        const double gr = g[u], dd = p[u];
        g[u] = gk;
        p[u] = pk;
        const Divisor<double> r(2.0 * (1.0 + gr) - gk);  // gr = 0 in the bottom layer
        pk = r.quot(dd - pk);
        gk = r.quot(gr);  // the next layer's gam = gr_k / bet_k
        if (k0 + u == nz - 1) bot[col] = pk;
      }
    });
    // layers past the bottom hand pp of interface nz up unchanged
#pragma unroll
    for (int u = 0; u < LV; ++u) {
      if (k0 + u >= nz) {
        p[u] = 0.0;
        g[u] = -1.0;
      }
    }
  }
  // ---- chain C (down): pp back substitution; from the surface
  chain(false, bot[col], 0.0, [&](double& pk, double&) {
    ppn = pk;  // pp at the bottom interface (nz, where the layers end)
#pragma unroll
    for (int u = LV - 1; u >= 0; --u) {
      p[u] = p[u] - g[u] * pk;  // gam = 0 in layer 0
      pk = p[u];
    }
  });
  // ---- aa of layers 1 .. nz - 1 (sim1_solver.py:57-66, into g) and the
  // surface's p1, then the right-hand sides of w (into p)
  double ab = 0.0;  // aa below the set's last layer
  {
    const double gml = gm_of(*ptr(f.cappa, lay(LV - 1)));
    xc(0, set) = gml;
    xc(1, set) = dz[LV - 1];
    barrier();
    double gm0 = xc(0, set - 1), dz0 = xc(1, set - 1);
    double pe0 = pem0;
    const double wsr = f.wsd[c2];
#pragma unroll
    for (int u = 0; u < LV; ++u) {
      const int k = k0 + u;
      const double gmk = u + 1 < LV ? gm_of(*ptr(f.cappa, lay(u))) : gml;
      const double pn = u + 1 < LV && k + 1 < nz ? p[u + 1 < LV ? u + 1 : u] : ppn;
      const double w1 = *ptr(f.w, lay(u));
      g[u] = k == 0 ? 0.0 : t1g * 0.5 * (gm0 + gmk) / (dz0 + dz[u]) * (pe0 + p[u]);
      const double rhs = k == 0 ? dm[u] * w1 + dt * pn : dm[u] * w1 + dt * (pn - p[u]);
      gm0 = gmk;
      dz0 = dz[u];
      pe0 = pem[u];
      if (k == nz - 1) {
        // dz of the bottom layer makes room for p1, which takes aa's place below it
        dz[u] = t1g * gmk / dz[u] * (pem[u] + pn);
        p[u] = rhs - dz[u] * wsr;
        ab = dz[u];
      } else {
        p[u] = rhs;
      }
    }
    barrier();
    xc(0, set) = g[0];
    barrier();
    if (k0 + LV < nz) ab = xc(0, set + 1);
  }
  // ---- chain D (up): w forward elimination; aa (in g) becomes the back
  // substitution's factor, the right-hand side (in p) w
  chain(true, 1.0, 0.0, [&](double& bet, double& wp) {
    // aa = 0 in layer 0: gam = 0, bet = dm - an there
#pragma unroll
    for (int u = 0; u < LV; ++u) {
      const double an = u + 1 < LV && k0 + u != nz - 1 ? g[u + 1 < LV ? u + 1 : u] : ab;
      const Divisor<double> r(bet);
      const double gam = r.quot(g[u]);
      bet = dm[u] - (g[u] + an + g[u] * gam);
      wp = (p[u] - g[u] * wp) / bet;
      p[u] = wp;
      g[u] = gam;
    }
  });
#pragma unroll
  for (int u = 0; u < LV; ++u)
    if (k0 + u >= nz) p[u] = g[u] = 0.0;
  // ---- chain E (down): w back substitution; carries gam_k+1 w_k+1
  chain(false, 0.0, 0.0, [&](double& gw, double&) {
#pragma unroll
    for (int u = LV - 1; u >= 0; --u) {
      p[u] = p[u] - gw;
      gw = g[u] * p[u];
    }
  });
  // ---- chain F (up): pe from the change of w (into p), of the interface
  // below
#pragma unroll
  for (int u = 0; u < LV; ++u) {
    const double w1 = *ptr(f.w, lay(u));
    const double wk = p[u];
    p[u] = k0 + u < nz ? dm[u] * (wk - w1) * rdt : 0.0;
    if constexpr (!C) {
      if (keep && k0 + u < nz) *ptr(f.w, lay(u)) = (S)wk;
    }
  }
  double pet = 0.0;  // the set's top interface
  chain(true, 0.0, 0.0, [&](double& a, double&) {
    pet = a;
#pragma unroll
    for (int u = 0; u < LV; ++u) {
      a = a + p[u];
      p[u] = a;
    }
  });
  // ---- finalize of the interface pressures
  if (keep) {
    if (set == 0) {
      if constexpr (C) {
        *ptr(f.pef, c) = ptop;
      } else {
        const double pk3k = o.use_logp ? o.peln1 : o.ptk;
        *ptr(f.pk3, c) = pk3k;
        *ptr(f.ppe, c) = o.beta < -0.1 ? 0.0 + ptop : 0.0;  // new pe is 0 at the top
        if (o.last_call) {
          *ptr(f.peln, c) = o.peln1;
          *ptr(f.pk, c) = pk3k;
          *ptr(f.pe, c) = ptop;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < LV; ++u) {
      if (k0 + u < nz) {
        const OFF ob = itf(u + 1);
        if constexpr (C) {
          *ptr(f.pef, ob) = p[u] + pem[u];
        } else {
          const double peln = log(pem[u]);
          const double pk3k = o.use_logp ? peln : exp(o.kappa * peln);
          *ptr(f.pk3, ob) = pk3k;
          *ptr(f.ppe, ob) = o.beta < -0.1 ? p[u] + pem[u] : p[u];
          if (o.last_call) {
            *ptr(f.peln, ob) = peln;
            *ptr(f.pk, ob) = pk3k;
            *ptr(f.pe, ob) = pem[u];
          }
        }
      }
    }
  }
  // ---- chain G (down): p1 (sim1_solver.py:90-96, into p), its own-level
  // part first; gr formed again
  xc(0, set) = p[0];
  xc(1, set) = dm[0];
  barrier();
  {
    const double pen = xc(0, set + 1), dmn = xc(1, set + 1);
    double pa = pet;
#pragma unroll
    for (int u = 0; u < LV; ++u) {
      const bool last = k0 + u >= nz - 1;
      const double pc = u + 1 < LV ? p[u + 1 < LV ? u + 1 : u] : pen;
      const double dm1 = u + 1 < LV ? dm[u + 1 < LV ? u + 1 : u] : dmn;
      const double pb = p[u];
      g[u] = last ? 0.0 : dm[u] / dm1;
      p[u] = last ? (pa + 2.0 * pb) * 1.0 / 3.0
                  : (pa + 2.0 * (1.0 + g[u]) * pb + g[u] * pc) * 1.0 / 3.0;
      // layers past the bottom hand up 0: their value times the bottom layer's
      // gr = 0 is NaN where pe is infinite
      if (k0 + u >= nz) p[u] = 0.0;
      pa = pb;
    }
  }
  chain(false, 0.0, 0.0, [&](double& a, double&) {
#pragma unroll
    for (int u = LV - 1; u >= 0; --u) {
      p[u] = p[u] - g[u] * a;  // gr = 0 in the bottom layer
      a = p[u];
    }
  });
  // ---- the dz update (sim1_solver.py:97-101), then chain H (down): the
  // height / geopotential integration from the surface
#pragma unroll
  for (int u = 0; u < LV; ++u) {
    const double pt = *ptr(f.pt, lay(u)), cp = *ptr(f.cappa, lay(u));
    const double pmk = pm[u * RC];
    const double maxp = p_fac * dm[u] > p[u] + pmk ? p_fac * pmk : p[u] + pmk;
    const double dzn = -dm[u] * kRdgas * pt * exp((cp - 1.0) * log(maxp));
    if constexpr (!C) {
      if (keep && k0 + u < nz) *ptr(f.delz, lay(u)) = dzn;
    }
    g[u] = k0 + u < nz ? (C ? dzn * kGrav : dzn) : 0.0;
  }
  const double surf = f.surf[c2];
  chain(false, surf, 0.0, [&](double& a, double&) {
#pragma unroll
    for (int u = LV - 1; u >= 0; --u) {
      a = a - g[u];
      g[u] = a;
    }
  });
  if (keep) {
    if (set == 0) *ptr(f.z, c + (OFF)nz * sk) = surf;
#pragma unroll
    for (int u = 0; u < LV; ++u)
      if (k0 + u < nz) *ptr(f.z, lay(u)) = g[u];
  }
}

template <int LV>
int riem_waves(int nk) {
  return (nk - 1 + 2 * LV - 1) / (2 * LV);
}
template <int LV>
size_t riem_lds_bytes(int nk) {
  const int nw = riem_waves<LV>(nk);
  return (size_t)(5 + 2 * (2 * nw + 2) + 2 * nw * LV) * RC * sizeof(double);
}

// every byte offset in a tile fits 32 bits
static bool riem_narrow(const fv3_domain* dom) {
  return ((int64_t)dom->nk * dom->sk) * (int64_t)sizeof(double) < (int64_t)1 << 32;
}

// Microseconds of a launch on `waves` waves of columns (64 each), by the forms
// below.  Measured over 3 .. 127 layers on 18 to 3840 waves, FP64 and FP32
// inputs; the estimates hold within about 15 %.
//
// One thread per column: 2.1 us a layer (RiemannSolver3 2.5) at the latency of
// its sweeps, more where memory bounds them, in rounds of the workgroups whose
// column array fits the LDS (1024 up to 80 interfaces, 512 from 106 on).
static double riem_column_us(int nz, int64_t waves, bool c, bool fp32) {
  const int64_t lds = ((int64_t)(nz + 1) * RW * 8 + 1279) / 1280 * 1280;  // as allocated
  const int64_t round = 256 * std::min<int64_t>(16, 160 * 1024 / lds);
  const bool small = c ? waves < 2000 : nz <= 40 && waves < 2000;
  const double rate = c ? (fp32 ? (small ? 2.75 : 2.8) : (small ? 3.05 : 3.1))
                        : (fp32 ? (small ? 3.5 : 4.1) : (small ? 3.9 : 4.6));
  auto layer = [&](int64_t w) {
    return w == 0 ? 0.0 : std::max((c ? 2.1 : 2.5) + 0.6e-3 * w, rate * 1e-3 * w);
  };
  double t = (waves / round) * layer(round) + layer(waves % round);
  if (waves > round && round <= 1024)
    t = std::max(t, (c ? 3.9 : fp32 ? 4.8 : 5.1) * 1e-3 * waves);
  return nz * t + 4.5;
}

// Levels over a workgroup, lv to a thread: up to four waves (two of lv 8) a
// latency and a time per wave of columns; more of them in rounds of the
// workgroups whose registers fit the chip (16 waves to a CU at lv 5, 8 at lv 8).
static double riem_levels_us(int lv, int nz, int64_t waves, bool c) {
  const int nw = (nz + 2 * lv - 1) / (2 * lv);
  if (nw > 8) return 1e30;
  static const double few5[5][3] = {{}, {14, 6, 18}, {25, 8, 38}, {33, 10, 66}, {41, 15, 91}};
  static const double few8[3][3] = {{}, {19, 6, 30}, {36, 12, 76}};
  if (nw <= (lv == 5 ? 4 : 2)) {
    const double* f = lv == 5 ? few5[nw] : few8[nw];
    return std::max(f[0], (f[1] + f[2] * 1e-3 * waves) * (c ? 1.0 : 1.1));
  }
  // alone, per round of RiemannSolverC, of RiemannSolver3
  static const double round5[4][3] = {{51, 65, 80}, {58, 57.5, 59}, {66, 62, 63}, {74, 64, 68}};
  static const double round8[6][3] = {{48, 44, 47}, {58, 53, 57}, {52, 53, 53},
                                      {60, 60, 60}, {68, 68, 67}, {76, 76, 75}};
  const double* r = lv == 5 ? round5[nw - 5] : round8[nw - 3];
  const int per_cu = (lv == 5 ? 16 : 8) / nw;
  const double rounds = 2.0 * waves / (256.0 * per_cu);
  if (rounds <= 1.0) return r[0];
  return c || per_cu == 1 ? (c ? r[1] : r[2]) * std::ceil(rounds) : r[2] * (rounds + 0.35);
}

// The form with the least time: one thread per column (0), or 5 or 8 levels a
// thread.  Few layers take the column form (RiemannSolverC on six C96 tiles, 4
// layers: 17 against 22 us), as do layer counts that fill the levels' waves
// badly on many columns (50 layers: 147 against 200 us) and those above 80,
// where 8 levels a thread leave one workgroup to a CU (100 layers on six C128
// tiles: 722 against 887 us).  Below half a workgroup a CU the levels' latency
// alone counts.  The rates are those of calls alone; inside the acoustic call,
// among a gigabyte of other fields, RiemannSolverC's column form, which reads its
// inputs in six sweeps, takes more (79 layers, six C96 tiles: 236 us alone and
// 285 us there, 5 levels a thread 258 and 259 us), hence kColumnInCall between
// the few layers that fit the caches and the many where 8 levels lose by more.
constexpr double kColumnInCall = 1.16;
static int riem_form(int nz, int64_t waves, bool c, bool fp32) {
  if (waves >= 100 && nz <= (waves < 500 ? 4 : fp32 ? 7 : 6)) return 0;
  if (waves <= 128) return nz <= 80 ? 5 : 8;
  const double t0 = riem_column_us(nz, waves, c, fp32) *
                    (c && nz > 16 && nz <= 80 ? kColumnInCall : 1.0);
  const double t5 = riem_levels_us(5, nz, waves, c), t8 = riem_levels_us(8, nz, waves, c);
  if (t0 <= t5 && t0 <= t8) return 0;
  return t5 <= t8 ? 5 : 8;
}

template <bool C, typename S, int LV, int NW>
void riem_launch_as(const fv3_domain* dom, hipStream_t s, const Dom& d, Box2 bx,
                    const Riem3Opts& o, double dt, double p_fac, const RiemFields<S>& f) {
  const dim3 grid((unsigned)((bx.nib * bx.njb + RC - 1) / RC), (unsigned)d.ntiles);
  hipLaunchKernelGGL((riem_kernel<C, S, LV, NW>), grid, dim3(64, riem_waves<LV>(dom->nk)),
                     riem_lds_bytes<LV>(dom->nk), s, d, bx, o, dt, p_fac, f);
}

template <bool C, typename S>
void riem_launch(const fv3_domain* dom, hipStream_t s, const Dom& d, Box2 bx, const Riem3Opts& o,
                 double dt, double p_fac, const RiemFields<S>& f) {
  const int64_t waves = ((int64_t)bx.nib * bx.njb + RW - 1) / RW * d.ntiles;
  // the level kernels' byte offsets in a tile are 32 bits wide
  const int form =
      riem_narrow(dom) ? riem_form(dom->nk - 1, waves, C, sizeof(S) == 4) : 0;
  if (form == 5) {
    riem_launch_as<C, S, 5, 8>(dom, s, d, bx, o, dt, p_fac, f);
  } else if (form == 8) {
    riem_launch_as<C, S, 8, 8>(dom, s, d, bx, o, dt, p_fac, f);
  } else {
    const dim3 grid((unsigned)(((int64_t)bx.nib * bx.njb + RW - 1) / RW), (unsigned)d.ntiles);
    hipLaunchKernelGGL((riem_column_kernel<C, S>), grid, dim3(RW),
                       (size_t)dom->nk * RW * sizeof(double), s, d, bx, o, dt, p_fac, f);
  }
}

static int check_riem(const fv3_domain* dom, const char* who, int i1, int i2, int j1, int j2,
                      int64_t slab) {
  int rc = check_domain(dom, who);
  if (rc) return rc;
  FV3_REQUIRE(dom->nk >= 4, FV3_E_ARG, "%s: need at least 4 levels", who);
  FV3_REQUIRE(dom->nk <= kRiemMaxLevels, FV3_E_UNSUPPORTED,
              "%s: at most %d interface levels (got %d)", who, kRiemMaxLevels, dom->nk);
  FV3_REQUIRE(i1 >= 0 && j1 >= 0 && i2 < dom->ni && j2 < dom->nj, FV3_E_ARG,
              "%s: box outside the storage", who);
  FV3_REQUIRE(slab >= (int64_t)(dom->ntiles - 1) * dom->st + dom->sk * dom->nk, FV3_E_ARG,
              "%s: workspace slab too small", who);
  return FV3_OK;
}

template <typename S>
int riem_solver_c(const fv3_domain* dom, double dt2, double ptop, double p_fac, const S* cappa,
                  const double* hs, const double* ws, const S* ptc, const S* q_con,
                  const S* delpc, double* gz, double* pef, const S* w3, double* work,
                  int64_t work_slab, void* stream) {
  const char* who = "fv3_riem_solver_c";
  if (!dom) {
    set_error("%s: domain is NULL", who);
    return FV3_E_ARG;
  }
  const int i1 = dom->isc - 1, i2 = dom->iec + 1, j1 = dom->jsc - 1, j2 = dom->jec + 1;
  int rc = check_riem(dom, who, i1, i2, j1, j2, work_slab);
  if (rc) return rc;
  FV3_REQUIRE(cappa && hs && ws && ptc && q_con && delpc && gz && pef && w3 && work, FV3_E_ARG,
              "%s: NULL pointer", who);
  if (dom->ntiles == 0) return FV3_OK;
  Box2 bx{i1, j1, i2 - i1 + 1, j2 - j1 + 1};
  Dom d = to_dom(dom);
  Riem3Opts o{};
  o.ptop = ptop;
  RiemFields<S> f{};
  f.cappa = cappa;
  f.qc = q_con;
  f.dp = delpc;
  f.pt = ptc;
  f.surf = hs;
  f.wsd = ws;
  f.z = gz;
  f.w = const_cast<S*>(w3);  // read only in this solver
  f.pef = pef;
  f.work = work;
  f.slab = work_slab;
  // cappa, ptc, q_con, delpc, gz, w3 read; gz, pef written (per cell-level)
  TimedLaunch timed("riem_c_kernel", as_stream(stream),
                    (4.0 * sizeof(S) + 4.0 * sizeof(double)) * bx.nib * bx.njb *
                        (double)dom->nk * d.ntiles);
  riem_launch<true, S>(dom, as_stream(stream), d, bx, o, dt2, p_fac, f);
  FV3_HIP_CHECK_LAUNCH(who);
  return FV3_OK;
}

template <typename S>
int riem_solver3(const fv3_domain* dom, int last_call, double dt, double ptop, double p_fac,
                 int use_logp, double beta, const S* cappa, const double* zs, const double* wsd,
                 double* delz, const S* q_con, const S* delp, const S* pt, double* zh, double* pe,
                 double* ppe, double* pk3, double* pk, double* peln, S* w, double* work,
                 int64_t work_slab, void* stream) {
  const char* who = "fv3_riem_solver3";
  if (!dom) {
    set_error("%s: domain is NULL", who);
    return FV3_E_ARG;
  }
  const int i1 = dom->isc, i2 = dom->iec, j1 = dom->jsc, j2 = dom->jec;
  int rc = check_riem(dom, who, i1, i2, j1, j2, work_slab);
  if (rc) return rc;
  FV3_REQUIRE(cappa && zs && wsd && delz && q_con && delp && pt && zh && pe && ppe && pk3 &&
                  pk && peln && w && work,
              FV3_E_ARG, "%s: NULL pointer", who);
  FV3_REQUIRE(ptop > 0.0, FV3_E_ARG, "%s: ptop must be positive", who);
  if (dom->ntiles == 0) return FV3_OK;
  Box2 bx{i1, j1, i2 - i1 + 1, j2 - j1 + 1};
  Riem3Opts o;
  o.last_call = last_call ? 1 : 0;
  o.use_logp = use_logp ? 1 : 0;
  o.beta = beta;
  o.dt = dt;
  o.ptop = ptop;
  o.p_fac = p_fac;
  o.peln1 = log(ptop);
  o.kappa = kRdgas / kCpAir;
  o.ptk = exp(o.kappa * o.peln1);
  o.rgrav = 1.0 / kGrav;
  Dom d = to_dom(dom);
  RiemFields<S> f{};
  f.cappa = cappa;
  f.qc = q_con;
  f.dp = delp;
  f.pt = pt;
  f.surf = zs;
  f.wsd = wsd;
  f.z = zh;
  f.w = w;
  f.delz = delz;
  f.pe = pe;
  f.ppe = ppe;
  f.pk3 = pk3;
  f.pk = pk;
  f.peln = peln;
  f.work = work;
  f.slab = work_slab;
  // cappa, q_con, delp, pt, zh, w read; zh, ppe, pk3, delz, w written, plus
  // pe, pk and peln on the last call (per cell-level)
  TimedLaunch timed("riem3_kernel", as_stream(stream),
                    ((5.0 * sizeof(S) + (6.0 + 3.0 * o.last_call) * sizeof(double))) * bx.nib * bx.njb *
                        (double)dom->nk * d.ntiles);
  riem_launch<false, S>(dom, as_stream(stream), d, bx, o, dt, p_fac, f);
  FV3_HIP_CHECK_LAUNCH(who);
  return FV3_OK;
}
}  // namespace fv3

extern "C" {

int32_t fv3_plan_riem(int32_t nz, int64_t waves, int32_t solver_c, int32_t fp32) {
  return fv3::riem_form(nz, waves, solver_c != 0, fp32 != 0);
}

int32_t fv3_riem_solver_c_f64(const fv3_domain* dom, double dt2, double ptop, double p_fac,
                              const double* cappa, const double* hs, const double* ws,
                              const double* ptc, const double* q_con, const double* delpc,
                              double* gz, double* pef, const double* w3, double* work,
                              int64_t work_slab, void* stream) {
  return fv3::riem_solver_c<double>(dom, dt2, ptop, p_fac, cappa, hs, ws, ptc, q_con, delpc, gz,
                                    pef, w3, work, work_slab, stream);
}

int32_t fv3_riem_solver_c_mixed(const fv3_domain* dom, double dt2, double ptop, double p_fac,
                                const float* cappa, const double* hs, const double* ws,
                                const float* ptc, const float* q_con, const float* delpc,
                                double* gz, double* pef, const float* w3, double* work,
                                int64_t work_slab, void* stream) {
  return fv3::riem_solver_c<float>(dom, dt2, ptop, p_fac, cappa, hs, ws, ptc, q_con, delpc, gz,
                                   pef, w3, work, work_slab, stream);
}

int32_t fv3_riem_solver3_f64(const fv3_domain* dom, int32_t last_call, double dt, double ptop,
                             double p_fac, int32_t use_logp, double beta, const double* cappa,
                             const double* zs, const double* wsd, double* delz,
                             const double* q_con, const double* delp, const double* pt,
                             double* zh, double* pe, double* ppe, double* pk3, double* pk,
                             double* peln, double* w, double* work, int64_t work_slab,
                             void* stream) {
  return fv3::riem_solver3<double>(dom, last_call, dt, ptop, p_fac, use_logp, beta, cappa, zs,
                                   wsd, delz, q_con, delp, pt, zh, pe, ppe, pk3, pk, peln, w,
                                   work, work_slab, stream);
}

int32_t fv3_riem_solver3_mixed(const fv3_domain* dom, int32_t last_call, double dt, double ptop,
                               double p_fac, int32_t use_logp, double beta, const float* cappa,
                               const double* zs, const double* wsd, double* delz,
                               const float* q_con, const float* delp, const float* pt,
                               double* zh, double* pe, double* ppe, double* pk3, double* pk,
                               double* peln, float* w, double* work, int64_t work_slab,
                               void* stream) {
  return fv3::riem_solver3<float>(dom, last_call, dt, ptop, p_fac, use_logp, beta, cappa, zs,
                                  wsd, delz, q_con, delp, pt, zh, pe, ppe, pk3, pk, peln, w,
                                  work, work_slab, stream);
}
}
