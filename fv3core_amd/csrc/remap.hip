// Vertical remap of one scalar: RemapProfile (cs_profile) + MapSingle
// (fv3core/stencils/remap_profile.py:119-638, map_single.py:12-173): the kernel,
// its launcher and the C entry points.
#include "common.hpp"
#include "divide.hpp"
#include "remap_profile.hpp"
#include "timing.hpp"

#include <algorithm>
#include <mutex>

namespace fv3 {

// Layers of the tallest column that map_layers_kernel takes.
constexpr int kMapMaxLayers = 128;

// The same remap with a column's layers spread over a workgroup.
//
// What bounds it: one thread per column runs 79 layers x four sweeps in
// series, with its intermediates in memory; a C96 tile has 144 waves of them
// for 1024 SIMDs, and even 1536 waves (a C128 cube) hide little of two
// dependent divisions per layer.  But only the two recurrences of the edge
// values pass from layer to layer: the limiter reads a fixed window, and the
// walk of a target layer can start at its own first source layer.  Here MC
// columns by sets of LV layers share a workgroup, 64 / MC sets to a wave; the
// column's values sit in LDS, the recurrences run as chains from set to set,
// and everything else runs for all layers at once.  Sums and recurrences keep
// the order of the sweeps, so the results are the column kernel's bit for bit.
//
// Measured (kord 9, FP64, one field; one thread per column -> this kernel), 79
// layers: six C12 tiles 124 -> 18 us, six C51 159 -> 42, one C96 158 -> 29, six
// C96 221 -> 108, six C128 298 -> 178; 127 layers: six C12 198 -> 24, six C96
// 385 -> 254.  What bounds it now: the chains' latency at three waves a SIMD,
// which the five LDS arrays allow.
//
// planes: layer means; source interfaces; edge values, then a4_2; a4_3; a4_4.
// Layers at and past km compute on clamped values and reach no store.
template <typename T, int LV, int MC>
__global__ void __launch_bounds__(256)
    map_layers_kernel(Dom d, RemapArgs a, T* __restrict__ q1, const T* __restrict__ pe1,
                      const T* __restrict__ pe2, const T* __restrict__ qs) {
  extern __shared__ double lds_raw[];
  constexpr int SPW = 64 / MC;  // sets in a wave
  const int lane = threadIdx.x, col = lane & (MC - 1), sub = lane / MC;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.y), nwave = blockDim.y;
  const int km = a.km, k0 = (wave * SPW + sub) * LV;
  const int rows = nwave * SPW * LV + 1;
  T* const slot = reinterpret_cast<T*>(lds_raw);  // 2 x 2 x MC: a chain's carried values
  T* const bot = slot + 4 * MC;                   // the lowest edge value
  int* const odd = reinterpret_cast<int*>(bot + MC);  // columns with an unordered interface
  T* const PQ = bot + 2 * MC + col;
  T* const PP = PQ + rows * MC;
  T* const PE = PP + rows * MC;
  T* const PA3 = PE + rows * MC;
  T* const PA4 = PA3 + rows * MC;
  auto sl = [&](int v, int w) -> T& { return slot[(v * 2 + (w & 1)) * MC + col]; };
  // the waves exchange through LDS only: a barrier need not wait for loads and
  // stores in flight
  auto barrier = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  // A chain up (down) the column: the sets take turns on the values v0, v1 the
  // one before left.  Every wave passes nwave barriers.
  auto chain = [&](bool up, T v0, T v1, auto body) {
    const int turn = up ? wave : nwave - 1 - wave;
    for (int w = 0; w < turn; ++w) barrier();
    if (turn > 0) {
      v0 = sl(0, turn);
      v1 = sl(1, turn);
    }
#pragma unroll
    for (int h = 0; h < SPW; ++h) {
      const int s = up ? h : SPW - 1 - h;
      if (sub == s) body(v0, v1);
      if (h + 1 < SPW) {
        v0 = __shfl(v0, s * MC + col);
        v1 = __shfl(v1, s * MC + col);
      } else if (sub == s) {
        sl(0, turn + 1) = v0;
        sl(1, turn + 1) = v1;
      }
    }
    for (int w = turn; w < nwave; ++w) barrier();
  };

  const int ncol = a.ni_box * a.nj_box;
  const int n0 = (int)blockIdx.x * MC + col;
  const bool keep = n0 < ncol;  // columns past the box: clamped loads, no stores
  const int n = keep ? n0 : ncol - 1;
  const int i = a.i1 + n % a.ni_box, j = a.j1 + n / a.ni_box;
  const int t = blockIdx.y;
  const int64_t c = (int64_t)t * d.st + (int64_t)j * d.sj + i;
  const T* const P2 = pe2 + c;
  const int64_t sk = d.sk;

  // ---- inputs
  T p2[LV + 1];
  {
    T q[LV], p[LV + 1];
#pragma unroll
    for (int u = 0; u < LV; ++u) q[u] = q1[c + min(k0 + u, km - 1) * sk];
#pragma unroll
    for (int u = 0; u <= LV; ++u) p[u] = pe1[c + min(k0 + u, km) * sk];
#pragma unroll
    for (int u = 0; u <= LV; ++u) p2[u] = P2[min(k0 + u, km) * sk];
    if (k0 == 0) odd[col] = 0;
#pragma unroll
    for (int u = 0; u < LV; ++u) {
      PQ[(k0 + u) * MC] = q[u];
      PP[(k0 + u) * MC] = p[u];
    }
    if (k0 + LV == rows - 1) PP[(rows - 1) * MC] = p[LV];
    barrier();
#pragma unroll
    for (int u = 0; u < LV; ++u)
      if (!(p[u] <= p[u + 1] && p2[u] <= p2[u + 1])) odd[col] = 1;
  }

  // ---- (1) set_initial_vals: forward elimination, in every layer
  // bet = s - gam, ev = (r - ev) / bet, gam = g / bet with the carried ev and
  // gam; r, g become ev and gam
  T r[LV], g[LV];
  {
    T s[LV];
    const int kp = max(k0 - 1, 0);
    T q_up = PQ[kp * MC], p_up = PP[k0 * MC];
    T dp_up = p_up - PP[kp * MC];
#pragma unroll
    for (int u = 0; u < LV; ++u) {
      const int k = k0 + u;
      const T q = PQ[k * MC], pn = PP[(k + 1) * MC];
      const T dp = pn - p_up;
      const T d4 = dp_up / dp;
      s[u] = T(2) + d4 + d4;
      g[u] = d4;
      if (a.iv == -2) {
        r[u] = T(3) * (q_up + q);
        if (k == km - 1) {
          const T qsv = qs ? qs[(int64_t)t * d.st2 + (int64_t)j * d.sj2 + i] : T(0);
          r[u] = r[u] - d4 * qsv;
        }
        if (k == 0) {  // ev = 1.5 q, gam = 0.5
          r[u] = T(3) * q;
          s[u] = T(2);
          g[u] = T(1);
        }
      } else {
        r[u] = T(3) * (q_up + d4 * q);
        if (k == 0) {
          const T gr = (PP[2 * MC] - pn) / dp;
          s[u] = gr * (gr + T(0.5));
          r[u] = (gr + gr) * (gr + T(1)) * q + PQ[MC];
          g[u] = T(1) + gr * (gr + T(1.5));
        }
      }
      q_up = q;
      p_up = pn;
      dp_up = dp;
    }
    chain(true, T(0), T(0), [&](T& ev, T& gam) {
#pragma unroll
      for (int u = 0; u < LV; ++u) {
        const T bet = s[u] - gam;
        const Divisor<T> by(bet);
        ev = by.quot(r[u] - ev);
        gam = by.quot(g[u]);
        r[u] = ev;
        g[u] = gam;
      }
    });
  }
  // the lowest edge value (iv = -2: given, and not part of the recurrence)
#pragma unroll
  for (int u = 0; u < LV; ++u) {
    if (k0 + u == km - 1) {
      if (a.iv == -2) {
        bot[col] = T(0);
        PE[km * MC] = qs ? qs[(int64_t)t * d.st2 + (int64_t)j * d.sj2 + i] : T(0);
      } else {
        const T pm = PP[(km - 1) * MC];
        const T d4 = (pm - PP[(km - 2) * MC]) / (PP[km * MC] - pm);
        const T a_bot = T(1) + d4 * (d4 + T(1.5));
        const T e = (T(2) * d4 * (d4 + T(1)) * PQ[(km - 1) * MC] + PQ[(km - 2) * MC] -
                     a_bot * r[u]) /
                    (d4 * (d4 + T(0.5)) - a_bot * g[u]);
        bot[col] = e;
        PE[km * MC] = e;
      }
      if (a.iv == -2) g[u] = T(0);
    } else if (k0 + u >= km) {  // layers past the bottom hand the value up unchanged
      r[u] = T(0);
      g[u] = T(-1);
    }
  }
  barrier();
  // ---- (2) back substitution
  chain(false, bot[col], T(0), [&](T& ev, T&) {
#pragma unroll
    for (int u = LV - 1; u >= 0; --u) {
      ev = r[u] - g[u] * ev;
      r[u] = ev;
    }
  });
#pragma unroll
  for (int u = 0; u < LV; ++u)
    if (k0 + u < km) PE[(k0 + u) * MC] = r[u];
  barrier();

  // ---- (3) limiter steps, from two layers above the set's first
  {
    const int s0 = k0 - 2, sf = max(s0, 0);
    RemapLimiter<T> lim(a.kord, a.iv, km, a.qmin, PQ[sf * MC], PQ[min(sf + 1, km - 1) * MC], T(0));
    lim.am1 = PQ[max(s0 - 1, 0) * MC];
    RemapCoef<T> o[LV];
#pragma unroll
    for (int m = 0; m < LV + 3; ++m) {
      const int s = s0 + m;
      if (m == 2 && k0 == 0) {
        lim = RemapLimiter<T>(a.kord, a.iv, km, a.qmin, PQ[0], PQ[MC], PE[0]);
      }
      const T ap2 = PQ[min(max(s + 2, 0), km - 1) * MC];
      const T wp1 = PE[min(max(s + 1, 0), km) * MC];
      RemapCoef<T> v;
      lim.step(s, ap2, wp1, v);
      if (m >= 3) o[m < 3 ? 0 : m - 3] = v;
    }
    barrier();
#pragma unroll
    for (int u = 0; u < LV; ++u) {
      PE[(k0 + u) * MC] = o[u].a2;
      PA3[(k0 + u) * MC] = o[u].a3;
      PA4[(k0 + u) * MC] = o[u].a4;
    }
    barrier();
  }

  // ---- (4) lagrangian_contributions (map_single.py:19-66): target layer k's
  // overlap walk over source layers L, from the layer that holds its top
  {
    int L = 0;
    if (k0 > 0 && k0 < km) {
      if (odd[col] == 0) {
        // the first layer whose lower interface is not above p2[0]
        L = k0;
        while (L > 0 && PP[L * MC] >= p2[0]) --L;
        while (L < km - 1 && PP[(L + 1) * MC] < p2[0]) ++L;
      } else {
        // interfaces out of order: where the walk from the top arrives
        for (int k = 0; k < k0; ++k) {
          const T p2n = P2[(k + 1) * sk];
          if (p2n <= PP[(L + 1) * MC]) continue;
          if (L < km - 1) ++L;
          while (L < km - 1 && PP[(L + 1) * MC] < p2n) ++L;
        }
      }
    }
    T pL, pR, c1, c2, c3, c4;
    auto layer = [&]() __attribute__((always_inline)) {
      pL = PP[L * MC];
      pR = PP[(L + 1) * MC];
      c1 = PQ[L * MC];
      c2 = PE[L * MC];
      c3 = PA3[L * MC];
      c4 = PA4[L * MC];
    };
    layer();
#pragma unroll
    for (int u = 0; u < LV; ++u) {
      const int k = k0 + u;
      if (k < km) {
        const T p2k = p2[u], p2n = p2[u + 1];
        const T dpl = pR - pL;
        const T pl = (p2k - pL) / dpl;
        T out;
        if (p2n <= pR) {
          const T pr = (p2n - pL) / dpl;
          out = c2 + T(0.5) * (c4 + c3 - c2) * (pr + pl) -
                (c4 * T(1) / T(3)) * (pr * (pr + pl) + pl * pl);
        } else {
          T qsum = (pR - p2k) * (c2 + T(0.5) * (c4 + c3 - c2) * (T(1) + pl) -
                                 (c4 * T(1) / T(3)) * (T(1) + pl * (T(1) + pl)));
          // valid columns never pass the last layer; the bound only keeps a
          // malformed column inside its storage
          if (L < km - 1) {
            ++L;
            layer();
          }
          while (L < km - 1 && pR < p2n) {
            qsum += (pR - pL) * c1;
            ++L;
            layer();
          }
          const T dpx = p2n - pL;
          const T esl = dpx / (pR - pL);
          qsum += dpx * (c2 + T(0.5) * esl * (c3 - c2 + c4 * (T(1) - T(2.0 / 3.0) * esl)));
          out = qsum / (p2n - p2k);
        }
        if (keep) q1[c + (int64_t)k * sk] = out;
      }
    }
  }
}

template <typename T, int LV, int MC>
static int map_layers_launch(const Dom& d, const RemapArgs& a, T* q1, const T* pe1, const T* pe2,
                             const T* qs, void* stream, const char* who) {
  const int nwave = (a.km + LV * 64 / MC - 1) / (LV * 64 / MC);
  const int rows = nwave * (64 / MC) * LV + 1;
  const size_t lds = sizeof(T) * MC * (6 + 5 * (size_t)rows);  // at most 52 KB
  const dim3 grid((unsigned)(((int64_t)a.ni_box * a.nj_box + MC - 1) / MC), (unsigned)d.ntiles);
  hipLaunchKernelGGL((map_layers_kernel<T, LV, MC>), grid, dim3(64, nwave), lds, as_stream(stream), d,
                     a, q1, pe1, pe2, qs);
  FV3_HIP_CHECK_LAUNCH(who);
  return FV3_OK;
}

// The forms of the remap, which give the same bits: one thread per column in
// four sweeps or with the limiter fused into the walk, and layers spread over a
// workgroup (up to kMapMaxLayers).
enum MapForm { kMapSweeps = 0, kMapFused = 1, kMapLayers = 2 };

// The form with the least time on `waves` waves of columns (64 each).  Sets of 5
// layers and 16 columns up to 80 layers (10 layers: 259 us, 8 layers by 8
// columns: 287 us, 5 by 32: 245 us, against 178 us on six C128 tiles) take
// 0.030 us per wave of columns and 20 layers, 8 by 8 above them 0.272 us per
// wave, where 16 columns leave one workgroup to a CU (127 layers on six C96
// tiles: 322 against 254 us).  One thread per column takes 2.3 us a layer at its
// latency (less in launches of a few workgroups) and more once memory bounds it,
// so few layers on many columns are its: 10 layers on six C128 tiles 34 against
// 58 us, 81 layers 309 against 435 us.  Its fused form moves fewer bytes over a
// longer dependent chain: it wins where two waves a SIMD cover the chain, or
// where the nine column arrays of the sweeps (from 280 MB) do not fit the last-level
// cache (137 layers, six C128 tiles: 531 against 597 us; 96 C48 tiles 1204
// against 1698 us).  In FP32 the lines lie where its own times put them.  The
// rates are those of calls on data that the last one left in the caches; on cold
// data the four sweeps, which read a column four times, take 5 to 25 % more, the
// fused form up to 15 % and the spread form the same, hence the two factors (100
// layers, six C128 tiles, fused against spread: 383 and 436 us warm, 389 and 437
// cold; 32 layers on 96 C48 tiles in FP32 135 and 117, 151 and 118).
constexpr double kSweepsCold = 1.15, kFusedCold = 1.06;
static MapForm map_form(int km, int64_t waves, bool fp32) {
  const double w = (double)waves;
  const bool fused = waves >= 2 * kSimdsPerGpu ||
                     9.0 * 64.0 * w * km * (fp32 ? 4 : 8) >= 280e6;
  const MapForm column = fused ? kMapFused : kMapSweeps;
  if (km > kMapMaxLayers) return column;
  double layers, busy;
  if (km <= 80) {
    const double n = (km + 19) / 20;  // waves of a workgroup
    if (n == 1)
      layers = fp32 ? 8.0 + 0.0175 * w : 6.0 + 0.034 * w;
    else
      layers = fp32 ? 11.0 + 0.0175 * n * w : 12.0 + 0.030 * n * w;
    layers = std::max(fp32 ? 14.4 : 15.3, layers);
  } else {
    layers = fp32 ? 18.0 + 0.134 * w : 20.0 + 0.272 * w;
  }
  // up to 32 layers a column's arrays stay in the caches
  if (km <= 32)
    busy = fp32 ? 0.25 + 0.00108 * w : 0.21 + 0.00185 * w;
  else
    busy = fp32 ? 0.35 + 0.0013 * w : 0.7 + 0.0021 * w;
  const double lone = fp32 ? std::min(1.75, 1.35 + 0.008 * w) : std::min(2.3, 1.5 + 0.01 * w);
  const double cold = fused ? kFusedCold : kSweepsCold;
  return cold * (3.0 + km * std::max(lone, busy)) < layers ? column : kMapLayers;
}

template <typename T>
static int map_single_launch(const fv3_domain* dom, int kord, int iv, int i1, int i2, int j1,
                             int j2, T* q1, const T* pe1, const T* pe2, const T* qs, double qmin,
                             T* work, int64_t work_slab, void* stream) {
  const char* who = "fv3_map_single";
  int rc = check_domain(dom, who);
  if (rc) return rc;
  FV3_REQUIRE(q1 && pe1 && pe2 && work, FV3_E_ARG, "%s: NULL pointer", who);
  FV3_REQUIRE(kord <= 10, FV3_E_UNSUPPORTED, "%s: kord %d not implemented", who, kord);
  const int akord = kord < 0 ? -kord : kord;
  // The reference also accepts kord <= -11: for 10 < |kord| <= 16 it runs no
  // inner-level limiter and above 16 no constraints at all.  Those forms are
  // not built; they are rejected instead of running the kord-10 limiter.
  FV3_REQUIRE(akord <= 10, FV3_E_UNSUPPORTED,
              "%s: |kord| %d > 10 not implemented (only kord in -10..10)", who, akord);
  const int km = dom->nk;
  FV3_REQUIRE(km >= 6, FV3_E_ARG, "%s: need at least 6 layers (got %d)", who, km);
  FV3_REQUIRE(i1 >= 0 && j1 >= 0 && i2 < dom->ni && j2 < dom->nj && i2 >= i1 - 1 &&
                  j2 >= j1 - 1,
              FV3_E_ARG, "%s: box outside the storage", who);
  FV3_REQUIRE(work_slab >= (int64_t)(dom->ntiles - 1) * dom->st + dom->sk * (km + 1),
              FV3_E_ARG, "%s: workspace slab too small", who);
  const int nib = i2 - i1 + 1, njb = j2 - j1 + 1;
  if (nib <= 0 || njb <= 0 || dom->ntiles == 0) return FV3_OK;
  RemapArgs a{akord, iv, km, i1, j1, nib, njb, qmin, work_slab};
  Dom d = to_dom(dom);
  dim3 grid((unsigned)(((int64_t)nib * njb + 255) / 256), d.ntiles);
  // q1, pe1, pe2 read and q1 written once per cell-level of the box
  TimedLaunch timed("map_single_kernel", as_stream(stream),
                    4.0 * sizeof(T) * (double)nib * njb * km * d.ntiles);
  switch (map_form(km, ((int64_t)nib * njb + 63) / 64 * d.ntiles, sizeof(T) == 4)) {
    case kMapLayers:
      return km <= 80 ? map_layers_launch<T, 5, 16>(d, a, q1, pe1, pe2, qs, stream, who)
                      : map_layers_launch<T, 8, 8>(d, a, q1, pe1, pe2, qs, stream, who);
    case kMapFused:
      hipLaunchKernelGGL((map_single_kernel<T, true>), grid, dim3(256), 0, as_stream(stream), d, a,
                         q1, pe1, pe2, qs, work);
      break;
    default:
      hipLaunchKernelGGL((map_single_kernel<T, false>), grid, dim3(256), 0, as_stream(stream), d, a,
                         q1, pe1, pe2, qs, work);
  }
  FV3_HIP_CHECK_LAUNCH(who);
  return FV3_OK;
}

// ---- scratch of the entry point that allocates nothing
// The six column slabs of map_single_kernel live in one file-scope device
// array; every GPU the library runs on holds its own copy until the process
// ends.  Host code never passes the array's name to a kernel (on the host it
// is only a stand-in): it uses the device address hipGetSymbolAddress gives
// for the current device, kept per device.
constexpr size_t kNoAllocScratchBytes = size_t(96) << 20;
constexpr int kRemapSlabs = 6;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxDevices];

static int scratch_on_current_device(void** out, const char* who) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  FV3_REQUIRE(e == hipSuccess, FV3_E_HIP, "%s: hipGetDevice failed: %s", who,
              hipGetErrorString(e));
  FV3_REQUIRE(dev >= 0 && dev < kMaxDevices, FV3_E_HIP, "%s: device %d out of range", who, dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    FV3_REQUIRE(e == hipSuccess && p != nullptr, FV3_E_HIP,
                "%s: hipGetSymbolAddress(scratch) failed on device %d: %s", who, dev,
                hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return FV3_OK;
}

static int map_single_noalloc(const fv3_domain* dom, int kord, int iv, int i1, int i2, int j1,
                              int j2, double* q1, const double* pe1, const double* pe2,
                              const double* qs, double qmin, void* stream) {
  const char* who = "fv3_map_single_noalloc_f64";
  int rc = check_domain(dom, who);
  if (rc) return rc;
  FV3_REQUIRE(dom->st >= 0, FV3_E_ARG, "%s: negative tile stride", who);
  const int64_t tiles_before = dom->ntiles > 0 ? dom->ntiles - 1 : 0;
  // slab length in doubles, rounded to 256 bytes so every slab stays aligned
  const int64_t slab = (tiles_before * dom->st + dom->sk * (int64_t)(dom->nk + 1) + 31) / 32 * 32;
  const int64_t max_slab = (int64_t)(kNoAllocScratchBytes / sizeof(double) / kRemapSlabs);
  FV3_REQUIRE(slab <= max_slab, FV3_E_ARG,
              "%s: the columns need %lld bytes of scratch (6 slabs of %lld doubles), above the "
              "%zu-byte maximum",
              who, (long long)(slab * kRemapSlabs * (int64_t)sizeof(double)), (long long)slab,
              kNoAllocScratchBytes);
  void* p = nullptr;
  rc = scratch_on_current_device(&p, who);
  if (rc) return rc;
  return map_single_launch<double>(dom, kord, iv, i1, i2, j1, j2, q1, pe1, pe2, qs, qmin,
                                   static_cast<double*>(p), slab, stream);
}

}  // namespace fv3

extern "C" {

int32_t fv3_plan_map_single(int32_t km, int64_t waves, int32_t fp32) {
  return fv3::map_form(km, waves, fp32 != 0);
}

int32_t fv3_map_single_noalloc_f64(const fv3_domain* d, int32_t kord, int32_t mode, int32_t i1,
                                   int32_t i2, int32_t j1, int32_t j2, double* q1,
                                   const double* pe1, const double* pe2, const double* qs,
                                   double qmin, void* stream) {
  return fv3::map_single_noalloc(d, kord, mode, i1, i2, j1, j2, q1, pe1, pe2, qs, qmin, stream);
}

int32_t fv3_map_single_f64(const fv3_domain* d, int32_t kord, int32_t mode, int32_t i1,
                           int32_t i2, int32_t j1, int32_t j2, double* q1, const double* pe1,
                           const double* pe2, const double* qs, double qmin, double* work,
                           int64_t work_slab, void* stream) {
  return fv3::map_single_launch<double>(d, kord, mode, i1, i2, j1, j2, q1, pe1, pe2, qs, qmin,
                                        work, work_slab, stream);
}

int32_t fv3_map_single_f32(const fv3_domain* d, int32_t kord, int32_t mode, int32_t i1,
                           int32_t i2, int32_t j1, int32_t j2, float* q1, const float* pe1,
                           const float* pe2, const float* qs, double qmin, float* work,
                           int64_t work_slab, void* stream) {
  return fv3::map_single_launch<float>(d, kord, mode, i1, i2, j1, j2, q1, pe1, pe2, qs, qmin,
                                       work, work_slab, stream);
}
}
