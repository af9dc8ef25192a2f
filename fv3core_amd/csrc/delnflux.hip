// The stand-alone del-n fluxes (DelnFlux / DelnFluxNoSG): added to, or stored
// as, the caller's fluxes.
#include "delnflux.hpp"

#include <cmath>

namespace fv3 {

int strip_segment_rows(int rows, int64_t planes, const StripCost& cost) {
  int best = 0;
  double least = 0.0;
  for (int nb = 1; nb <= rows; ++nb) {
    const int seg = (rows + nb - 1) / nb;
    const double w = (double)planes * ((rows + seg - 1) / seg) / kSimdsPerGpu;
    if (w > cost.free && seg > cost.most) continue;
    const double n = cost.whole ? std::ceil(w) : w;
    const double step = w <= 3.0 ? cost.lone + cost.wave * n : cost.lone3 + cost.wave3 * n;
    const double t = step * (seg + cost.extra + cost.lead);
    if (best == 0 || t < least) {
      best = seg;
      least = t;
    }
    if (seg <= cost.least) break;
  }
  return best;
}

// fx, fy of an interface from its del-n flux f2: fx + f2 (ADD), fx + 0.5 damp
// (mass(i-1) + mass(i)) f2 (MASS) or f2 (STORE, STORE_MASS).
template <typename T>
struct DelnFluxEpilogue {
  T *fx, *fy;
  const T* mass;
  int mode;
  T dk;
  int64_t sj;

  struct In {
    T fx, fy, m, mw, ms;
  };
  __device__ __forceinline__ void plane(const Dom& d, int, T dk_, int64_t off3, int64_t) {
    fx += off3;
    fy += off3;
    mass = mass ? mass + off3 : nullptr;
    dk = dk_;
    sj = d.sj;
  }
  template <typename C>
  __device__ __forceinline__ In load(const C& c, int j) const {
    In n{};
    if (mode == FV3_DELN_ADD || mode == FV3_DELN_MASS) {
      n.fx = c.f(fx, j);
      n.fy = c.f(fy, j);
    }
    if (mode == FV3_DELN_MASS) {
      n.m = c.f(mass, j);
      n.mw = c.f(mass, j, -1);
      n.ms = c.f(mass, j - 1);
    }
    return n;
  }
  __device__ __forceinline__ T flux(T old, T m0, T m1, T f2) const {
    if (mode == FV3_DELN_ADD) return old + f2;
    if (mode == FV3_DELN_MASS) return old + T(0.5) * dk * (m0 + m1) * f2;
    return f2;
  }
  __device__ __forceinline__ void apply(const In& n, int i, int j, T f0, T, T g0, T, bool fxo,
                                        bool fyo, bool) const {
    const int64_t row = (int64_t)j * sj;
    if (fxo) (fx + row)[i] = flux(n.fx, n.mw, n.m, f0);
    if (fyo) (fy + row)[i] = flux(n.fy, n.ms, n.m, g0);
  }
};

template <typename T>
static int delnflux_launch(const fv3_domain* dom, int mode, const int32_t* nord4, const T* q,
                           const T* mass, const T* damp, const T* del6_u, const T* del6_v,
                           const T* rarea, T* fx, T* fy, void* stream) {
  const char* who = "fv3_delnflux";
  int rc = check_domain(dom, who);
  if (rc) return rc;
  FV3_REQUIRE(nord4 && q && damp && del6_u && del6_v && rarea && fx && fy, FV3_E_ARG,
              "%s: required pointer is NULL", who);
  FV3_REQUIRE(mode >= 0 && mode <= 3, FV3_E_ARG, "%s: bad mode %d", who, mode);
  FV3_REQUIRE(mode != FV3_DELN_MASS || mass, FV3_E_ARG, "%s: mass is required", who);
  DelnFluxEpilogue<T> epi{};
  epi.fx = fx;
  epi.fy = fy;
  epi.mass = mass;
  epi.mode = mode;
  const int use_damp = mode == FV3_DELN_ADD || mode == FV3_DELN_STORE;
  // q read, fx / fy read and written (per cell-level of the compute domain)
  const double bytes = 5.0 * sizeof(T) * (double)(dom->iec - dom->isc + 1) *
                       (dom->jec - dom->jsc + 1) * dom->nk * dom->ntiles;
  return deln_launch<T>(dom, nord4, use_damp, q, damp, del6_u, del6_v, rarea, epi, bytes, stream,
                        who);
}

}  // namespace fv3

extern "C" {

int32_t fv3_plan_delnflux_rows(int32_t rows, int64_t planes, int32_t fp32, int32_t most) {
  fv3::StripCost cost = fv3::deln_cost(fp32 != 0);
  if (most > 0) cost.most = most;
  return fv3::strip_segment_rows(rows, planes, cost);
}

int32_t fv3_delnflux_f64(const fv3_domain* d, int32_t mode, const int32_t nord4[4],
                         const double* q, const double* mass, const double* damp,
                         const double* del6_u, const double* del6_v, const double* rarea,
                         double* fx, double* fy, void* stream) {
  return fv3::delnflux_launch<double>(d, mode, nord4, q, mass, damp, del6_u, del6_v, rarea,
                                      fx, fy, stream);
}

int32_t fv3_delnflux_f32(const fv3_domain* d, int32_t mode, const int32_t nord4[4],
                         const float* q, const float* mass, const float* damp,
                         const float* del6_u, const float* del6_v, const float* rarea,
                         float* fx, float* fy, void* stream) {
  return fv3::delnflux_launch<float>(d, mode, nord4, q, mass, damp, del6_u, del6_v, rarea, fx,
                                     fy, stream);
}
}
