// Building blocks of the wave-strip kernels: one wave of 64 lanes owns a strip
// of columns and marches up its rows, neighbours across i by lane shifts.
#pragma once

#include <algorithm>

#include "common.hpp"

namespace fv3 {

// Whole-wave shifts by one lane with DPP: wave_shr:1 (lane L reads lane
// L - 1) and wave_shl:1 (lane L reads lane L + 1); the lane without a source
// receives 0.  They are register moves on the VALU, without the LDS round
// trip of a general lane permute.
constexpr int kWaveShr1 = 0x138;
constexpr int kWaveShl1 = 0x130;

template <int CTRL>
__device__ __forceinline__ int dpp32(int v) {
  return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, true);
}
template <int CTRL, typename T>
__device__ __forceinline__ T dpp_shift(T v) {
  if constexpr (sizeof(T) == 8) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)dpp32<CTRL>((int)(unsigned)u);
    const unsigned hi = (unsigned)dpp32<CTRL>((int)(unsigned)(u >> 32));
    return __builtin_bit_cast(T, ((unsigned long long)hi << 32) | lo);
  } else if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(T, dpp32<CTRL>(__builtin_bit_cast(int, v)));
  } else {
    return (T)dpp32<CTRL>((int)v);
  }
}
template <typename T>
__device__ __forceinline__ T lane_dn(T v, int d) {  // value of lane + d
  for (int n = 0; n < d; ++n) v = dpp_shift<kWaveShl1>(v);
  return v;
}
template <typename T>
__device__ __forceinline__ T lane_up(T v, int d) {  // value of lane - d
  for (int n = 0; n < d; ++n) v = dpp_shift<kWaveShr1>(v);
  return v;
}

// One lane's column of a strip.  Loads read rows and columns clamped into the
// storage, unconditionally; what lanes or rows outside the storage load feeds
// nothing that is kept.  The column offset is passed through an empty asm at
// each use so that the compiler keeps (uniform row address) + (32-bit lane
// offset), the scalar-base form of the global loads, instead of hoisting
// 64-bit per-lane pointers.
template <typename T>
struct StripColumn {
  int i, ni, nj;
  uint32_t off0, offm, offp;  // byte offsets of columns i, i - 1, i + 1
  int64_t sj, sj2;
  __device__ __forceinline__ StripColumn(const Dom& d, int i_)
      : i(i_), ni(d.ni), nj(d.nj), sj(d.sj), sj2(d.sj2) {
    auto at = [&](int c) { return (uint32_t)min(max(c, 0), d.ni - 1) * (uint32_t)sizeof(T); };
    off0 = at(i);
    offm = at(i - 1);
    offp = at(i + 1);
  }
  __device__ __forceinline__ static T get(const T* __restrict__ p, int64_t row, uint32_t off) {
    asm volatile("" : "+v"(off));
    return *(const T*)((const char*)(p + row) + off);
  }
  __device__ __forceinline__ int64_t row(int j, int64_t stride) const {
    return (int64_t)__builtin_amdgcn_readfirstlane(min(max(j, 0), nj - 1)) * stride;
  }
  // fields (row stride sj) and IJ metric terms (sj2) at row j, column i + di
  __device__ __forceinline__ T f(const T* __restrict__ p, int j, int di = 0) const {
    return get(p, row(j, sj), di == 0 ? off0 : di < 0 ? offm : offp);
  }
  __device__ __forceinline__ T m(const T* __restrict__ p, int j, int di = 0) const {
    return get(p, row(j, sj2), di == 0 ? off0 : di < 0 ? offm : offp);
  }
  // Stores v to row j of field p where keep holds (in a row and column of the
  // storage), without a branch: a buffer store whose range is the row drops the
  // offsets past it.  Loads and stores are counted by one counter in order, so
  // behind a branch the next wait for loads would also wait for every store
  // that might have been issued.
  __device__ __forceinline__ void store(T* p, int j, T v, bool keep) const {
    const uint64_t a = (uint64_t)(p + row(j, sj));
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a),
                   hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((uint64_t)hi << 32 | lo), 0, ni * (int)sizeof(T), 0x00027000);
    const uint32_t off = keep ? (uint32_t)i * (uint32_t)sizeof(T) : 0x80000000u;
    if constexpr (sizeof(T) == 8) {
      typedef uint32_t Pair __attribute__((ext_vector_type(2)));
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(Pair, v), rsrc, off, 0, 0);
    } else {
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), rsrc, off, 0, 0);
    }
  }
};

// Runs step(row, cur, next) for rows r0 .. r1, where cur holds the row's loads
// and step starts those of row + 1 into next.  Two rows per pass, with the
// buffers in turn: copying next to cur would wait for the loads just started.
template <typename ROW, typename F>
__device__ __forceinline__ void strip_march(int r0, int r1, ROW a, F step) {
  ROW b;
  for (int r = r0;;) {
    step(r, a, b);
    if (++r > r1) return;
    step(r, b, a);
    if (++r > r1) return;
  }
}

// How a launch is cut: columns from i0 in strips of `width` (the lanes left of
// a wave's 64 once its neighbours are taken off), rows j0 .. j1 in segments.
struct StripPlan {
  int i0, j0, j1, width, nbi, nbj, seg;
};

// Runs body(d, i, j, rows, k, t) for every strip (first column i), segment
// (first row j), level and tile, one wave each, NW waves to a workgroup.
template <int NW, typename F>
__global__ void __launch_bounds__(64 * NW) strip_kernel(Dom d, StripPlan p, F body) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int per_plane = p.nbi * p.nbj, total = per_plane * d.nk * d.ntiles;
  const int unit = xcd_logical_block(blockIdx.x, (total + NW - 1) / NW) * NW + wave;
  if (unit >= total) return;
  const int plane = unit / per_plane, within = unit % per_plane;
  const int j = p.j0 + within / p.nbi * p.seg;
  body(d, p.i0 + within % p.nbi * p.width, j, min(p.seg, p.j1 + 1 - j), plane % d.nk, plane / d.nk);
}

// What a march costs, for the choice of its segments: a step takes lone us plus
// wave us for each wave on its SIMD up to three, lone3 plus wave3 above that
// (whole waves where `whole`); a segment marches its rows, `extra` rows beside
// them and `lead` steps' worth of launch and first loads.  No more segments are
// tried once they have `least` rows, and where a SIMD has more than `free` waves
// they are at most `most` rows.
struct StripCost {
  double lone, wave, lone3, wave3;
  bool whole;
  int extra;
  double lead;
  int least, most;
  double free = 3.0;
};

// Rows per segment over `rows` rows of `planes` strips: the segment count with
// the least time by the march's cost.
int strip_segment_rows(int rows, int64_t planes, const StripCost& cost);

// Strips over columns [i0, i1] and rows [j0, j1] of every level and tile, in
// segments by the march's cost.
template <int NW = 4, typename F>
inline int launch_strips(hipStream_t s, const Dom& d, int i0, int i1, int j0, int j1, int width,
                         const StripCost& cost, const F& body, const char* who) {
  StripPlan p{i0, j0, j1, width, (i1 - i0 + width) / width, 1, j1 - j0 + 1};
  p.seg = strip_segment_rows(p.seg, (int64_t)p.nbi * d.nk * d.ntiles, cost);
  p.nbj = (j1 - j0 + p.seg) / p.seg;
  const int64_t total = (int64_t)p.nbi * p.nbj * d.nk * d.ntiles;
  FV3_REQUIRE(total < (int64_t)1 << 30, FV3_E_ARG, "%s: grid too large", who);
  const int64_t blocks = (total + NW - 1) / NW;
  const int64_t launched = (blocks + kNumXcd - 1) / kNumXcd * kNumXcd;
  hipLaunchKernelGGL((strip_kernel<NW, F>), dim3((unsigned)launched), dim3(64, NW), 0, s, d, p,
                     body);
  FV3_HIP_CHECK_LAUNCH(who);
  return FV3_OK;
}

}  // namespace fv3
