// Building blocks of the wave-strip kernels: one wave of 64 lanes owns a strip
// of columns and marches up its rows, neighbours across i by lane shifts.
#pragma once

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
  int i, nj;
  uint32_t off0, offm, offp;  // byte offsets of columns i, i - 1, i + 1
  int64_t sj, sj2;
  __device__ __forceinline__ StripColumn(const Dom& d, int i_)
      : i(i_), nj(d.nj), sj(d.sj), sj2(d.sj2) {
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
};

}  // namespace fv3
