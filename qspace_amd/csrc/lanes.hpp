// lanes.hpp -- sums and exchanges across a wave's lanes, and 1/sqrt (device)
#pragma once

#include <hip/hip_runtime.h>

namespace qsx {
namespace {

// v of the lane that the DPP row pattern CTRL names (a row is 16 lanes,
// active or inactive as a whole)
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
constexpr int DPP_XOR1 = 0xB1;          // quad_perm 1,0,3,2
constexpr int DPP_XOR2 = 0x4E;          // quad_perm 2,3,0,1
constexpr int DPP_HALF_MIRROR = 0x141;  // lane i of a half row takes 7 - i
constexpr int DPP_MIRROR = 0x140;       // lane i of a row takes 15 - i
constexpr int DPP_ROR4 = 0x124;         // rotation within the row
constexpr int DPP_ROR8 = 0x128;
template <int L>
constexpr int DPP_BCAST = 0x150 + L;    // lane L of the row to the whole row

// sum over the 16 lanes of a row, the same bits in every lane: pairs, quads,
// half rows, rows; each step adds two equal-bit partial sums in either
// order, so all lanes agree
__device__ __forceinline__ double seg_sum(double v) {
  v += dpp_mov<DPP_XOR1>(v);
  v += dpp_mov<DPP_XOR2>(v);
  v += dpp_mov<DPP_HALF_MIRROR>(v);
  v += dpp_mov<DPP_MIRROR>(v);
  return v;
}

// v + (v of the same lane of the other row of a pair of rows), the same bits
// in both
__device__ __forceinline__ double row_pair_sum(double v) {
  const long long b = __double_as_longlong(v);
  const auto lo = __builtin_amdgcn_permlane16_swap((int)b, (int)b, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((int)(b >> 32), (int)(b >> 32), false, false);
  return __longlong_as_double(((long long)hi[0] << 32) | (unsigned int)lo[0]) +
         __longlong_as_double(((long long)hi[1] << 32) | (unsigned int)lo[1]);
}

__device__ __forceinline__ double read_lane(double v, int l) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// v + (v of the lane 32 away), the same bits in both
__device__ __forceinline__ double half_pair_sum(double v) {
  const long long b = __double_as_longlong(v);
  const auto lo = __builtin_amdgcn_permlane32_swap((int)b, (int)b, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((int)(b >> 32), (int)(b >> 32), false, false);
  return __longlong_as_double(((long long)hi[0] << 32) | (unsigned int)lo[0]) +
         __longlong_as_double(((long long)hi[1] << 32) | (unsigned int)lo[1]);
}

// sum over the wave (all lanes active), the same bits in every lane
__device__ __forceinline__ double wave_sum(double v) { return half_pair_sum(row_pair_sum(seg_sum(v))); }

// 1/sqrt(x): the hardware's estimate and one third-order correction
__device__ __forceinline__ double rsqrt_d(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

}  // namespace
}  // namespace qsx
