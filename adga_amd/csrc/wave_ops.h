// Wave-level moves and reductions of the pivot searches (64-wide wavefronts).
#pragma once

#include "adga_common.h"

namespace adga {

// component-wise select of two complex values (a select of whole structs can turn into a select of
// their addresses, which forces register arrays into scratch memory)
template <typename T>
__device__ __forceinline__ cplx<T> csel(bool c, cplx<T> a, cplx<T> b) {
  return mk<T>(c ? a.re : b.re, c ? a.im : b.im);
}

// Lane moves inside 16-lane rows (DPP row_ror) and reductions over a row: every lane of the row
// ends with the row's result.
template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
  return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false);
}
template <int CTRL>
__device__ __forceinline__ float dpp_v(float v) {
  return __int_as_float(dpp_i<CTRL>(__float_as_int(v)));
}
template <int CTRL>
__device__ __forceinline__ double dpp_v(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = dpp_i<CTRL>((int)b), hi = dpp_i<CTRL>((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <typename T>
__device__ __forceinline__ T row_max(T v) {  // no NaN among the values
  T o = dpp_v<0x121>(v);
  v = o > v ? o : v;
  o = dpp_v<0x122>(v);
  v = o > v ? o : v;
  o = dpp_v<0x124>(v);
  v = o > v ? o : v;
  o = dpp_v<0x128>(v);
  return o > v ? o : v;
}
__device__ __forceinline__ int row_min(int v) {
  v = min(v, dpp_i<0x121>(v));
  v = min(v, dpp_i<0x122>(v));
  v = min(v, dpp_i<0x124>(v));
  return min(v, dpp_i<0x128>(v));
}
template <typename T>
__device__ __forceinline__ T lane_value(T v, int l);
template <>
__device__ __forceinline__ float lane_value(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
template <>
__device__ __forceinline__ double lane_value(double v, int l) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// the wave's maximum, the same value in every lane
template <typename T>
__device__ __forceinline__ T wave_max(T v) {
  v = row_max(v);
  const T a = lane_value(v, 0), b = lane_value(v, 16), c = lane_value(v, 32), d = lane_value(v, 48);
  const T ab = a > b ? a : b, cd = c > d ? c : d;
  return ab > cd ? ab : cd;
}

// the wave's maximum of unsigned words, uniform: 16-lane rows, then across them (row_bcast 15 and 31) into lane 63
__device__ __forceinline__ unsigned wave_umax(unsigned v) {
  auto step = [](unsigned x, int o) { return max(x, (unsigned)o); };
  v = step(v, dpp_i<0x121>((int)v));
  v = step(v, dpp_i<0x122>((int)v));
  v = step(v, dpp_i<0x124>((int)v));
  v = step(v, dpp_i<0x128>((int)v));
  v = step(v, __builtin_amdgcn_update_dpp((int)v, (int)v, 0x142, 0xa, 0xf, false));
  v = step(v, __builtin_amdgcn_update_dpp((int)v, (int)v, 0x143, 0xc, 0xf, false));
  return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}
// The lanes whose 64-bit keys are the wave's largest, as a mask: by the upper words, which as a rule leave one
// lane, then by the lower ones.
__device__ __forceinline__ unsigned long long wave_argmax(unsigned long long key) {
  const unsigned hi = (unsigned)(key >> 32), lo = (unsigned)key;
  unsigned long long m = __ballot(hi == wave_umax(hi));
  if (__popcll(m) > 1) {
    const bool in = (m >> (threadIdx.x & 63)) & 1;
    m &= __ballot(lo == wave_umax(in ? lo : 0u));
  }
  return m;
}

}  // namespace adga
