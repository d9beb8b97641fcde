// lanes.hpp -- lane exchanges within a wave shared by the gfx950 kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace pgsvt {

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}

// v + the value of the lane 16 (32) away: the row (half) swap of gfx950 leaves
// both addends in one lane, without a trip through LDS (__shfl_xor is a
// ds_bpermute: 31-frame 8 x 8 patches, whose dot products end in one, took
// 205 ms for 1.36 M matrices of 64 x 31 with it)
__device__ __forceinline__ float add_row16(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}
__device__ __forceinline__ float add_half32(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}
__device__ __forceinline__ double add_row16(double v) {
  const uint2 u = __builtin_bit_cast(uint2, v);
  const auto x = __builtin_amdgcn_permlane16_swap(u.x, u.x, false, false);
  const auto y = __builtin_amdgcn_permlane16_swap(u.y, u.y, false, false);
  return __builtin_bit_cast(double, make_uint2((uint32_t)x[0], (uint32_t)y[0])) +
         __builtin_bit_cast(double, make_uint2((uint32_t)x[1], (uint32_t)y[1]));
}
__device__ __forceinline__ double add_half32(double v) {
  const uint2 u = __builtin_bit_cast(uint2, v);
  const auto x = __builtin_amdgcn_permlane32_swap(u.x, u.x, false, false);
  const auto y = __builtin_amdgcn_permlane32_swap(u.y, u.y, false, false);
  return __builtin_bit_cast(double, make_uint2((uint32_t)x[0], (uint32_t)y[0])) +
         __builtin_bit_cast(double, make_uint2((uint32_t)x[1], (uint32_t)y[1]));
}

// The empty asm statement on entry makes v an opaque, already rounded
// value.  Without it the compiler contracts the caller's product into the
// first butterfly add, fma(x_i, x_j, neighbour's rounded product), which
// rounds differently in the two lanes of a pair: the lanes then hold
// different sums and apply different rotations (seen as singular values
// off by 1e-2 of s_max on near-degenerate column pairs).
template <int L>
__device__ __forceinline__ float group_sum(float v) {
  asm volatile("" : "+v"(v));
  if (L >= 2) v += dpp_f<0xB1>(v);   // quad_perm [1,0,3,2]
  if (L >= 4) v += dpp_f<0x4E>(v);   // quad_perm [2,3,0,1]
  if (L >= 8) v += dpp_f<0x141>(v);  // row_half_mirror
  if (L >= 16) v += dpp_f<0x140>(v); // row_mirror
  if (L >= 32) v = add_row16(v);
  if (L >= 64) v = add_half32(v);
  return v;
}

// FP64 (the divergence factors and the precision-study path): the same
// DPP steps on both halves of the double; after each step the lanes that
// are paired next hold equal partial sums, so the result is the one of
// the lane-swap (xor) butterfly and bit-identical in every lane
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
  const int2 h = __builtin_bit_cast(int2, v);
  int2 o;
  o.x = __builtin_amdgcn_update_dpp(0, h.x, CTRL, 0xF, 0xF, false);
  o.y = __builtin_amdgcn_update_dpp(0, h.y, CTRL, 0xF, 0xF, false);
  return __builtin_bit_cast(double, o);
}
template <int L>
__device__ __forceinline__ double group_sum(double v) {
  asm volatile("" : "+v"(v));
  if (L >= 2) v += dpp_d<0xB1>(v);   // quad_perm [1,0,3,2]
  if (L >= 4) v += dpp_d<0x4E>(v);   // quad_perm [2,3,0,1]
  if (L >= 8) v += dpp_d<0x141>(v);  // row_half_mirror
  if (L >= 16) v += dpp_d<0x140>(v); // row_mirror
  if (L >= 32) v = add_row16(v);
  if (L >= 64) v = add_half32(v);
  return v;
}

// f(std::integral_constant<int, K>) for K = K0 .. K1 - 1, in order
template <int K0, int K1, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (K0 < K1) {
    f(std::integral_constant<int, K0>());
    static_for<K0 + 1, K1>(f);
  }
}

// d_0 w_0 v_0 as each form of the overlap-add has always rounded it: patches
// up to 4 x 4 d_0 (w_0 v_0), larger ones (d_0 w_0) v_0; never contracted.
template <bool SMALL>
__device__ __forceinline__ float lead_product(float d0, float w0, float v0) {
#pragma clang fp contract(off)
  return SMALL ? d0 * (w0 * v0) : (d0 * w0) * v0;
}

}  // namespace pgsvt
