// Sums over a wave's lanes in fp64, as kgs_common.h's of floats, and a lane's squares towards them.
#pragma once

#include "kgs_common.h"

namespace kgs {

__device__ __forceinline__ double xor16_sum(double x) {
  const uint2 u = __builtin_bit_cast(uint2, x);
  const auto lo = __builtin_amdgcn_permlane16_swap(u.x, u.x, true, false), hi = __builtin_amdgcn_permlane16_swap(u.y, u.y, true, false);
  return __builtin_bit_cast(double, make_uint2(lo[0], hi[0])) + __builtin_bit_cast(double, make_uint2(lo[1], hi[1]));
}
__device__ __forceinline__ double xor32_sum(double x) {
  const uint2 u = __builtin_bit_cast(uint2, x);
  const auto lo = __builtin_amdgcn_permlane32_swap(u.x, u.x, true, false), hi = __builtin_amdgcn_permlane32_swap(u.y, u.y, true, false);
  return __builtin_bit_cast(double, make_uint2(lo[0], hi[0])) + __builtin_bit_cast(double, make_uint2(lo[1], hi[1]));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(double x) {
  const int2 u = __builtin_bit_cast(int2, x);
  return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_update_dpp(0, u.x, CTRL, 0xf, 0xf, false),
                                              __builtin_amdgcn_update_dpp(0, u.y, CTRL, 0xf, 0xf, false)));
}
__device__ __forceinline__ double wave_sum(double x) {
  x += dpp_move<0xB1>(x);
  x += dpp_move<0x4E>(x);
  x += dpp_move<0x141>(x);
  x += dpp_move<0x140>(x);
  return xor32_sum(xor16_sum(x));
}

// A row's sum of squares while its values pass as MFMA operands: a lane's eight of a k-step in fp32, on from there in fp64, so that
// the sum is as good as rounded once. Relative rms error over normal rows of 4096: so 2.8e-8; a chain of MFMAs of x with itself 1.2e-7 at 16
// k-steps, 3.2e-7 at 128; the producers' workgroups' sums, added exactly (add_exact in decode_common.h), 3.0e-8. Four columns 30 times the others: 3.1e-8,
// 4.3e-7 at 128, 3.7e-8.
typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));
__device__ __forceinline__ double add_squares(double sum, bf16x8 v) {
  const bf16x8v b = __builtin_bit_cast(bf16x8v, v);
  float f = 0.f;
#pragma unroll
  for (int i = 0; i < 8; i += 2) f = __builtin_amdgcn_fdot2_f32_bf16(bf16x2v{b[i], b[i + 1]}, bf16x2v{b[i], b[i + 1]}, f, false);
  return sum + f;
}

}  // namespace kgs
