// Pieces shared by the kernels that split FP32 operands into two FP16 values (split.hpp: the
// SM block; wgrad.hpp: its weight gradient).  Values are scaled by a power of two so that the
// largest finite magnitude lies in [2^t, 2^(t+1)), then v = hi + lo: hi, lo FP16, |error|
// below 2^-23 |v| or 2^-25 (half of FP16's smallest denormal; the matrix cores take
// denormals as they are).
#pragma once

#include <type_traits>

#include "common.hpp"

namespace mlpcg {
namespace split {

typedef f16 h8 __attribute__((ext_vector_type(8)));
typedef float f16x __attribute__((ext_vector_type(16)));
typedef unsigned u32x4s __attribute__((ext_vector_type(4)));

// magnitude bits of a finite value, 0 of others
__device__ __forceinline__ unsigned finite_bits(float v) {
  const unsigned u = __float_as_uint(v) & 0x7fffffffu;
  return u < 0x7f800000u ? u : 0u;
}
__device__ __forceinline__ unsigned magnitude(float v) { return __float_as_uint(v) & 0x7fffffffu; }
constexpr unsigned kInfinity = 0x7f800000u;
// the larger one, NaN if one is (v_maximum3_f32)
__device__ __forceinline__ float max_nan(float a, float b) { return __builtin_elementwise_maximum(a, b); }
// a magnitude in the order of its size, 0 above all (v_lshl_add_u32)
__device__ __forceinline__ unsigned small_bits(float v) { return (__float_as_uint(v) << 1) - 1u; }
// 2^e of the largest finite magnitude (its bits); 0 counts as 1
__device__ __forceinline__ int exponent_of(unsigned bits) {
  return bits == 0u ? 0 : (int)(bits >> 23) - 127;
}
__device__ __forceinline__ float pow2(int e) { return __uint_as_float((unsigned)(e + 127) << 23); }
// small_bits of 2^-2 before a scaling by 2^e: smaller values have fewer than 23 bits in two FP16
// values (2^-24 is FP16's smallest step)
__device__ __forceinline__ unsigned least_bits(int e) { return small_bits(ldexpf(0.25f, -e)); }

__device__ __forceinline__ unsigned wave_max(unsigned v) {
  auto step = [](unsigned x, auto ctrl, auto rows) {
    const unsigned o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, decltype(ctrl)::value, decltype(rows)::value,
                                                             0xf, false);
    return x > o ? x : o;
  };
  typedef std::integral_constant<int, 0xf> All;
  v = step(v, std::integral_constant<int, 0x111>(), All());
  v = step(v, std::integral_constant<int, 0x112>(), All());
  v = step(v, std::integral_constant<int, 0x114>(), All());
  v = step(v, std::integral_constant<int, 0x118>(), All());
  v = step(v, std::integral_constant<int, 0x142>(), std::integral_constant<int, 0xa>());
  v = step(v, std::integral_constant<int, 0x143>(), std::integral_constant<int, 0xc>());
  return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, bytes, 0x00020000);
}
__device__ __forceinline__ float ld_as(__amdgpu_buffer_rsrc_t r, unsigned boff, int soff, const float*) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, boff, soff, 0));
}
__device__ __forceinline__ float ld_as(__amdgpu_buffer_rsrc_t r, unsigned boff, int soff, const bf16*) {
  return (float)__builtin_bit_cast(bf16, __builtin_amdgcn_raw_buffer_load_b16(r, boff, soff, 0));
}
__device__ __forceinline__ float ld_as(__amdgpu_buffer_rsrc_t r, unsigned boff, int soff, const f16*) {
  return (float)__builtin_bit_cast(f16, __builtin_amdgcn_raw_buffer_load_b16(r, boff, soff, 0));
}

}  // namespace split
}  // namespace mlpcg
