// Rounding fp32 values to 16-bit parts and packed dot products, shared by the expected-side GEMMs and the kernels
// that make their operands.
#pragma once
#include "common.h"

__device__ __forceinline__ uint32_t to_bf16_bits(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (u >> 16) | 0x40u;       // NaN stays NaN (quiet)
  u += 0x7FFFu + ((u >> 16) & 1u);                                    // round to nearest even
  return u >> 16;
}

template <int DT>
__device__ __forceinline__ uint32_t round_bits(float f) {
  if constexpr (DT == SDC_BF16) return to_bf16_bits(f);
  else return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)f);
}

template <int DT>
__device__ __forceinline__ float bits_value(uint32_t b) {
  return half_to_f32<DT>((uint16_t)b);
}

// fp32 -> hi, mid, lo parts of 8 values (checksum._split3), packed as three u32x4
template <int DT>
__device__ __forceinline__ void split8(const float* v, u32x4* parts) {
  uint32_t h[8], md[8], lo[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    h[i] = round_bits<DT>(v[i]);
    const float r = v[i] - bits_value<DT>(h[i]);
    md[i] = round_bits<DT>(r);
    lo[i] = round_bits<DT>(r - bits_value<DT>(md[i]));
  }
  uint32_t* o0 = reinterpret_cast<uint32_t*>(&parts[0]);
  uint32_t* o1 = reinterpret_cast<uint32_t*>(&parts[1]);
  uint32_t* o2 = reinterpret_cast<uint32_t*>(&parts[2]);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    o0[i] = h[2 * i] | (h[2 * i + 1] << 16);
    o1[i] = md[2 * i] | (md[2 * i + 1] << 16);
    o2[i] = lo[2 * i] | (lo[2 * i + 1] << 16);
  }
}

// a . b + c over the two 16-bit halves of a and b (fp32 accumulation)
template <int DT>
__device__ __forceinline__ float pk_dot2(uint32_t a, uint32_t b, float c) {
  if constexpr (DT == SDC_BF16)
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c, false);
  else
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, a), __builtin_bit_cast(f16x2, b), c, false);
}
