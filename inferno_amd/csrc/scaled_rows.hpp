// Rows of activations as f16 values in units of a power of two per run of
// SPAN values: the largest of a run lies in [2^14, 2^15), so that f16 neither
// overflows nor loses small ones, whatever the rows' own size. A lane holds
// four neighbouring values, a wavefront 256.
#pragma once
#include <cfloat>

#include "gemv_common.hpp"

namespace inferno {
namespace scaled {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void load4(const uint16_t* x, float v[4]) {
  const uint2 w = ld_u2(reinterpret_cast<const uint8_t*>(x));
  v[0] = bits_to_f32(w.x << 16);
  v[1] = bits_to_f32(w.x & 0xffff0000u);
  v[2] = bits_to_f32(w.y << 16);
  v[3] = bits_to_f32(w.y & 0xffff0000u);
}
__device__ __forceinline__ void load4(const float* x, float v[4]) {
  const uint4 w = ld_u4(reinterpret_cast<const uint8_t*>(x));
  v[0] = bits_to_f32(w.x);
  v[1] = bits_to_f32(w.y);
  v[2] = bits_to_f32(w.z);
  v[3] = bits_to_f32(w.w);
}

// The run's exponent: its values times 2^e, the sums of them times 2^-e.
// (Infinities and NaN are left out; a subnormal maximum has exponent field 0,
// and 2^141 puts it below 2^15 all the same.)
template <int SPAN>
__device__ __forceinline__ int run_exponent(const float v[4]) {
  float m = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) m = fabsf(v[j]) <= FLT_MAX ? fmaxf(m, fabsf(v[j])) : m;
#pragma unroll
  for (int o = 1; o < SPAN / 4; o <<= 1) m = fmaxf(m, __shfl_xor(m, o, kWave));
  return m > 0.f ? 141 - int((f32_to_bits(m) >> 23) & 255u) : 0;
}

// Four halfs in the k order 0 2 1 3.
__device__ __forceinline__ void put4(uint16_t* out, const _Float16 q[4]) {
  const half2v a = {q[0], q[2]}, b = {q[1], q[3]};
  *reinterpret_cast<uint2*>(out) =
      make_uint2(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b));
}

}  // namespace scaled
}  // namespace inferno
