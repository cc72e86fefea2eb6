// Exact three-plane bf16 split of fp32 values (operands of products of six bf16 planes).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mpq {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pk_bf16(float x, float y) {
  const f32x2_t v = {x, y};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));  // v_cvt_pk_bf16_f32 (RNE)
}

// Three bf16 planes of the pair (x, y), each packed low = x, high = y:
// x = rn(x) + rn(x - rn(x)) + rn(rest) up to 2^-24 |x|.
__device__ __forceinline__ void split3(float x, float y, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = pk_bf16(x, y);
  const float rx = x - __builtin_bit_cast(float, h << 16);
  const float ry = y - __builtin_bit_cast(float, h & 0xffff0000u);
  m = pk_bf16(rx, ry);
  const float sx = rx - __builtin_bit_cast(float, m << 16);
  const float sy = ry - __builtin_bit_cast(float, m & 0xffff0000u);
  l = pk_bf16(sx, sy);
}

}  // namespace mpq
