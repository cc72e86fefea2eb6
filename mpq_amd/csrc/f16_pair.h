// fp32 values as pairs of f16 planes (the operands of the split products in gemm.hip).
//
// With a power-of-two scale s that brings the largest of a group of values below 2^15, x s is held as
//   h = rn(x s), l = rn(x s - h)   (rn: round to nearest f16)
// The residual x s - h is exact in fp32 and at most 2^-11 |x s|, so h + l differs from x s by at most
// 2^-23 |x s|, or 2^-25 where l is subnormal (values more than 2^14 below the largest).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mpq {

typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2p_t __attribute__((ext_vector_type(2)));

// Columns of one scale group of the left operand: its producers write 1024-column chunks per work-group.
constexpr int kPairChunk = 1024;

__device__ __forceinline__ f16x2_t pk_f16(float x, float y) {
  const f32x2p_t v = {x, y};
  return __builtin_convertvector(v, f16x2_t);  // v_cvt_pk_f16_f32 (RNE)
}

// Planes of the pair (x s, y s), each packed low = x, high = y.
__device__ __forceinline__ void split2(float x, float y, float s, uint32_t& h, uint32_t& l) {
  const f16x2_t hv = pk_f16(x * s, y * s);
  const f16x2_t lv = pk_f16(fmaf(x, s, -(float)hv.x), fmaf(y, s, -(float)hv.y));
  h = __builtin_bit_cast(uint32_t, hv);
  l = __builtin_bit_cast(uint32_t, lv);
}

// Power of two that brings a group whose largest magnitude is m (m >= 0) to [2^top, 2^(top+1)); at most
// 2^126 (so that its reciprocal is normal), 1 for a group that is zero or not finite.
__device__ __forceinline__ float pair_scale(float m, int top) {
  if (!(m > 0.f) || !(m < INFINITY)) return 1.f;
  int e;
  (void)frexpf(m, &e);  // m in [2^(e-1), 2^e)
  const int k = top + 1 - e;
  return ldexpf(1.f, k > 126 ? 126 : k);
}

// The packed left operand of a split product (M x K, K % 32 == 0, Mp = M rounded up to 128):
//   planes [Mp/128][K/16][2][256 chunks][8 f16], chunk (blk*2 + h)*32 + r holding row 128 mt + 32 blk + r
//   at k = 16 ks + 8 h + (0..7), scaled by the scale of (row, k / 1024);
//   then the reciprocal scales, float [ceil(K/1024)][Mp].
__device__ __forceinline__ float* pair_inv_scales(uint4* At, int64_t Mp, int64_t K) {
  return reinterpret_cast<float*>(At + Mp * K / 4);
}

// Planes of x[b][j0 .. j0+3] (j0 % 4 == 0, row b) scaled by s at their place in the packed operand.
__device__ __forceinline__ void store_pair4(uint4* __restrict__ At, int64_t K, int64_t b, int64_t j0, float4 v, float s) {
  const int64_t KS = K / 16;
  const int64_t mt = b >> 7;
  const int r = (int)(b & 31), blk = (int)((b >> 5) & 3);
  const int64_t ks = j0 >> 4;
  const int h = (int)((j0 >> 3) & 1), half = (int)((j0 >> 2) & 1);
  const int c = (blk * 2 + h) * 32 + r;
  uint2 hi, lo;
  split2(v.x, v.y, s, hi.x, lo.x);
  split2(v.z, v.w, s, hi.y, lo.y);
  uint2* base = reinterpret_cast<uint2*>(At + (mt * KS + ks) * 512 + c) + half;
  base[0] = hi;
  base[512] = lo;
}

// One work-group (256 threads) packs 1024 columns of row b: thread t's four values are columns
// 1024 chunk + 4 t + (0..3) (zero where the column does not exist).  `red`: 4 floats of LDS.
__device__ __forceinline__ void pack_pair_chunk(uint4* __restrict__ At, int64_t M, int64_t K, int64_t b, int64_t chunk,
                                                float4 v, float* red) {
  float m = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  const float s = pair_scale(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])), 14);
  const int64_t j0 = chunk * kPairChunk + 4 * (int64_t)threadIdx.x;
  if (j0 < K) store_pair4(At, K, b, j0, v, s);
  const int64_t Mp = (M + 127) / 128 * 128;
  if (threadIdx.x == 0) pair_inv_scales(At, Mp, K)[chunk * Mp + b] = 1.f / s;
}

}  // namespace mpq
