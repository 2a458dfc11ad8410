// f32 values as pairs of f16 (hi + lo) scaled by powers of two, for f16 MFMAs
// that compute f32 products: hi = f16(v), lo = f16(v - hi), so hi + lo is v to
// 2^-23 or better (one bit short of f32 for a quarter of the values) wherever
// |v| >= 2^-2, and to an absolute 2^-25 below.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rtg {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ unsigned f16_bits(float v) {
  const _Float16 h = (_Float16)v;
  return (unsigned)__builtin_bit_cast(uint16_t, h);
}
// The pair of v: hi in *hi, lo in *lo (f16 bits in the low half).
__device__ __forceinline__ void f16_split(float v, unsigned* hi, unsigned* lo) {
  const _Float16 h = (_Float16)v;
  const _Float16 l = (_Float16)(v - (float)h);
  *hi = (unsigned)__builtin_bit_cast(uint16_t, h);
  *lo = (unsigned)__builtin_bit_cast(uint16_t, l);
}
// Index (in f16 elements) of (row, k)'s hi in a row-major pair matrix of K
// columns, K % 32 == 0: each row is K / 32 groups of [32 hi][32 lo], 128 bytes
// each; the lo sits 32 elements after the hi.
__host__ __device__ inline size_t pair_index(size_t row, int k, int K) {
  return row * 2 * (size_t)K + (size_t)(k >> 5) * 64 + (k & 31);
}
// Stores the pairs of four consecutive columns (col % 4 == 0).
__device__ __forceinline__ void pair_store4(uint16_t* base, size_t row, int col, int K, const float4& v) {
  unsigned h[4], l[4];
  f16_split(v.x, &h[0], &l[0]);
  f16_split(v.y, &h[1], &l[1]);
  f16_split(v.z, &h[2], &l[2]);
  f16_split(v.w, &h[3], &l[3]);
  uint16_t* p = base + pair_index(row, col, K);
  *reinterpret_cast<uint2*>(p) = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
  *reinterpret_cast<uint2*>(p + 32) = make_uint2(l[0] | l[1] << 16, l[2] | l[3] << 16);
}

}  // namespace rtg
