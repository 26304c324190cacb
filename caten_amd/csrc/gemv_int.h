// Products of 4-bit weights with a vector as integers on the matrix cores: the vector's digits, where they lie in LDS, and a
// chunk's product (gemv_int.hip says what for).
#pragma once
#include "common.h"

namespace cthip {

typedef int v4i __attribute__((ext_vector_type(4)));

// A chunk's sums are taken times 2^-28 and its power of two times 2^28: a weight row's scale, a multiple of 2^-24, times that power is then exact down to
// chunks of subnormal numbers, and in range as far up as the vector kernels' sums of nibble times input are.
// four consecutive k of a chunk (eight neighbouring lanes hold one): digit words of the four elements, and what undoes the
// chunk's power of two (and the 16 of a nibble).  A chunk with one infinity keeps its sign there and nothing else, 2^e becomes infinity: the product is
// what it is of floats.  With a NaN, or with infinities whose products would be added up before they are infinite, 2^e becomes NaN (as the vector kernels' sums do).
__device__ __forceinline__ float int_digits(const float *v, unsigned *w) {
  unsigned m = 0;
#pragma unroll
  for (int e = 0; e < 4; e++) m = max(m, __float_as_uint(v[e]) & 0x7fffffffu);  // (as integers: a NaN is the largest)
  m = max(m, (unsigned)__builtin_amdgcn_mov_dpp((int)m, 0xB1, 0xf, 0xf, true));   // quad_perm 1, 0, 3, 2
  m = max(m, (unsigned)__builtin_amdgcn_mov_dpp((int)m, 0x4E, 0xf, 0xf, true));   // quad_perm 2, 3, 0, 1
  m = max(m, (unsigned)__builtin_amdgcn_mov_dpp((int)m, 0x141, 0xf, 0xf, true));  // row_half_mirror
  const unsigned E = max(m >> 23, 7u);  // (a unit is 2^(E - 156); at 7 the smallest subnormal number, of which every float is a multiple)
  const bool finite = m < 0x7f800000u;
  // (the factor itself may lie past the largest float; 30 bits and a sign)
  int x[4], infs = 0;
#pragma unroll
  for (int e = 0; e < 4; e++) x[e] = (int)rintf(__builtin_amdgcn_ldexpf(v[e], 156 - (int)E));
  if (__builtin_expect(__any(!finite), 0)) {  // (uniform: the eight lanes of a chunk are together)
    // an infinity stays one of 2^30 and what is beside it becomes nothing
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (!finite) x[e] = (int)__builtin_amdgcn_fmed3f(__builtin_amdgcn_ldexpf(v[e], -512), -0x1p30f, 0x1p30f);
#pragma unroll
    for (int e = 0; e < 4; e++) infs += abs(x[e]) >> 30;
    infs += __builtin_amdgcn_mov_dpp(infs, 0xB1, 0xf, 0xf, true);
    infs += __builtin_amdgcn_mov_dpp(infs, 0x4E, 0xf, 0xf, true);
    infs += __builtin_amdgcn_mov_dpp(infs, 0x141, 0xf, 0xf, true);
  }
  unsigned t[4];
#pragma unroll
  for (int e = 0; e < 4; e++) t[e] = ((unsigned)x[e] + 0x808080u) ^ 0x808080u;  // bytes: signed digits, the highest in byte 3
  const unsigned a01 = __builtin_amdgcn_perm(t[1], t[0], 0x05010400u), a23 = __builtin_amdgcn_perm(t[3], t[2], 0x05010400u);
  const unsigned b01 = __builtin_amdgcn_perm(t[1], t[0], 0x07030602u), b23 = __builtin_amdgcn_perm(t[3], t[2], 0x07030602u);
  w[0] = __builtin_amdgcn_perm(b23, b01, 0x07060302u);
  w[1] = __builtin_amdgcn_perm(b23, b01, 0x05040100u);
  w[2] = __builtin_amdgcn_perm(a23, a01, 0x07060302u);
  w[3] = __builtin_amdgcn_perm(a23, a01, 0x05040100u);
  return m > 0x7f800000u || infs > 1 ? __uint_as_float(0x7fc00000u) : finite ? __uint_as_float((E - 5u) << 23) : INFINITY;
}
// digits of elements 4 k .. 4 k + 3 and, from a chunk's first lane, its power of two: 128 bytes per chunk, [half of its k][digit][16 bytes]
__device__ __forceinline__ void int_digits_put(unsigned char *dig, float *sx, int k, const unsigned *w, float down) {
  unsigned *o = (unsigned *)(dig + (size_t)(k >> 2) * 64) + (k & 3);
#pragma unroll
  for (int r = 0; r < 4; r++) o[4 * r] = w[r];
  if (k % 8 == 0) sx[k >> 3] = down;
}
// 16 bytes of a weight row against the chunk's digits (a0: its first 16 k, a1: the others), without the two scales
__device__ __forceinline__ float int_chunk(uint4 q, v4i a0, v4i a1) {
  v4i r = {0, 0, 0, 0};
  const unsigned dw[4] = {q.x, q.y, q.z, q.w};
  v4i lo, hi;
#pragma unroll
  for (int t = 0; t < 4; t++) {  // 16 (n - 8): the nibble in the byte's upper half, its top bit turned
    lo[t] = (int)(((dw[t] << 4) & 0xf0f0f0f0u) ^ 0x80808080u);
    hi[t] = (int)((dw[t] & 0xf0f0f0f0u) ^ 0x80808080u);
  }
  r = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, lo, r, 0, 0, 0);
  r = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, hi, r, 0, 0, 0);
  return fmaf((float)(r[0] * 256 + r[1]), 0x1p-12f, (float)(r[2] * 256 + r[3]) * 0x1p-28f);
}

}  // namespace cthip
