// GEMM operands in memory as 6-bit digits (gemm_digits.hip): layout, and how a row's values become digits.
#pragma once
#include "planes.h"

namespace cthip {

// Input rows.  A block of 32 consecutive k of a row has four digits per value, floats of 6 bits (1 sign, 2 exponent, 3 fraction bits: 0 .. 7.5), and a
// power of two per digit, 2^(e - 127), e - 5, e - 10, e - 15 for the digits 0 .. 3:  x = sum digit_t 2^(e - 5 t - 127), off by at most 2^-19 of the
// block's largest value.  Digit 2 j + h of row r lies where lane 32 h + r % 32 of instruction j of v_mfma_scale_f32_32x32x64_f8f6f4 reads it: one
// instruction sums two digits' products, the halves of its 64 k.
//   data    [rows / 32][K / 32] records of 3072 bytes: [j][lane]{16 bytes} [j][lane]{8 bytes}, value i of the block at bits 6 i .. 6 i + 5
//   scales  [K / 32][rows to 32] of 4 bytes: the exponents of digits 0, 2, 1, 3
constexpr int kDigitRecord = 3072;
inline int64_t digit_row_bytes(int64_t rows, int nkb) { return (rows + 31) / 32 * nkb * (kDigitRecord + 128); }

// Weights of 4 bits: records of 1024 bytes for 32 rows and a block of 32 k, [row]{16 bytes} [row]{8 bytes} [row]{scale as a float} and 128 bytes to spare, so
// that a record is one load of 16 bytes per lane.  A digit is (nibble - 8) / 2, exact; the scale is doubled.
constexpr int kDigitWRecord = 1024;

struct DigitGemmArgs : PlaneGemmArgs {
  const float *col_bias;  // the bias, added in front of everything else (`bias` is null)
  unsigned char *digits;  // non-null: the result goes out as digits instead of C
  int kper;               // blocks of 32 k per share of K (blockIdx.y); share s writes its sums to C + s M N
};

#if defined(__HIPCC__)
typedef int v8i_dg __attribute__((ext_vector_type(8)));
typedef unsigned v6u_dg __attribute__((ext_vector_type(6)));
typedef float v32f_dg __attribute__((ext_vector_type(32)));

// A block of 32 values of row `row` (k = 32 kb ..) as digits, into an operand of rows32 rows (a multiple of 32) and nkb blocks.  v is used up.
__device__ __forceinline__ void store_digits32(unsigned char *data, int64_t rows32, int nkb, int64_t row, int kb, float *v) {
  float m = fabsf(v[0]);
#pragma unroll
  for (int i = 1; i < 32; i++) m = __builtin_elementwise_maximum(m, fabsf(v[i]));  // (a NaN stays)
  // the largest value comes to 2 .. 4: what a digit leaves is then at most 1/8, 2^-5 of what the next one holds
  const bool top = !(m < INFINITY);
  const int e = max((int)(__float_as_uint(m) >> 23) - 1, 1);
  unsigned char *rec = data + ((row >> 5) * nkb + kb) * kDigitRecord + (row & 31) * 16;
  unsigned char *rec8 = data + ((row >> 5) * nkb + kb) * kDigitRecord + 2048 + (row & 31) * 8;
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const float s = __uint_as_float((unsigned)max(e - 5 * t, 1) << 23);
    v16f x, y;
#pragma unroll
    for (int i = 0; i < 16; i++) x[i] = v[2 * i], y[i] = v[2 * i + 1];
    v6u_dg d = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(x, y, s);
    if (t > 0 && e - 5 * t < 1)  // past the smallest power of two
#pragma unroll
      for (int i = 0; i < 6; i++) d[i] = 0;
    if (t < 3) {
      const v32f_dg b = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(d, s);
#pragma unroll
      for (int i = 0; i < 32; i++) v[i] -= b[i];  // exact
    }
    *(uint4 *)(rec + (t >> 1) * 1024 + (t & 1) * 512) = make_uint4(d[0], d[1], d[2], d[3]);
    *(uint2 *)(rec8 + (t >> 1) * 512 + (t & 1) * 256) = make_uint2(d[4], d[5]);
  }
  const unsigned e1 = max(e - 5, 1), e2 = max(e - 10, 1), e3 = max(e - 15, 1);
  ((unsigned *)(data + (rows32 >> 5) * nkb * kDigitRecord))[kb * rows32 + row] = top ? 0xffffffffu : (unsigned)e | e2 << 8 | e1 << 16 | e3 << 24;  // (255: not a number)
}
#endif

}  // namespace cthip
