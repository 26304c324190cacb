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
//   rests   [rows / 32][K / 32] of 4096 bytes: two bf16 terms per value, as v_mfma_f32_32x32x16_bf16 takes them, [term][8 s ..][lane]{8 k}: lane 32 h + r % 32 has k 16 h + 8 s .. + 7;
//           written and read where a block says so
//
// Two bf16 terms are off by 2^-18 of each value, digits by 2^-19 of a block's largest: less for most of what a Linear sums (normal values 1.03e-6 against 2.46e-6), but a result
// that the largest values do not reach (a weight of 4 bits is often exactly zero) has the small ones' error alone.  A block that would lose by that has three digits and, as two
// terms, what they leave, so that every value is off by 2^-18 of itself at most; its fourth exponent is 0, which no other has, and the products' kernel adds these terms' products
// behind its own loop.  Which blocks: digits_uneven_columns, digits_one_large, digits_uneven below.  So do blocks whose largest value is below 2^-110: a digit's power of two ends at 2^-126.
constexpr int kDigitRecord = 3072, kDigitScales = 128, kDigitRests = 4096;
inline int64_t digit_row_bytes(int64_t rows, int nkb) { return (rows + 31) / 32 * nkb * (kDigitRecord + kDigitScales + kDigitRests); }

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
typedef unsigned v16u_dg __attribute__((ext_vector_type(16)));
typedef float v32f_dg __attribute__((ext_vector_type(32)));

// 32 values over s as floats of 6 bits, x[i] and y[i] the values 2 i and 2 i + 1.  (Written out, for the builtin lets the result take the scale's register, and then what comes out is wrong.)
__device__ __forceinline__ v6u_dg digits_of(v16f x, v16f y, float s) {
  v6u_dg d;
  asm("s_nop 0\n\tv_cvt_scalef32_2xpk16_fp6_f32 %0, %1, %2, %3" : "=&v"(d) : "v"(x), "v"(y), "v"(s));
  return d;
}
// The largest magnitude of a block (a NaN stays)
__device__ __forceinline__ float digits_top(const float *v) {
  float m = fabsf(v[0]);
#pragma unroll
  for (int i = 1; i < 32; i++) m = __builtin_elementwise_maximum(m, fabsf(v[i]));
  return m;
}
// What decides whether a block of a row has its rest as terms; m: its largest magnitude.  Error of a result that the large columns of a block do not reach, against two terms'
// (a model of both on the host; rows of normal values, k of 32 columns r times as large, their weights zero; without such columns 0.4):
//   k, r                        1, 8  1, 32  1, 64  1, 256  1, 1000   4, 8  4, 32  4, 256   16, 32  16, 256   24, 32  24, 256   one row of 32, k = 1, r = 16  32   64
//   digits alone                1.3   5.3    10     42      165       2.1   8.4    67       12      93        13      100       3.6                            7.2  14
//   uneven columns, one large   1.3   3.8    3.3    1.3     1.0       2.1   1.3    1.0      11      1.0       13      1.0       3.6                            7.2  2.2
//   uneven row, one large       1.3   1.5    1.2    1.0     1.0       1.9   1.2    1.0      3.2     1.0       12      1.8       (a row by itself: as on the left)
//     (28 columns of 32 and more: as digits alone up to 256, 240 at 1000; 31 of 32: as digits alone at any, for a single value that is small says nothing)
// Blocks that have a rest without need, of 100000: columns: normal values, Laplace's, GELU(x) 0, x SiLU(y) 1; row: normal values 0.1, Laplace's 60, scaled by exp(y / 2) a column 70
// (of x SiLU(y), which no norm leaves, 16000).
//
// Of a column of a group's rows, how far it is below the largest values: half of log2(the rows' largest values' squares / its squares); past 18 in the mean square of the columns
// (fewer rows: more, for chance makes columns of a few rows small), or 2^13 and more in any.  Lanes 0 .. 31 (32 .. 63) hold the rows, all of them active; `in`: this lane's row counts.  A row is taken
// relative to the power of two of its largest value.  True in every lane of the half or in none.
__device__ __forceinline__ bool digits_uneven_columns(const float *v, float m, bool in) {
  const int lane = threadIdx.x & 63;
  const bool ok = in && m > 0.0f && m < INFINITY;
  // (the largest value comes to 0.5 .. 1, past 2^126 to less than 4, so that squares may be held to 0 .. 1, a bit of their instruction that makes a NaN 0: a row that is not finite counts as
  // nothing, and the others are looked at without it)
  const float up = ok ? __uint_as_float((253u - min(max(__float_as_uint(m) >> 23, 1u), 252u)) << 23) : 0.0f;
  float s[32];
#pragma unroll
  for (int i = 0; i < 32; i++) {
    const float t = v[i] * up;
    s[i] = __builtin_amdgcn_fmed3f(t * t, 0.0f, 1.0f);
  }
  // a column's sum to each lane: half of the columns a step, to the lanes that keep them
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(s[i]), __float_as_uint(s[i + 16]), false, false);
    s[i] = __uint_as_float(t[0]) + __uint_as_float(t[1]);
  }
#define CTHIP_DIGITS_STEP(N, DPP)                                                                                                            \
  for (int i = 0; i < N; i++) {                                                                                                              \
    const float keep = lane & N ? s[i + N] : s[i], give = lane & N ? s[i] : s[i + N];                                                        \
    s[i] = keep + __uint_as_float((unsigned)__builtin_amdgcn_mov_dpp((int)__float_as_uint(give), DPP, 0xf, 0xf, true));                      \
  }
#pragma unroll
  CTHIP_DIGITS_STEP(8, 0x140)  // row_mirror
#pragma unroll
  CTHIP_DIGITS_STEP(4, 0x141)  // row_half_mirror
#pragma unroll
  CTHIP_DIGITS_STEP(2, 0x1b)  // quad_perm 3, 2, 1, 0
  CTHIP_DIGITS_STEP(1, 0xb1)  // quad_perm 1, 0, 3, 2
#undef CTHIP_DIGITS_STEP
  auto half_sum = [](float t) __attribute__((always_inline)) {
    t += __uint_as_float((unsigned)__builtin_amdgcn_mov_dpp((int)__float_as_uint(t), 0xb1, 0xf, 0xf, true));
    t += __uint_as_float((unsigned)__builtin_amdgcn_mov_dpp((int)__float_as_uint(t), 0x4e, 0xf, 0xf, true));
    t += __uint_as_float((unsigned)__builtin_amdgcn_mov_dpp((int)__float_as_uint(t), 0x141, 0xf, 0xf, true));
    t += __uint_as_float((unsigned)__builtin_amdgcn_mov_dpp((int)__float_as_uint(t), 0x140, 0xf, 0xf, true));
    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(t), __float_as_uint(t), false, false);
    return __uint_as_float(p[0]) + __uint_as_float(p[1]);
  };
  const float top = ok ? m * up : 0.0f;
  const float all = half_sum(top * top);
  const unsigned long long rows = __ballot(ok);
  const float n = (float)__popc((unsigned)(lane & 32 ? rows >> 32 : rows));
  const float below = s[0] > 0.0f ? 0.5f * (__builtin_amdgcn_logf(all) - __builtin_amdgcn_logf(s[0])) : 0.0f;  // (logf: of base 2)
  const unsigned long long lost = __ballot(below > 13.0f);
  return half_sum(below * below) * n > 32.0f * (18.0f * n + 24.0f) || (unsigned)(lane & 32 ? lost >> 32 : lost) != 0;
}
// A value past all others of its block together, in this row (beside columns: a token's own)
__device__ __forceinline__ bool digits_one_large(const float *v, float m) {
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < 32; i++) s += fabsf(v[i]);
  return s < 1.5f * m;
}
// Where a thread has a row by itself, and rows are what a norm leaves, of one magnitude but for a few values: what log2(largest / value) has past 4.5, summed, past 32 (normal values
// 3.8, off by 3.3; the logarithm's fraction taken as linear; zeros lose nothing).  (Its mean square past 30 in that place took 24 of 32 columns 256 times as large for even in half of the rows.)
__device__ __forceinline__ bool digits_uneven(const float *v, float m) {
  const unsigned top = max(__float_as_uint(m) << 1, 9u << 23) - (9u << 23);
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < 32; i++) s += (float)(top - min((__float_as_uint(v[i]) << 1) - 1u, top));
  return s > 32.0f * 0x1p24f;
}

// A block of 32 values of row `row` (k = 32 kb ..) as digits, into an operand of rows32 rows (a multiple of 32) and nkb blocks; m: their largest magnitude, rest: what the last
// digit would hold and all below it as terms.  v is used up.
__device__ __forceinline__ void store_digits32(unsigned char *data, int64_t rows32, int nkb, int64_t row, int kb, float *v, float m, bool rest) {
  // the largest value comes to 2 .. 4: what a digit leaves is then at most 1/8, 2^-5 of what the next one holds
  const bool top = !(m < INFINITY);
  const int e = max((int)(__float_as_uint(m) >> 23) - 1, 1);
  const int64_t group = (row >> 5) * nkb + kb, groups = (rows32 >> 5) * nkb;
  unsigned char *rec = data + group * kDigitRecord + (row & 31) * 16;
  unsigned char *rec8 = data + group * kDigitRecord + 2048 + (row & 31) * 8;
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const float s = __uint_as_float((unsigned)max(e - 5 * t, 1) << 23);
    v16f x, y;
#pragma unroll
    for (int i = 0; i < 16; i++) x[i] = v[2 * i], y[i] = v[2 * i + 1];
    v6u_dg d = digits_of(x, y, s);
    if (t > 0 && e - 5 * t < 1)  // past the smallest power of two
#pragma unroll
      for (int i = 0; i < 6; i++) d[i] = 0;
    if (t == 3) {
      rest = (rest || e < 16) && !top;
      if (rest) {
        float left = 0.0f;
#pragma unroll
        for (int i = 0; i < 32; i++) left = fmaxf(left, fabsf(v[i]));
        rest = left != 0.0f;
      }
      if (rest) {
        uint4 *o = (uint4 *)(data + groups * (kDigitRecord + kDigitScales) + group * kDigitRests) + (row & 31);
#pragma unroll
        for (int q = 0; q < 4; q++) {  // k 8 q .. + 7: half q / 2, slice q % 2
          unsigned h[4], l[4];
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const float v0 = v[8 * q + 2 * i], v1 = v[8 * q + 2 * i + 1];
            h[i] = pack_bf16_pl(v0, v1);
            l[i] = pack_bf16_pl(v0 - __uint_as_float(h[i] << 16), v1 - __uint_as_float(h[i] & 0xffff0000u));
          }
          o[(q & 1) * 64 + (q >> 1) * 32] = make_uint4(h[0], h[1], h[2], h[3]);
          o[128 + (q & 1) * 64 + (q >> 1) * 32] = make_uint4(l[0], l[1], l[2], l[3]);
        }
#pragma unroll
        for (int i = 0; i < 6; i++) d[i] = 0;
      }
    } else {
      const v32f_dg b = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(d, s);
#pragma unroll
      for (int i = 0; i < 32; i++) v[i] -= b[i];  // exact
    }
    *(uint4 *)(rec + (t >> 1) * 1024 + (t & 1) * 512) = make_uint4(d[0], d[1], d[2], d[3]);
    *(uint2 *)(rec8 + (t >> 1) * 512 + (t & 1) * 256) = make_uint2(d[4], d[5]);
  }
  const unsigned e1 = max(e - 5, 1), e2 = max(e - 10, 1), e3 = rest ? 0 : max(e - 15, 1);
  ((unsigned *)(data + groups * kDigitRecord))[kb * rows32 + row] = top ? 0xffffffffu : (unsigned)e | e2 << 8 | e1 << 16 | e3 << 24;  // (255: not a number)
}
#endif

}  // namespace cthip
