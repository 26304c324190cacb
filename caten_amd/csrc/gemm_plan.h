// What launch_gemm (matmul.hip) makes of a product: kept apart from the kernels so that the CPU can check it (tests/host/launch_rules.cpp).
#pragma once
#include <stdint.h>

#include <algorithm>
#include <cmath>

#include "../../include/caten_hip.h"

namespace cthip {

// Operands of the products: fp32, rounded to bf16, split in two / three bf16 terms (2^-16 / fp32-grade)
enum { GEMM_FP32 = 0, GEMM_BF16 = 1, GEMM_BF16X3 = 2, GEMM_BF16X6 = 3 };
struct TilePlan {
  int ks;     // workgroups that share the reduction axis
  double us;  // estimate
};

// How many workgroups share the reduction axis of a tile, and what the launch (with the one that adds the shares up) then takes, in microseconds:
// per round of tiles over an XCD a start and a time per step of 64, plus, where shares are added, a launch and their bytes (`deferred`: the bytes; the
// next launch adds them on its way).  Fitted to 1 .. 16 shares of 3800 products, from (16, 16, 100) to (1024, 12288, 4096): mean loss against the best share count 0.0 - 0.7 % a kernel,
// above 10 % in at most 3 of 217.  Two workgroups per compute unit of a tile, which filled the chip and was the rule before, took for 700^3 at two terms 14.0 us
// (one share: 9.8), 512^3 9.3 (8.2), 400 x 2304 x 768 Q8_0 24 (14: shares that an XCD has no room for), 70 x 1280 x 5120 23 (15).
// weights: the type of a weight matrix as the second operand, -1 for row-major floats.  On fp32 operands weights run k_gemm_f32 (no staging wavefronts: a step of
// 64 is 1.8 us, of k_gemm_f32pc 1.2; by that one's row 7.5 % lost, 64 rows of f32 11264 x 2048 74 us, now 43); at one term fp32 weights are the bytes that count.
inline TilePlan tile_plan(int M, int N, int K, int precision, int weights, bool aligned, bool deferred, int compute_units) {
  struct Cost {
    double start, step, unaligned;            // one round
    double start_n, step_n, unaligned_n;      // several: every compute unit at work
  };
  static const Cost costs[9] = {{1.0, 1.22, 1.55, 1.1, 1.05, 1.20}, {1.7, 0.37, 0.73, 1.15, 0.37, 0.50}, {1.2, 0.57, 0.86, 1.2, 0.53, 0.64}, {1.6, 0.85, 1.10, 3.0, 0.88, 0.98},
                                {0.6, 0.70, 0.70, 3.6, 0.60, 0.60}, {2.0, 0.72, 0.72, 2.0, 0.87, 0.87}, {2.0, 0.90, 0.90, 2.0, 1.10, 1.10},
                                {1.3, 1.78, 2.26, 0.95, 1.27, 1.45}, {0.55, 0.48, 0.48, 0.1, 0.48, 0.48}};
  // k_gemm_f32pc; k_gemm_split, one .. three terms; k_gemm_qpc, one .. three; k_gemm_f32; k_gemm_split, one term, fp32 weights
  const bool f32 = weights >= 0 && precision == GEMM_FP32, quant = !f32 && (weights == CTHIP_Q8_0 || weights == CTHIP_Q4_0);
  const int terms = precision == GEMM_FP32 ? 0 : precision == GEMM_BF16 ? 1 : precision == GEMM_BF16X3 ? 2 : 3;
  const Cost &c = costs[f32 ? 7 : quant ? 3 + terms : weights == CTHIP_F32 && terms == 1 ? 8 : terms];
  const bool two = !quant && terms != 3 && !f32;  // a second workgroup on a compute unit is that much of a round cheaper
  const int tm = (M + 63) / 64, tn = (N + (quant ? 127 : 63)) / (quant ? 128 : 64), nsteps = (K + 63) / 64;
  int64_t most = (int64_t)tm * tn;  // tiles of an XCD
  for (int rx = 1; rx <= 8; rx *= 2) most = std::min(most, (int64_t)((tm + rx - 1) / rx) * ((tn + 8 / rx - 1) / (8 / rx)));
  TilePlan best = {1, 1e30};
  for (int ks = 1; ks <= 16 && ks <= std::max(nsteps, 1); ks++) {
    const int steps = (nsteps + ks - 1) / ks, shares = steps ? (nsteps + steps - 1) / steps : 1;
    if (shares < ks) continue;  // the same steps as with fewer
    const double n = (double)(most * shares) * 8.0 / compute_units;
    // (Quantised tiles: no shares past one round.  Over 868 products that loses nothing, mean loss 0.6 % with them and without, at single ones up to 8 %, 203 x 12288 x 4096 107 us / 98;
    // and another order of a prompt's sums puts other quants into a Q8_0 cache, tokens a few steps on included.)
    if (quant && shares > 1 && n > 1.0) break;
    const double rounds = n <= 1.0 ? 1.0 : n <= 2.0 && two ? 1.85 : n <= 4.0 ? ceil(n) : 0.5 * ceil(2.0 * n);
    const double tile = n <= 1.0 ? c.start + (aligned ? c.step : c.unaligned) * steps : c.start_n + (aligned ? c.step_n : c.unaligned_n) * steps;
    const double sum = shares > 1 ? (deferred ? 0.3 : f32 ? 4.0 : 2.6) + (deferred ? 0.6e-6 : f32 ? 0.34e-6 : 0.85e-6) * 4.0 * shares * M * N : 0.0;
    const double us = 2.0 + rounds * tile + sum;
    if (us < best.us) best = {ks, us};
  }
  return best;
}

// ---- products whose operands lie in planes of bf16 terms (gemm_planes.hip) ----
inline int plane_terms(int precision) { return precision == GEMM_BF16X6 ? 3 : precision == GEMM_BF16X3 ? 2 : 1; }

// Which tile: the one whose rounds over the chip cost least.  A compute unit holds `resident` workgroups; alone a workgroup
// reaches `one`, together they reach `all` (TFLOP/s of results, measured at 1536^3, 2048^3 and 4096^3).
struct PlaneTile {
  int bm, bn, resident;
  double one, all;
  double idle = 1.0;  // share of a round's time that a single tile takes in the last one
};
inline double plane_tile_us(const PlaneTile &t, int M, int N, int nkb, int cus) {
  const int64_t tiles = (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn), slots = (int64_t)cus * t.resident;
  const double work = 2.0 * t.bm * t.bn * 32.0 * nkb * cus * 1e-6;  // MFLOP of a tile on every compute unit
  const int64_t full = tiles / slots, left = tiles - full * slots;
  double us = 2.0 + full * work * t.resident / t.all;
  if (t.resident == 1) us += (double)M * N * 4e-7;  // nothing runs under the stores (4500 x 4500 x 600 at one term: 63 us in tiles of 128, 73 of 256)
  if (left <= cus) {  // (a few tiles in the last round take less than a full round of them: `idle`)
    if (left) us += work / t.one * (full || t.resident == 1 ? t.idle + (1.0 - t.idle) * (double)left / cus : 1.0);
  } else {  // between one tile per compute unit and a full round, steeper at the start: the shared units wait for both
    const double one = work / t.one, all = work * t.resident / t.all;
    us += one + (all - one) * (0.4 + 0.6 * (double)(left - cus) / (double)(slots - cus));
  }
  return us;
}

struct PlanePick {
  int tile;   // of the list for the terms (planes_gemm)
  double us;  // estimate of the launch
};
// nkb: blocks of 32 k; ints_b: B is one plane of integers with scales
inline PlanePick plane_pick(int M, int N, int nkb, int terms, bool ints_b, int cus) {
  // one term: 4096^3 in tiles of 64 x 64 .. 256 x 256 337, 265, 209, 202, 160 us, 2048^3 56, 49, 45, 46, 72, 1536^3 34, 36, 37, 39, 61
  static const PlaneTile plane1[] = {{64, 64, 2, 330, 480, 0.5}, {128, 64, 3, 400, 650}, {128, 128, 2, 600, 880}, {128, 128, 2, 600, 922}, {256, 256, 1, 1290, 1290, 0.76}};
  // two: 4096^3 580, 428, 376, 357, 346 us, 2048^3 81, 70, 69, 77, 137, 1536^3 45, 47, 51, 55, 109
  static const PlaneTile plane[] = {{64, 64, 2, 200, 275, 0.5}, {128, 64, 3, 230, 365}, {128, 128, 2, 353, 438}, {128, 128, 2, 307, 469}, {256, 256, 1, 490, 490, 0.76}};
  // three: 3000 x 4100 x 5000 883, 795, 732, 4096^3 1026, 861, 655
  static const PlaneTile plane6[] = {{64, 64, 3, 110, 160}, {128, 64, 2, 110, 170}, {128, 256, 1, 205, 205, 0.6}};
  static const PlaneTile ints[] = {{64, 64, 4, 240, 245}, {128, 128, 2, 370, 400}, {128, 192, 2, 368, 430}};
  const PlaneTile *tiles = ints_b ? ints : terms == 3 ? plane6 : terms == 2 ? plane : plane1;
  const int n = ints_b || terms == 3 ? 3 : 5;
  PlanePick best = {0, 1e30};
  for (int i = 0; i < n; i++) {
    const double t = plane_tile_us(tiles[i], M, N, nkb, cus);
    if (t < best.us) best = {i, t};
  }
  return best;
}

// ---- Linears whose operands lie as 6-bit digits (gemm_digits.hip): tile and shares of K ----
struct DigitsPick {
  int tile, ks, fullest;  // tile: of the list; fullest: tiles of the fullest compute unit
  double us;              // of the launch, and with shares of what adds them up
};
// What the result is: rows of floats, rows as digits, SwiGLU of (gate, up) columns as digits (a wavefront's columns have to be whole blocks of results), or raw sums of a share of K
enum { kDigitsPlain = 0, kDigitsOut = 1, kDigitsOutPairs = 2, kDigitsShares = 3 };
// shares: whether K may be split (deferred: the launch behind adds the shares up on its way).  A launch is its ends and a time per block of 32 k of the fullest compute unit, us:
// `first` (and `filled` times the share of the compute units that have a tile: a step of 128 x 128 takes 0.34 us on 60 of them, 0.41 on 240), and `more` (`many` past two) for each
// further tile.  Fitted to weights out of memory: 64 x 64 / 64 x 128 / 128 x 128 for 100 x 3072 x 1024 10.0 / 12.3 / 18.5,
// 300 x 2560 x 2048 15.7 / 19.4 / 29.6, 200 x 11264 x 2048 34 / 28 / 33, 280 x 4096 x 4096 40 / 35 / 52, 1900 x 2048 x 5632 98 / 71 / 80, 1900 x 11264 x 2048 195 / 133 / 128.
inline DigitsPick digits_pick(int M, int N, int nkb, int out, bool shares, bool deferred, int cus) {
  static const struct {
    int bm, bn;
    double ends, first, filled, more, many;
  } tiles[] = {{64, 64, 4.4, 0.175, 0.0, 0.095, 0.14}, {64, 128, 5.0, 0.235, 0.0, 0.14, 0.18}, {128, 128, 7.6, 0.32, 0.10, 0.26, 0.30}};
  DigitsPick best = {1, 1, 1, 1e30};
  for (int ks = 1; ks <= (shares ? 8 : 1); ks++) {
    const int per = (nkb + ks - 1) / ks;
    if ((nkb + per - 1) / per != ks || (ks > 1 && per < 8)) continue;
    for (int t = out == kDigitsOutPairs ? 1 : 0; t < 3; t++) {
      const int64_t of_xcd = ((int64_t)((M + tiles[t].bm - 1) / tiles[t].bm) * ((N + tiles[t].bn - 1) / tiles[t].bn) + 7) / 8 * ks;
      const int fullest = (int)((of_xcd * 8 + cus - 1) / cus);
      const double us = tiles[t].ends + (out ? 2.5 : 0.0) + per * (tiles[t].first + tiles[t].filled * std::min(1.0, of_xcd * 8.0 / cus) + (fullest <= 2 ? tiles[t].more : tiles[t].many) * (fullest - 1)) +
                        (ks > 1 ? (deferred ? 0.3 : 2.6) + (deferred ? 0.6e-6 : 0.85e-6) * 4.0 * ks * M * N : 0.0);
      if (us < best.us) best = {t, ks, fullest, us};
    }
  }
  return best;
}

// Microseconds of a product (M, N, K) through planes: two passes over the operands (about 4.2 TB/s; none for operands that
// lie in planes already) and a denser GEMM.
inline double planes_us(int M, int N, int K, int terms, bool ints_b, double pass_bytes, int cus) {
  if ((int64_t)((K + 31) / 32) * 64 * 3 * 256 >= (1ll << 31)) return INFINITY;  // 32-bit offsets within a tile's rows
  const double us = plane_pick(M, N, (K + 31) / 32, terms, ints_b, cus).us;
  return (ints_b ? us * terms / 2.0 + 4.0 : us + 2.0) + (pass_bytes > 0 ? pass_bytes / 4.2e6 + 5.0 : 0.0);
}

// At sizes that the caches hold planes_us is off by what is put right here: fitted to both sides of 2280 products, a third of them with fewer than 500 k, from (200, 200, 64) to
// (5000, 5000, 5000), at one to three terms, rows of whole 16-byte pieces or not: mean loss against the faster side 0.5 - 0.7 %, above 10 % in 55.  (0.8 us + 8 and a sixth of the time that the
// result's bytes take, 4 % on top, whatever the terms: 0.5 - 1.8 %, 103; 3338 x 3584 x 116 at one term 27 us, now 21, 4452 x 2292 x 292 at three 83, now 70.)
inline bool matmul_planes_faster(int M, int N, int K, int precision, int cus) {
  if (precision == GEMM_FP32 || M < 64 || N < 64 || K < 64) return false;
  const int terms = plane_terms(precision);
  const bool aligned = K % 4 == 0 && N % 4 == 0;
  const double us = planes_us(M, N, K, terms, false, ((double)M + N) * K * (4 + 2 * terms), cus), out = 4e-6 * M * N;
  const double planes = aligned ? 0.83 * us + 8.0 : terms == 3 ? 0.95 * us + 8.0 : 0.94 * us + 10.4 + out / 4.0;
  return planes < tile_plan(M, N, K, precision, -1, aligned, false, cus).us;
}

// Linears over 4-bit weights at two terms: digits against tiles that convert their operands; shares: whether K may be split (no activation behind the sums).  x_bytes, w_bytes: what the
// passes move that write the rows' and the weights' digits (0: there already).  Over 17 matrices (768 x 768 .. 22016 x 4096), 64 .. 2000 rows, weights out of memory, with and without an
// activation: 0.5 % behind the faster side on average (shares taken for granted and a pass at 5 us + 4.2 TB/s: 2 %, and 1.5 times as long for 72 x 4096 x 11008 with an activation, 71 us
// for 48).
inline bool digits_fit(int K) { return (int64_t)(K / 32) * 4096 * 8 < (1ll << 31); }  // 32-bit offsets within a tile's rows
inline bool linear_digits_faster(int M, int N, int K, int type, double x_bytes, double w_bytes, bool shares, int cus) {
  const double us = digits_pick(M, N, K / 32, kDigitsPlain, shares, false, cus).us + (x_bytes > 0 ? x_bytes / 6e6 + 3.0 : 0.0) + (w_bytes > 0 ? w_bytes / 4.2e6 + 5.0 : 0.0);
  return us < tile_plan(M, N, K, GEMM_BF16X3, type, true, false, cus).us;
}

// The same for a Linear over weights (N, K).  planes_us and tile_plan are each off by what depends on the format: an integer or a half weight is fewer bytes for the tiles and one plane or
// two for the products, an fp32 one is split by every tile.  One ratio each, and planes no faster than 2.5 TB/s (64 rows of f16 22016 x 4096 112 us, in tiles 74), fitted to both sides of
// 3220 products (64 .. 2048 rows over (96, 4096) .. (22016, 4096), one to three terms, matrices out of the cache and out of memory): mean loss against the faster side 0.0 - 1.1 % a class.
// (With 1.04 for all, 0.92 of it for a few tiles of fp16, up to 7 %: fp32 4096 x 4096 over 900 rows 150 us, now 128, Q4_0 2560 x 2048 over 900 57 / 47, f16 at three terms
// 2048 x 2048 over 700 57 / 42.)  fp16 at two terms is where cache and memory part, 4 bytes a weight against 2: 1280 x 5120 over 900 rows, tiles / planes, 65 / 78 us out of the
// cache, 64 / 111 out of memory, 4800 x 1600 over 512 44 / 35 and 44 / 46; the ratio is right out of memory.
// prompt: in a session's prompt the weights come out of memory, what is in front writes planes, and behind tiles a norm adds the shares up: the older ratios, which were
// fitted there (by the others llama-1.1b f16 640 rows 5.4 -> 7.0 ms, q4_0 64 rows 1.63 -> 1.83, gpt2-medium q4_0 128 rows 1.50 -> 1.68).
inline bool linear_planes_faster(int M, int N, int K, int precision, int type, double pass_bytes, bool prompt, int cus) {
  static const double ratio[3][3] = {{0.84, 1.12, 1.20}, {0.84, 1.00, 0.88}, {0.84, 0.68, 1.0}};  // terms; fp32, fp16, integers
  const int terms = plane_terms(precision);
  const bool ints = type == CTHIP_Q8_0 || type == CTHIP_Q4_0;
  double us = planes_us(M, N, K, terms, ints, pass_bytes, cus);
  if (prompt) {
    // (fp16 tiles, two to a compute unit, are at their best while that is one round: prompts with them / planes, GPT-2 medium 300 rows 1.89 / 2.03 ms, large 256 rows
    // 3.16 / 3.48; 350 rows of the 1.1B shape 4.33 / 3.90)
    const int64_t tiles = (int64_t)((M + 63) / 64) * ((N + 63) / 64);
    us *= type != CTHIP_F16 ? 1.04 : tiles <= 2 * cus ? 1.4 : tiles <= 4 * cus ? 1.13 : 1.04;
  } else {
    const double plane_bytes = (double)N * ((K + 31) / 32) * 64 * (ints ? 1 : type == CTHIP_F16 && terms > 2 ? 2 : terms);
    us = std::max(us * ratio[terms - 1][ints ? 2 : type == CTHIP_F16 ? 1 : 0], plane_bytes / 2.5e6);
  }
  return us < tile_plan(M, N, K, precision, type, true, false, cus).us;
}

}  // namespace cthip
