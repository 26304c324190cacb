// What launch_gemm (matmul.hip) makes of a product: kept apart from the kernels so that the CPU can check it (tests/host/launch_rules.cpp).
#pragma once
#include <algorithm>
#include <cmath>

namespace cthip {

// Operands of the products: fp32, rounded to bf16, split in two / three bf16 terms (2^-16 / fp32-grade)
enum { GEMM_FP32 = 0, GEMM_BF16 = 1, GEMM_BF16X3 = 2, GEMM_BF16X6 = 3 };
struct TilePlan {
  int ks;     // workgroups that share the reduction axis
  double us;  // estimate
};

// How many workgroups share the reduction axis of a tile, and what the launch (with the one that adds the shares up) then takes, in microseconds:
// per round of tiles over an XCD a start and a time per step of 64, plus, where shares are added, a launch and their bytes (`deferred`: the bytes; the
// next launch adds them on its way).  Fitted to 1 .. 8 shares of 20 shapes from (20, 232, 144) to (512, 2048, 5632), to which it keeps
// within 15 %.  Two workgroups per compute unit of a tile, which filled the chip and was the rule before, took for 700^3 at two terms 14.0 us
// (one share: 9.8), 512^3 9.3 (8.2), 400 x 2304 x 768 Q8_0 24 (14: shares that an XCD has no room for), 70 x 1280 x 5120 23 (15).
// packed: the second operand is a weight matrix, which fp32 operands meet in k_gemm_f32 (no staging wavefronts: a step of 64 is 1.8 us, of k_gemm_f32pc 1.2).  Its row
// is fitted to 1 .. 16 shares of 1050 products, f32 / f16 / Q8_0 / Q4_0 weights of (96, 4096) .. (12288, 4096) over 8 .. 1024 rows: mean loss against the best
// share count 1 %, above 10 % in 4; by k_gemm_f32pc's row 7.5 %, above 10 % in 326 (64 rows f32 11264 x 2048 74 us, now 43), by shares that fill the chip 12 %.
inline TilePlan tile_plan(int M, int N, int K, int precision, bool packed, bool quant, bool aligned, bool deferred, int compute_units) {
  struct Cost {
    double start, step, unaligned;            // one round
    double start_n, step_n, unaligned_n;      // several: every compute unit at work
  };
  static const Cost costs[8] = {{1.0, 1.22, 1.55, 1.1, 1.05, 1.20}, {1.7, 0.37, 0.73, 1.15, 0.37, 0.50}, {1.2, 0.57, 0.86, 1.2, 0.53, 0.64},
                                {1.6, 0.85, 1.10, 3.0, 0.88, 0.98}, {2.0, 0.55, 0.55, 2.0, 0.66, 0.66}, {2.0, 0.72, 0.72, 2.0, 0.87, 0.87},
                                {2.0, 0.90, 0.90, 2.0, 1.10, 1.10},   // k_gemm_f32pc; k_gemm_split, one .. three terms; k_gemm_qpc, one .. three
                                {1.3, 1.78, 2.26, 0.95, 1.27, 1.45}};  // k_gemm_f32
  const bool f32 = packed && precision == GEMM_FP32;
  const Cost &c = costs[f32 ? 7 : precision == GEMM_FP32 ? 0 : (quant ? 3 : 0) + (precision == GEMM_BF16 ? 1 : precision == GEMM_BF16X3 ? 2 : 3)];
  const bool two = !quant && precision != GEMM_BF16X6 && !f32;  // a second workgroup on a compute unit is that much of a round cheaper
  const int tm = (M + 63) / 64, tn = (N + (quant ? 127 : 63)) / (quant ? 128 : 64), nsteps = (K + 63) / 64;
  int64_t most = (int64_t)tm * tn;  // tiles of an XCD
  for (int rx = 1; rx <= 8; rx *= 2) most = std::min(most, (int64_t)((tm + rx - 1) / rx) * ((tn + 8 / rx - 1) / (8 / rx)));
  TilePlan best = {1, 1e30};
  for (int ks = 1; ks <= 16 && ks <= std::max(nsteps, 1); ks++) {
    const int steps = (nsteps + ks - 1) / ks, shares = steps ? (nsteps + steps - 1) / steps : 1;
    if (shares < ks) continue;  // the same steps as with fewer
    const double n = (double)(most * shares) * 8.0 / compute_units;
    // (shares of quantised tiles only where compute units are left for them: in a second round they gain 8 % at the most, 203 x 12288 x 4096 107 -> 98 us,
    // and reorder the sums of a prompt, which a Q8_0 cache answers with other quants)
    if (quant && shares > 1 && n > 1.0) break;
    const double rounds = n <= 1.0 ? 1.0 : n <= 2.0 && two ? 1.85 : n <= 4.0 ? ceil(n) : 0.5 * ceil(2.0 * n);
    const double tile = n <= 1.0 ? c.start + (aligned ? c.step : c.unaligned) * steps : c.start_n + (aligned ? c.step_n : c.unaligned_n) * steps;
    const double sum = shares > 1 ? (deferred ? 0.3 : f32 ? 4.0 : 2.6) + (deferred ? 0.6e-6 : f32 ? 0.34e-6 : 0.85e-6) * 4.0 * shares * M * N : 0.0;
    const double us = 2.0 + rounds * tile + sum;
    if (us < best.us) best = {ks, us};
  }
  return best;
}

}  // namespace cthip
