// The rules that choose between launches (caten_amd/csrc/gemv_plan.h, gemm_plan.h) against times of both sides, taken on the card: where one side is 4 % faster or more the
// rule has to take it.  Exit status 1 and a line for every one that it does not.
#include <stdio.h>

#include "../../caten_amd/csrc/gemm_plan.h"
#include "../../caten_amd/csrc/gemv_plan.h"

using namespace cthip;

static int g_wrong = 0, g_checked = 0;
static void expect(const char *what, bool taken, bool want) {
  g_checked++;
  if (taken != want) g_wrong++, printf("WRONG %s: %s\n", what, taken ? "taken" : "not taken");
}

// single-row Linears on 4-bit weights, us: vector kernels, integer kernel; 256 compute units
static void integer_gemv() {
  static const struct {
    int rows, cols;
    double vec, integer;
  } t[] = {{4000, 4096, 6.3, 5.6}, {4352, 4096, 6.6, 7.5}, {4608, 4096, 6.6, 7.5}, {5120, 4096, 6.6, 7.6}, {5632, 4096, 7.1, 7.6}, {6656, 4096, 7.2, 7.8}, {9216, 4096, 8.3, 8.8},
           {12288, 4096, 10.1, 9.3}, {22016, 4096, 14.0, 12.7}, {4864, 3584, 6.3, 7.1}, {7168, 3584, 6.9, 7.2}, {10240, 3584, 8.9, 8.3}, {4608, 3072, 6.1, 6.5}, {5120, 2560, 5.9, 6.2},
           {5632, 2816, 6.5, 6.1}, {9216, 3968, 8.1, 9.4}, {13312, 3968, 10.2, 11.3}, {5120, 5120, 7.8, 8.0}, {9216, 6144, 11.3, 12.4}, {13312, 5760, 13.3, 15.6}, {17408, 6016, 15.8, 18.8},
           {12288, 6144, 13.1, 12.3}, {14336, 5120, 13.6, 13.0}, {50257, 5632, 33.2, 35.2}, {50257, 1280, 13.8, 9.3}, {5120, 10240, 15.2, 16.6}, {9216, 10240, 21.5, 22.4},
           {9216, 9728, 21.6, 20.6}, {5120, 6656, 11.5, 10.0}, {32000, 8192, 39.4, 35.0}, {2048, 4096, 5.1, 5.4}, {2560, 5632, 7.4, 6.4}, {4096, 11008, 12.5, 10.5}};
  for (const auto &c : t) {
    char what[96];
    snprintf(what, sizeof(what), "integer kernel for %d x %d (%.1f against %.1f us)", c.rows, c.cols, c.integer, c.vec);
    if (c.vec > 1.04 * c.integer || c.integer > 1.04 * c.vec) expect(what, gemv_int_pays(c.rows, c.cols, 256), c.integer < c.vec);
  }
}

// shares of K of a product of packed weights, us at 1, 2, 3, 4, 5, 6, 8, 10, 12, 16 of them (0: not timed): within 12 % of the best
static void shares_of_tiles() {
  static const int counts[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16};
  static const struct {
    int precision, type, m, rows, cols;
    double us[10];
  } t[] = {
      {0, CTHIP_F32, 64, 11264, 2048, {73.7, 54.8, 51.7, 43.5, 48.6, 49.8, 49.1, 48.8, 53.6, 62.2}},
      {0, CTHIP_Q8_0, 64, 11264, 2048, {71.6, 56.5, 52.4, 43.9, 49.0, 49.3, 47.5, 47.6, 50.8, 54.1}},
      {0, CTHIP_F32, 64, 4096, 4096, {133.6, 74.7, 54.9, 42.7, 42.1, 38.9, 32.4, 37.2, 34.7, 36.9}},
      {0, CTHIP_F32, 24, 4800, 1600, {56.5, 33.7, 25.8, 22.8, 21.7, 21.5, 20.1, 21.1, 20.8, 23.8}},
      {0, CTHIP_Q8_0, 100, 1280, 5120, {162.9, 91.7, 65.2, 50.6, 40.7, 38.6, 37.2, 32.8, 30.4, 31.5}},
      {0, CTHIP_F32, 48, 1600, 6400, {216.1, 113.3, 79.2, 60.0, 49.5, 43.3, 35.2, 36.3, 33.8, 29.0}},
      {0, CTHIP_F32, 180, 768, 3072, {102.8, 57.7, 41.0, 32.9, 28.9, 30.2, 25.7, 24.1, 25.7, 23.4}},
      {0, CTHIP_Q4_0, 100, 2048, 2048, {69.7, 40.0, 30.6, 24.9, 25.3, 26.6, 21.4, 21.2, 23.6, 25.5}},
      {0, CTHIP_F16, 256, 768, 768, {26.0, 17.8, 14.6, 13.6, 13.6, 14.4, 14.3, 14.3, 16.3, 0}},
      {0, CTHIP_F16, 24, 2048, 5632, {154.3, 82.2, 58.1, 44.5, 37.4, 32.2, 25.6, 30.3, 27.8, 23.1}},
      {0, CTHIP_F32, 700, 1024, 1024, {33.3, 32.0, 31.0, 27.4, 27.4, 31.4, 32.1, 31.9, 32.0, 37.8}},
      {0, CTHIP_Q8_0, 8, 1024, 4096, {125.8, 67.2, 48.1, 37.0, 31.7, 27.7, 22.2, 20.7, 19.0, 15.1}},
      {1, CTHIP_Q4_0, 100, 3072, 1024, {14.2, 12.3, 12.2, 11.7, 11.7, 15.4, 16.1, 16.0, 16.1, 22.2}},
      {1, CTHIP_Q4_0, 150, 2048, 1024, {14.2, 11.7, 11.0, 10.1, 10.1, 12.7, 13.1, 13.0, 13.0, 16.7}},
      {1, CTHIP_Q4_0, 300, 1024, 1024, {14.2, 12.4, 12.2, 11.8, 11.8, 12.7, 16.5, 16.5, 16.5, 20.6}},
      {1, CTHIP_Q4_0, 66, 12288, 4096, {44.6, 51.3, 53.3, 45.3, 49.9, 53.5, 54.9, 63.4, 69.0, 78.8}},
      {2, CTHIP_Q8_0, 100, 1280, 5120, {57.6, 34.0, 25.9, 21.5, 19.5, 18.3, 16.3, 16.1, 23.6, 20.7}},
      {2, CTHIP_Q8_0, 512, 768, 768, {11.7, 12.1, 11.6, 11.8, 11.8, 16.5, 16.4, 16.4, 21.7, 0}},
      {2, CTHIP_F16, 100, 1024, 4096, {33.6, 21.1, 16.8, 14.2, 13.1, 12.5, 12.0, 15.1, 14.6, 14.1}},
      {2, CTHIP_F16, 300, 2048, 2048, {19.2, 21.9, 19.1, 21.0, 22.0, 22.4, 23.2, 23.3, 28.1, 31.9}},
      {1, CTHIP_F32, 200, 1280, 1280, {13.9, 12.0, 11.4, 13.0, 13.2, 13.2, 15.1, 16.4, 16.4, 16.4}},
      {1, CTHIP_F32, 80, 2048, 1024, {9.7, 9.0, 8.6, 8.1, 8.2, 9.9, 8.9, 9.0, 8.9, 12.7}},
      {3, CTHIP_F32, 150, 2048, 5632, {69.1, 41.4, 54.2, 44.6, 39.4, 46.8, 40.5, 46.5, 50.4, 50.0}},
      {3, CTHIP_Q4_0, 100, 2048, 1024, {18.5, 14.1, 12.8, 11.5, 11.5, 11.2, 10.6, 10.6, 10.5, 15.9}},
  };
  for (const auto &c : t) {
    const int ks = tile_plan(c.m, c.rows, c.cols, c.precision, c.type, true, false, 256).ks, nsteps = (c.cols + 63) / 64;
    double best = 1e30, got = 1e30;
    for (int q = 0; q < 10; q++)
      if (c.us[q] > 0) {
        if (c.us[q] < best) best = c.us[q];
        if ((nsteps + counts[q] - 1) / counts[q] == (nsteps + ks - 1) / ks && c.us[q] < got) got = c.us[q];
      }
    if (got == 1e30) continue;  // a count that was not timed
    char what[128];
    snprintf(what, sizeof(what), "%d shares of %d x %d x %d, type %d, operands %d (%.1f against %.1f us)", ks, c.m, c.rows, c.cols, c.type, c.precision, got, best);
    expect(what, got <= 1.12 * best, true);
  }
}

// Linears over many rows (fp16 at two terms: out of memory), us: tiles that convert their operands, operands in planes (rows of the planes' passes that every call makes included)
static void linears_over_many_rows() {
  static const struct {
    int precision, type, m, rows, cols;
    double tiles, planes;
  } t[] = {
      {2, CTHIP_F16, 200, 2304, 768, 10.3, 15.9},
      {2, CTHIP_F16, 300, 1024, 1024, 12.0, 19.8},
      {2, CTHIP_F16, 200, 768, 3072, 13.5, 46.8},
      {2, CTHIP_F32, 900, 4096, 4096, 150.3, 128.5},
      {2, CTHIP_F32, 1600, 2048, 5632, 196.8, 146.1},
      {2, CTHIP_F32, 300, 2048, 2048, 21.3, 43.0},
      {2, CTHIP_F32, 2048, 768, 768, 18.3, 26.0},
      {2, CTHIP_F32, 900, 5632, 2048, 116.0, 89.9},
      {2, CTHIP_Q8_0, 1200, 5120, 1280, 64.0, 53.8},
      {2, CTHIP_Q8_0, 300, 6400, 1600, 44.9, 37.6},
      {2, CTHIP_Q8_0, 512, 768, 3072, 18.2, 35.4},
      {1, CTHIP_F16, 512, 1024, 4096, 19.6, 48.7},
      {1, CTHIP_F32, 512, 11264, 2048, 103.4, 63.9},
      {1, CTHIP_F32, 300, 1280, 5120, 26.4, 54.7},
      {1, CTHIP_Q8_0, 64, 12288, 4096, 29.5, 51.9},
      {1, CTHIP_Q8_0, 300, 1600, 6400, 31.5, 51.0},
      {3, CTHIP_F16, 700, 2048, 2048, 57.4, 42.2},
      {3, CTHIP_F16, 200, 768, 768, 9.9, 16.9},
      {3, CTHIP_F32, 2048, 3072, 3072, 304.5, 228.8},
      {3, CTHIP_F32, 200, 1280, 1280, 14.8, 34.2},
      {2, CTHIP_F16, 64, 22016, 4096, 73.5, 111.9},
      {2, CTHIP_F16, 64, 12288, 4096, 39.8, 95.7},
      {2, CTHIP_F16, 900, 1280, 5120, 64.0, 111.0},
      {2, CTHIP_F16, 640, 2048, 5632, 74.0, 122.0},
      {2, CTHIP_F16, 640, 11264, 2048, 123.1, 87.4},
      {2, CTHIP_F16, 1500, 4800, 1600, 107.1, 73.7},
      {2, CTHIP_F16, 640, 4800, 1600, 45.4, 51.9}};
  for (const auto &c : t) {
    const bool ints = c.type == CTHIP_Q8_0 || c.type == CTHIP_Q4_0;
    const int terms = plane_terms(c.precision), terms_b = ints ? 1 : c.type == CTHIP_F16 && terms > 2 ? 2 : terms;
    const bool stay = ints || (c.type == CTHIP_F16 && terms_b == 2);  // (gemm_planes.hip: weight_planes_stay)
    const double weights = (double)c.rows * c.cols;
    const double bytes = (double)c.m * c.cols * (4 + 2 * terms) + (stay ? 0.0 : weights * (c.type == CTHIP_F16 ? 2 : 4) + weights * 2 * terms_b);
    char what[96];
    snprintf(what, sizeof(what), "planes for %d rows of type %d %d x %d, %d terms (%.1f against %.1f us)", c.m, c.type, c.rows, c.cols, terms, c.planes, c.tiles);
    expect(what, linear_planes_faster(c.m, c.rows, c.cols, c.precision, c.type, bytes, false, 256), c.planes < c.tiles);
  }
}

// matrix products, us: tiles that convert their operands, operands in planes with the passes that make them
static void matrix_products() {
  static const struct {
    int precision, m, n, k;
    double tiles, planes;
  } t[] = {
      {1, 3338, 3584, 116, 28.5, 23.2},
      {1, 4124, 2716, 88, 27.2, 20.6},
      {2, 4124, 2716, 88, 31.5, 25.3},
      {2, 1992, 356, 480, 9.1, 17.8},
      {1, 4476, 1924, 1328, 85.4, 59.4},
      {3, 665, 933, 120, 7.2, 13.0},
      {3, 1317, 232, 221, 8.7, 13.7},
      {3, 4452, 2292, 292, 82.6, 70.0},
      {2, 2232, 1795, 459, 28.9, 41.0},
      {3, 1124, 1644, 476, 21.3, 27.7},
      {3, 1814, 885, 446, 22.0, 27.1},
      {1, 2988, 1092, 100, 11.1, 13.7},
      {2, 563, 461, 164, 7.1, 12.9},
      {2, 892, 761, 475, 10.9, 18.9},
      {1, 1789, 2401, 201, 18.6, 22.7},
      {1, 367, 251, 281, 8.4, 13.0},
      {1, 255, 397, 1685, 9.4, 30.0},
      {2, 2016, 1984, 4728, 160.5, 133.3},
      {3, 3792, 1168, 88, 25.9, 19.6},
      {2, 1084, 804, 3672, 57.4, 66.8},
      {2, 1740, 980, 1128, 25.3, 35.5},
      {2, 408, 536, 1968, 13.6, 41.7}};
  for (const auto &c : t) {
    char what[96];
    snprintf(what, sizeof(what), "planes for %d x %d x %d, operands %d (%.1f against %.1f us)", c.m, c.n, c.k, c.precision, c.planes, c.tiles);
    expect(what, matmul_planes_faster(c.m, c.n, c.k, c.precision, 256), c.planes < c.tiles);
  }
}

// Linears on 4-bit weights at two terms, us: tiles that convert their operands, 6-bit digits (the pass that writes the rows' included); shares of K where nothing but a bias follows, none
// behind an activation.  Sizes that the rule was not fitted to, but for the last: the side that it takes is within 9 % of the other.
static void digits_or_tiles() {
  static const struct {
    int m, n, k;
    bool shares;
    double tiles, digits;
  } t[] = {{80, 1536, 512, true, 8.9, 9.5}, {80, 1536, 512, false, 8.9, 11.9}, {170, 1536, 512, true, 10.5, 9.7}, {170, 1536, 512, false, 11.9, 12.2},
           {370, 1536, 512, true, 10.7, 10.1}, {370, 1536, 512, false, 12.1, 12.8}, {800, 1536, 512, true, 11.8, 12.8}, {800, 1536, 512, false, 13.2, 15.4},
           {1700, 1536, 512, true, 22.2, 16.2}, {1700, 1536, 512, false, 24.8, 21.2}, {80, 704, 2816, true, 12.0, 13.0}, {80, 704, 2816, false, 12.1, 23.9},
           {170, 704, 2816, true, 13.8, 15.1}, {170, 704, 2816, false, 14.0, 24.7}, {370, 704, 2816, true, 18.4, 19.1}, {370, 704, 2816, false, 18.5, 26.1},
           {800, 704, 2816, true, 28.6, 26.8}, {800, 704, 2816, false, 28.8, 29.4}, {1700, 704, 2816, true, 41.2, 35.6}, {1700, 704, 2816, false, 42.6, 40.0},
           {80, 2880, 960, true, 12.7, 12.0}, {80, 2880, 960, false, 12.8, 14.4}, {170, 2880, 960, true, 16.1, 12.6}, {170, 2880, 960, false, 17.4, 15.1},
           {370, 2880, 960, true, 17.2, 16.2}, {370, 2880, 960, false, 18.7, 21.1}, {800, 2880, 960, true, 32.8, 20.1}, {800, 2880, 960, false, 35.4, 25.0},
           {1700, 2880, 960, true, 53.4, 30.4}, {1700, 2880, 960, false, 57.8, 35.9}, {80, 3840, 1536, true, 15.2, 15.2}, {80, 3840, 1536, false, 15.4, 17.6},
           {170, 3840, 1536, true, 20.7, 16.4}, {170, 3840, 1536, false, 21.1, 19.1}, {370, 3840, 1536, true, 25.4, 21.6}, {370, 3840, 1536, false, 26.8, 26.6},
           {800, 3840, 1536, true, 50.3, 28.8}, {800, 3840, 1536, false, 53.8, 33.2}, {1700, 3840, 1536, true, 95.3, 49.9}, {1700, 3840, 1536, false, 99.4, 58.9},
           {80, 5376, 1344, true, 18.6, 14.5}, {80, 5376, 1344, false, 18.7, 17.0}, {170, 5376, 1344, true, 21.7, 15.8}, {170, 5376, 1344, false, 22.9, 18.5},
           {370, 5376, 1344, true, 42.1, 21.1}, {370, 5376, 1344, false, 45.0, 26.1}, {800, 5376, 1344, true, 63.4, 34.4}, {800, 5376, 1344, false, 67.3, 40.2},
           {1700, 5376, 1344, true, 107.3, 57.3}, {1700, 5376, 1344, false, 113.2, 66.2}, {80, 1792, 7168, true, 21.8, 20.8}, {80, 1792, 7168, false, 21.8, 49.1},
           {170, 1792, 7168, true, 29.0, 26.2}, {170, 1792, 7168, false, 29.4, 50.1}, {370, 1792, 7168, true, 56.8, 41.1}, {370, 1792, 7168, false, 55.4, 53.0},
           {800, 1792, 7168, true, 98.9, 68.8}, {800, 1792, 7168, false, 99.5, 73.9}, {1700, 1792, 7168, true, 182.5, 98.8}, {1700, 1792, 7168, false, 183.1, 101.7},
           {80, 6144, 2304, true, 25.2, 21.1}, {80, 6144, 2304, false, 25.4, 23.6}, {170, 6144, 2304, true, 33.4, 26.3}, {170, 6144, 2304, false, 34.7, 31.3},
           {370, 6144, 2304, true, 65.1, 33.4}, {370, 6144, 2304, false, 68.2, 37.9}, {800, 6144, 2304, true, 103.5, 56.4}, {800, 6144, 2304, false, 107.1, 60.1},
           {1700, 6144, 2304, true, 199.4, 94.3}, {1700, 6144, 2304, false, 207.1, 103.8}, {80, 8192, 3072, true, 31.7, 26.2}, {80, 8192, 3072, false, 31.8, 28.8},
           {170, 8192, 3072, true, 45.4, 33.3}, {170, 8192, 3072, false, 47.0, 38.3}, {370, 8192, 3072, true, 90.5, 45.5}, {370, 8192, 3072, false, 92.9, 50.3},
           {800, 8192, 3072, true, 178.1, 89.9}, {800, 8192, 3072, false, 182.4, 98.3}, {1700, 8192, 3072, true, 324.1, 166.2}, {1700, 8192, 3072, false, 328.4, 174.9}, {72, 4096, 11008, false, 48.0, 71.1}};
  for (const auto &c : t) {
    const bool digits = linear_digits_faster(c.m, c.n, c.k, CTHIP_Q4_0, (double)c.m * c.k * 8, 0.0, c.shares, 256);
    char what[128];
    snprintf(what, sizeof(what), "digits for %d rows of 4 bits %d x %d%s (%.1f against %.1f us)", c.m, c.n, c.k, c.shares ? "" : ", activation", c.digits, c.tiles);
    if (c.digits > 1.09 * c.tiles || c.tiles > 1.09 * c.digits) expect(what, digits, c.digits < c.tiles);
  }
}

// Their tiles, one share of K, us with 64 x 64, 64 x 128, 128 x 128: within 6 % of the best
static void tiles_of_digits() {
  static const struct {
    int m, n, k;
    double us[3];
  } t[] = {{80, 1536, 512, {9.5, 10.8, 14.0}}, {260, 1536, 512, {10.2, 11.5, 14.9}}, {520, 1536, 512, {10.7, 12.0, 15.3}}, {800, 1536, 512, {12.8, 12.7, 15.9}},
           {1100, 1536, 512, {13.7, 13.5, 16.5}}, {1700, 1536, 512, {17.6, 16.2, 18.0}}, {80, 704, 2816, {21.6, 26.3, 39.6}}, {260, 704, 2816, {23.3, 27.9, 41.1}},
           {520, 704, 2816, {24.4, 29.5, 42.3}}, {800, 704, 2816, {26.8, 32.3, 44.2}}, {1100, 704, 2816, {28.0, 32.9, 45.6}}, {1700, 704, 2816, {34.4, 35.5, 48.0}},
           {80, 2880, 960, {11.9, 14.0, 19.1}}, {260, 2880, 960, {13.3, 15.3, 20.7}}, {520, 2880, 960, {17.5, 17.5, 22.6}}, {800, 2880, 960, {23.2, 20.0, 24.9}},
           {1100, 2880, 960, {28.3, 22.6, 25.6}}, {1700, 2880, 960, {36.6, 30.2, 33.1}}, {80, 3840, 1536, {15.2, 18.1, 25.6}}, {260, 3840, 1536, {20.1, 20.6, 28.4}},
           {520, 3840, 1536, {30.0, 25.6, 31.3}}, {800, 3840, 1536, {37.7, 28.5, 34.0}}, {1100, 3840, 1536, {47.1, 38.7, 42.2}}, {1700, 3840, 1536, {66.0, 50.8, 49.8}},
           {80, 5376, 1344, {14.5, 17.1, 23.7}}, {260, 5376, 1344, {19.6, 19.7, 26.9}}, {520, 5376, 1344, {29.3, 25.7, 30.1}}, {800, 5376, 1344, {41.5, 34.5, 38.8}},
           {1100, 5376, 1344, {51.6, 39.6, 42.7}}, {1700, 5376, 1344, {74.8, 57.6, 58.4}}, {80, 1792, 7168, {47.0, 56.5, 90.7}}, {260, 1792, 7168, {49.5, 58.9, 91.4}},
           {520, 1792, 7168, {55.9, 63.1, 94.7}}, {800, 1792, 7168, {70.6, 69.1, 97.9}}, {1100, 1792, 7168, {84.8, 78.2, 100.3}}, {1700, 1792, 7168, {120.3, 98.3, 112.0}},
           {80, 6144, 2304, {21.1, 24.3, 35.4}}, {260, 6144, 2304, {31.1, 28.9, 39.7}}, {520, 6144, 2304, {54.2, 39.5, 46.3}}, {800, 6144, 2304, {68.5, 56.7, 59.6}},
           {1100, 6144, 2304, {92.1, 68.9, 68.0}}, {1700, 6144, 2304, {129.8, 99.5, 94.4}}, {80, 8192, 3072, {26.5, 31.0, 45.0}}, {260, 8192, 3072, {53.1, 43.0, 52.0}},
           {520, 8192, 3072, {85.1, 69.3, 76.0}}, {800, 8192, 3072, {115.8, 90.5, 89.8}}, {1100, 8192, 3072, {153.1, 117.3, 111.8}}, {1700, 8192, 3072, {224.0, 165.8, 161.5}}};
  for (const auto &c : t) {
    const int tile = digits_pick(c.m, c.n, c.k / 32, kDigitsPlain, false, false, 256).tile;
    char what[96];
    snprintf(what, sizeof(what), "digits of %d x %d x %d: tile %d takes %.1f us", c.m, c.n, c.k, tile, c.us[tile]);
    expect(what, c.us[tile] <= 1.06 * std::min(c.us[0], std::min(c.us[1], c.us[2])), true);
  }
}

// Their shares of K, us at 1, 2, 3, 4, 6, 8 of them: within 12 % of the best; a count that was not timed lies between two that are
static void shares_of_digits() {
  static const int counts[] = {1, 2, 3, 4, 6, 8};
  static const struct {
    int m, n, k;
    double us[6];
  } t[] = {{80, 704, 2816, {21.6, 17.3, 15.2, 14.0, 13.3, 12.9}}, {170, 704, 2816, {22.3, 18.3, 16.4, 15.3, 15.1, 16.2}}, {370, 704, 2816, {23.5, 20.9, 19.1, 20.3, 19.7, 21.6}},
           {800, 704, 2816, {26.8, 28.3, 25.7, 26.4, 26.2, 26.9}}, {80, 3840, 1536, {15.2, 15.8, 16.4, 16.5, 18.1, 18.3}},
           {170, 3840, 1536, {16.4, 20.9, 21.9, 22.6, 25.2, 19.2}}, {370, 3840, 1536, {20.5, 28.4, 29.1, 27.5, 31.5, 21.7}},
           {800, 3840, 1536, {28.5, 40.3, 42.4, 46.3, 52.1, 28.8}}, {80, 1792, 7168, {47.0, 31.8, 25.9, 23.1, 22.5, 20.7}},
           {170, 1792, 7168, {47.9, 33.3, 31.9, 28.0, 27.7, 26.8}}, {370, 1792, 7168, {50.7, 44.3, 40.7, 39.3, 44.3, 38.9}},
           {800, 1792, 7168, {69.1, 61.9, 66.8, 62.0, 65.7, 67.1}}, {80, 6144, 2304, {21.1, 23.1, 23.2, 23.3, 25.3, 25.4}},
           {170, 6144, 2304, {26.1, 30.5, 27.9, 29.3, 31.4, 35.8}}, {370, 6144, 2304, {33.4, 41.2, 42.7, 44.8, 50.3, 56.4}},
           {800, 6144, 2304, {56.7, 70.3, 75.1, 80.8, 91.7, 106.0}}};
  for (const auto &c : t) {
    const int ks = digits_pick(c.m, c.n, c.k / 32, kDigitsPlain, true, false, 256).ks;
    double best = 1e30, got = 0.0;
    for (int q = 0; q < 6; q++) {
      best = std::min(best, c.us[q]);
      if (counts[q] <= ks) got = c.us[q];
      if (counts[q] >= ks && (q == 0 || counts[q - 1] < ks)) got = std::max(got, c.us[q]);
    }
    char what[96];
    snprintf(what, sizeof(what), "%d shares of digits of %d x %d x %d (%.1f against %.1f us)", ks, c.m, c.n, c.k, got, best);
    expect(what, got <= 1.12 * best, true);
  }
}

int main() {
  integer_gemv();
  digits_or_tiles();
  tiles_of_digits();
  shares_of_digits();
  shares_of_tiles();
  linears_over_many_rows();
  matrix_products();
  printf("%d choices checked, %d wrong\n", g_checked, g_wrong);
  return g_wrong || !g_checked;
}
