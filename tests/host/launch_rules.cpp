// The rules that choose between launches (caten_amd/csrc/gemv_plan.h) against times of both sides, taken on the card: where one side is 4 % faster or more the
// rule has to take it.  Exit status 1 and a line for every one that it does not.
#include <stdio.h>

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

int main() {
  integer_gemv();
  printf("%d choices checked, %d wrong\n", g_checked, g_wrong);
  return g_wrong || !g_checked;
}
