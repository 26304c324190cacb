// The pieces of a copied row that the threads of a launch take (caten_amd/csrc/graph_plan.h): every element of a row once, nothing past it, at any size of launch.  Exit status 1
// and a line for every fault.
#include <stdio.h>

#include <vector>

#include "../../caten_amd/csrc/graph_plan.h"

using namespace cthip;

static int g_wrong = 0, g_walked = 0;

// what thread `tid` of workgroup `wg` stores of a row of n floats, as the kernel's loop has it
template <typename F>
static void walk(int64_t wg, int64_t nwg, int tid, int n, F store) {
  const GraphShare s = graph_share(wg, nwg, tid);
  g_walked++;
  if (s.first < n) store(s.first);
  for (int64_t t = s.first + s.step, k = 0; t < n; t += s.step)
    if (++k > n) {
      g_wrong++, printf("WRONG %lld workgroups, thread %d: no end\n", (long long)nwg, tid);
      return;
    } else {
      store(t);
    }
}

int main() {
  // small launches: all threads, rows shorter and longer than a piece for everyone
  for (int nwg : {1, 3, 12, 48})
    for (int n : {0, 4, 768, 1024, 4096, 4 * 256 * nwg, 4 * 256 * nwg + 4, 3 * 1024 * nwg + 20}) {
      std::vector<int> seen(n + 4, 0);
      for (int wg = 0; wg < nwg; wg++)
        for (int tid = 0; tid < kGraphAttnThreads; tid++)
          walk(wg, nwg, tid, n, [&](int64_t t) {
            if (t < 0 || t + 4 > n) g_wrong++, printf("WRONG %d workgroups, row of %d: piece at %lld\n", nwg, n, (long long)t);
            else seen[t]++;
          });
      for (int t = 0; t < n; t += 4)
        if (seen[t] != 1) g_wrong++, printf("WRONG %d workgroups, row of %d: piece %d stored %d times\n", nwg, n, t, seen[t]);
    }
  // large ones, up to the most batches and rows: no copy in front (n = 0) stores nothing, a short row is its first threads' and no one else's
  for (int64_t nwg : {(int64_t)1 << 19, ((int64_t)1 << 20) + 1, (int64_t)12 * 512 * 197, (int64_t)1 << 23, (int64_t)65535 * 65535})
    for (int n : {0, 768, 1 << 20})
      for (int64_t wg : {(int64_t)0, (int64_t)191, (int64_t)192, nwg / 2, nwg - 1})
        for (int tid : {0, 1, 127, 255})
          walk(wg, nwg, tid, n, [&](int64_t t) {
            if (t != 4 * (tid * nwg + wg) || t < 0 || t + 4 > n) g_wrong++, printf("WRONG %lld workgroups, row of %d, thread %d of %lld: piece at %lld\n", (long long)nwg, n, tid, (long long)wg, (long long)t);
          });
  printf("%d threads walked, %d wrong\n", g_walked, g_wrong);
  return g_wrong || !g_walked;
}
