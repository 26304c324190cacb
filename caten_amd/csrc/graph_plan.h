// Which pieces of a copied row a thread of k_graph_attn takes (graph_ops.hip): plain arithmetic, so that the host can walk it at any size of launch.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define CTHIP_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define CTHIP_HOST_DEVICE inline
#endif

namespace cthip {

// Pieces of four floats in turn over the workgroups: the first element of a thread's first piece, and how far its next one is.  (In 64 bits: a launch has up to 65535
// batches x 65535 rows workgroups, and with 2^20 + 1 of them the second piece of the last thread lies past 2^31.)
struct GraphShare {
  int64_t first, step;
};
constexpr int kGraphAttnThreads = 256;
CTHIP_HOST_DEVICE GraphShare graph_share(int64_t wg, int64_t nwg, int tid) { return {4 * (tid * nwg + wg), 4 * kGraphAttnThreads * nwg}; }

}  // namespace cthip
