// Small operations of a graph forward, collected so that chains of them run as one launch (graph_ops.hip).
#pragma once
#include "common.h"

namespace cthip {

struct CopyArgs {  // out[ob + sum i_q os_q] = in[ib + sum i_q is_q], i_q < ext_q; the last axis is the innermost
  float *out;
  const float *in;
  int ext[3];
  int64_t os[3], is[3];  // (bases are already in the pointers)
};

struct GraphOp {
  enum Kind { BMM, SOFTMAX, LAYERNORM, LINEAR, COPY } kind;
  BmmArgs bmm;
  CopyArgs copy;
  // SOFTMAX / LAYERNORM: out (rows, n) = f(x); LINEAR: out (rows, cols) = act(x (rows, n) . w^T + bias) + resid
  float *out;
  const float *x, *w, *g, *b, *bias, *resid;
  float eps;
  long long rows;
  int n, cols, act;
};

// While a collector is open on this thread an operation is queued; else it is launched at once.
int graph_op(const GraphOp &op);
int graph_ops_flush();                 // launches what is queued, fused where a chain allows it (nothing queued: 0)
bool graph_ops_collecting();
struct GraphCollector {                // open for the walk of one forward; its flush is the caller's
  GraphCollector();
  ~GraphCollector();
};
}  // namespace cthip
