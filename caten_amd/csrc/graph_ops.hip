// The small operations of a compiled graph's forward, several to a launch.
//
// A decode step of a compiled GPT-2 is 150 operations of 1 - 5 us; what bounds it is the host issuing them one by one (3.5 us
// each, the device waits) and, behind that, the 2.3 us a launch takes however little it does.  The walk of a forward
// (vm.hip) therefore queues operations whose addresses are known, and three kinds of neighbours share a launch:
//   * copies that do not touch each other's memory (the two cache assignments of a layer);
//   * scores -> softmax -> values [-> copy of the result]: a workgroup takes one row of one batch through all of them;
//   * a LayerNorm and the Linear over few rows that reads it: the Linear's workgroups normalise the row themselves.
// Every operation's result is still written where its own launch would have written it: a fused launch leaves the same
// buffers behind.  Anything else runs as before, in order.  GPT-2 small, 12 steps from a 16-token prompt: 7.3 -> 6.1 ms, the host
// 520 -> 250 us a step; what is left is the device's: 66 launches that are each a few round trips to memory.
#include <stdint.h>
#include <string.h>

#include <vector>

#include "graph_ops.h"

namespace cthip {

int matmul_routed(float *C, const float *A, const float *B, int M, int N, int K, int act, const float *bias, const float *residual, bool b_is_nk);

static thread_local std::vector<GraphOp> *t_queue = nullptr;
GraphCollector::GraphCollector() { t_queue = new std::vector<GraphOp>(); }
GraphCollector::~GraphCollector() {
  delete t_queue;
  t_queue = nullptr;
}
bool graph_ops_collecting() { return t_queue != nullptr; }

// ---- kernels ----
constexpr int kMaxCopies = 4;
struct CopyBatch {
  CopyArgs c[kMaxCopies];
  int first[kMaxCopies + 1];  // blocks [first[q], first[q + 1]) work on copy q
  bool vec[kMaxCopies];       // four elements of the innermost axis at a time
  int n;
};
__global__ __launch_bounds__(256) void k_copies(CopyBatch cb) {
  int q = 0;
  while (q + 1 < cb.n && (int)blockIdx.x >= cb.first[q + 1]) q++;
  const CopyArgs &c = cb.c[q];
  const int v = cb.vec[q] ? 4 : 1, e2 = c.ext[2] / v;
  const int64_t i = (int64_t)((int)blockIdx.x - cb.first[q]) * 256 + threadIdx.x;
  if (i >= (int64_t)c.ext[0] * c.ext[1] * e2) return;
  const int64_t i2 = i % e2 * v, r = i / e2, i1 = r % c.ext[1], i0 = r / c.ext[1];
  const float *s = c.in + i0 * c.is[0] + i1 * c.is[1] + i2 * c.is[2];
  float *o = c.out + i0 * c.os[0] + i1 * c.os[1] + i2 * c.os[2];
  if (cb.vec[q]) *(float4 *)o = *(const float4 *)s;
  else *o = *s;
}

// One row of one batch: scores (bmm.hip's KC layout), softmax, values (NC layout), copy.  Sums as in k_bmm.  The row's scores stay in
// LDS; a 12-head step at position 30: 8 us instead of six launches of 2.6 - 4.8, every one of them behind the host.
struct GraphAttn {
  BmmArgs s, v;
  float *probs;
  float *copy;               // null: no copy behind it
  int64_t cb, ci, cj;        // its strides per batch, row, column
  // copies of a contiguous row in front (a step's new key and value rows): the workgroups share them, and whoever needs a
  // key of the copied row reads it at its source
  float *pre_out[2];
  const float *pre_in[2];
  int pre_n[2];
};
constexpr int kGraphAttnMaxKeys = 2048;
__global__ __launch_bounds__(256) void k_graph_attn(GraphAttn a) {
  __shared__ float sc[kGraphAttnMaxKeys];
  __shared__ float4 part[16][16];
  __shared__ float red[8];
  const int tid = threadIdx.x, i = blockIdx.x, lane = tid & 63, wv = tid >> 6, c = tid & 15, g = tid >> 4;
  int bz = blockIdx.y;
  const int b2 = bz % a.s.nb[2];
  bz /= a.s.nb[2];
  const int b1 = bz % a.s.nb[1], b0 = bz / a.s.nb[1];
  auto off = [&](const BmmOperand &o) { return o.base + (int64_t)b0 * o.sb[0] + (int64_t)b1 * o.sb[1] + (int64_t)b2 * o.sb[2]; };
  const int N = a.s.N, K = a.s.K;
  const float *A = a.s.A + off(a.s.a) + (int64_t)i * a.s.a.si, *KB = a.s.B + off(a.s.b), *VB = a.v.B + off(a.v.b);
  auto at = [&](const float *p) __attribute__((always_inline)) {  // where what belongs at p can be read now
    const int64_t d0 = p - a.pre_out[0], d1 = p - a.pre_out[1];
    return d0 >= 0 && d0 < a.pre_n[0] ? a.pre_in[0] + d0 : d1 >= 0 && d1 < a.pre_n[1] ? a.pre_in[1] + d1 : p;
  };
  float4 vw[4];
  {
    // the first keys' values are asked for ahead of the scores: they arrive behind them
#pragma unroll
    for (int u = 0; u < 4; u++) vw[u] = *(const float4 *)at(VB + (int64_t)min(g + 16 * u, N - 1) * a.v.b.sk + (4 * c < a.v.N ? 4 * c : 0));
    // four passes of 16 keys asked for together (64-wide heads: one piece of each key per lane)
    const float *p0 = a.s.pre0 ? a.s.pre0 + off(a.s.p0) + (int64_t)i * a.s.p0.si : A, *p1 = a.s.pre1 ? a.s.pre1 + off(a.s.p1) + (int64_t)i * a.s.p1.si : A;
    const int64_t s0 = a.s.pre0 ? a.s.p0.sj : 0, s1 = a.s.pre1 ? a.s.p1.sj : 0;
    float *Crow = a.s.C + off(a.s.c) + (int64_t)i * a.s.c.si;
    for (int j0 = 0; j0 < N; j0 += 64) {
      float acc[4], e0[4], e1[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int j = min(j0 + 16 * u + g, N - 1);
        e0[u] = p0[j * s0];
        e1[u] = p1[j * s1];
      }
#pragma unroll
      for (int u = 0; u < 4; u++) acc[u] = 0.0f;
      for (int k0 = 4 * c; k0 < K; k0 += 64) {
        float4 w[4];
#pragma unroll
        for (int u = 0; u < 4; u++) w[u] = *(const float4 *)at(KB + (int64_t)min(j0 + 16 * u + g, N - 1) * a.s.b.sj + k0);
        const float4 x = *(const float4 *)(A + k0);
#pragma unroll
        for (int u = 0; u < 4; u++) {
          acc[u] = fmaf(x.x, w[u].x, acc[u]);
          acc[u] = fmaf(x.y, w[u].y, acc[u]);
          acc[u] = fmaf(x.z, w[u].z, acc[u]);
          acc[u] = fmaf(x.w, w[u].w, acc[u]);
        }
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int j = j0 + 16 * u + g;
        acc[u] = row16_sum(acc[u]);
        if (c == 0 && j < N) {
          float v = a.s.alpha * acc[u];
          if (a.s.pre0) v += e0[u];
          if (a.s.pre1) v += e1[u];
          Crow[j] = v;
          sc[j] = v;
        }
      }
    }
  }
  __syncthreads();
  float m = -INFINITY;
  for (int j = tid; j < N; j += 256) m = fmaxf(m, sc[j]);
  m = wave_max(m);
  if (lane == 0) red[wv] = m;
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float l = 0.0f;
  for (int j = tid; j < N; j += 256) {
    const float e = ct_exp(sc[j] - m);
    sc[j] = e;
    l += e;
  }
  l = wave_sum(l);
  if (lane == 0) red[4 + wv] = l;
  __syncthreads();
  const float inv = 1.0f / ((red[4] + red[5]) + (red[6] + red[7]));
  float *P = a.probs + off(a.v.a) + (int64_t)i * a.v.a.si;
  for (int j = tid; j < N; j += 256) {
    const float p = sc[j] * inv;
    sc[j] = p;
    P[j] = p;
  }
  __syncthreads();
  float *C = a.v.C + off(a.v.c) + (int64_t)i * a.v.c.si;
  float *Y = a.copy ? a.copy + (int64_t)blockIdx.y * a.cb + (int64_t)i * a.ci : nullptr;
  for (int d0 = 0; d0 < a.v.N; d0 += 64) {
    const int j4 = d0 + 4 * c;
    const bool live = j4 < a.v.N;
    const int jc = live ? j4 : 0;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int k0 = g; k0 < N; k0 += 64) {
      float4 w[4];
      if (k0 == g && d0 == 0) {
#pragma unroll
        for (int u = 0; u < 4; u++) w[u] = vw[u];
      } else {
#pragma unroll
        for (int u = 0; u < 4; u++) w[u] = *(const float4 *)at(VB + (int64_t)min(k0 + 16 * u, N - 1) * a.v.b.sk + jc);
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const float x = k0 + 16 * u < N ? sc[k0 + 16 * u] : 0.0f;
        acc.x = fmaf(x, w[u].x, acc.x);
        acc.y = fmaf(x, w[u].y, acc.y);
        acc.z = fmaf(x, w[u].z, acc.z);
        acc.w = fmaf(x, w[u].w, acc.w);
      }
    }
    part[g][c] = acc;
    __syncthreads();
    if (g == 0 && live) {
      float4 s = part[0][c];
#pragma unroll
      for (int q = 1; q < 16; q++) {
        const float4 t = part[q][c];
        s.x += t.x;
        s.y += t.y;
        s.z += t.z;
        s.w += t.w;
      }
      const float o[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const float v = a.v.alpha * o[q];
        C[(int64_t)(j4 + q) * a.v.c.sj] = v;
        if (Y) Y[(int64_t)(j4 + q) * a.cj] = v;
      }
    }
    __syncthreads();
  }
  // (the copies last: in front, everything else waited for their round trip to memory: 9.3 -> 8.1 us a launch of a 12-head step at position 27)
#pragma unroll
  for (int q = 0; q < 2; q++)
    for (int t = 4 * ((blockIdx.y * gridDim.x + blockIdx.x) * 256 + tid); t < a.pre_n[q]; t += 1024 * gridDim.x * gridDim.y)
      *(float4 *)(a.pre_out[q] + t) = *(const float4 *)(a.pre_in[q] + t);
}

// ---- what a chain may touch ----
struct Span {
  const char *lo, *hi;
};
static Span span(const float *p, std::initializer_list<std::pair<int64_t, int64_t>> axes) {  // (extent, stride) of every axis
  int64_t lo = 0, hi = 0;
  for (const auto &ax : axes) {
    const int64_t s = (ax.first - 1) * ax.second;
    if (s < 0) lo += s;
    else hi += s;
  }
  return {(const char *)(p + lo), (const char *)(p + hi + 1)};
}
static Span bmm_span(const BmmArgs &a, const float *p, const BmmOperand &o) {
  return span(p + o.base, {{a.nb[0], o.sb[0]}, {a.nb[1], o.sb[1]}, {a.nb[2], o.sb[2]}, {a.M, o.si}, {a.N, o.sj}, {a.K, o.sk}});
}
static Span rows_span(const float *p, long long rows, long long n) { return {(const char *)p, (const char *)(p + rows * n)}; }
static bool apart(const Span &a, const Span &b) { return a.hi <= b.lo || b.hi <= a.lo; }
static Span copy_span(const CopyArgs &c, bool out) {
  return out ? span(c.out, {{c.ext[0], c.os[0]}, {c.ext[1], c.os[1]}, {c.ext[2], c.os[2]}}) : span(c.in, {{c.ext[0], c.is[0]}, {c.ext[1], c.is[1]}, {c.ext[2], c.is[2]}});
}

// ---- launches ----
static int run_one(const GraphOp &op);
static int64_t copy_blocks(const CopyArgs &c, bool vec) { return ((int64_t)c.ext[0] * c.ext[1] * (c.ext[2] / (vec ? 4 : 1)) + 255) / 256; }
static bool copy_vec(const CopyArgs &c) {
  return c.os[2] == 1 && c.is[2] == 1 && c.ext[2] % 4 == 0 && c.os[0] % 4 == 0 && c.os[1] % 4 == 0 && c.is[0] % 4 == 0 && c.is[1] % 4 == 0 &&
         (((uintptr_t)c.out | (uintptr_t)c.in) & 15) == 0;
}
static int run_copies(const GraphOp *ops, int n) {
  CopyBatch cb;
  cb.n = n;
  cb.first[0] = 0;
  for (int q = 0; q < n; q++) {
    cb.c[q] = ops[q].copy;
    cb.vec[q] = copy_vec(cb.c[q]);
    cb.first[q + 1] = cb.first[q] + (int)copy_blocks(cb.c[q], cb.vec[q]);
  }
  if (cb.first[n] == 0) return 0;
  hipLaunchKernelGGL(k_copies, dim3(cb.first[n]), dim3(256), 0, state().stream, cb);
  CTHIP_LAUNCH_CHECK();
  return 0;
}

// [up to two copies,] scores, softmax, values [, a copy]; returns how many were launched, 0 = not this chain
static int run_attention(const GraphOp *ops, int left, int &rc) {
  int npre = 0;
  while (npre < left && npre < 2 && ops[npre].kind == GraphOp::COPY) npre++;
  const GraphOp *pre = ops;
  ops += npre;
  left -= npre;
  if (left < 3 || ops[0].kind != GraphOp::BMM || ops[1].kind != GraphOp::SOFTMAX || ops[2].kind != GraphOp::BMM) return 0;
  const BmmArgs &s = ops[0].bmm, &v = ops[2].bmm;
  const int64_t nb = (int64_t)s.nb[0] * s.nb[1] * s.nb[2];
  if (bmm_variant(s) != 1 || bmm_variant(v) != 2 || memcmp(s.nb, v.nb, sizeof(s.nb)) || s.M != v.M || s.N != v.K || s.N > kGraphAttnMaxKeys) return 0;
  if (s.post || s.act != CTHIP_ACT_NONE || v.pre0 || v.pre1 || v.post || v.act != CTHIP_ACT_NONE) return 0;
  // scores and probabilities as rows in order: [batch][row][key]
  auto rows = [&](const BmmOperand &o, int64_t inner) {
    return o.si == s.N && inner == 1 && (s.nb[2] == 1 || o.sb[2] == (int64_t)s.M * s.N) && (s.nb[1] == 1 || o.sb[1] == (int64_t)s.nb[2] * s.M * s.N) &&
           (s.nb[0] == 1 || o.sb[0] == (int64_t)s.nb[1] * s.nb[2] * s.M * s.N);
  };
  if (!rows(s.c, s.c.sj) || !rows(v.a, v.a.sk)) return 0;
  if (ops[1].x != s.C + s.c.base || ops[1].out != v.A + v.a.base || ops[1].rows != nb * s.M || ops[1].n != s.N) return 0;
  const Span outs[3] = {bmm_span(s, s.C, s.c), rows_span(ops[1].out, nb * s.M, s.N), bmm_span(v, v.C, v.c)};
  const Span ins[5] = {bmm_span(s, s.A, s.a), bmm_span(s, s.B, s.b), bmm_span(v, v.B, v.b),
                       s.pre0 ? bmm_span(s, s.pre0, s.p0) : Span{nullptr, nullptr}, s.pre1 ? bmm_span(s, s.pre1, s.p1) : Span{nullptr, nullptr}};
  for (int p = 0; p < 3; p++) {
    for (const Span &in : ins)
      if (in.lo && !apart(outs[p], in)) return 0;
    for (int q = 0; q < p; q++)
      if (!apart(outs[p], outs[q])) return 0;
  }
  GraphAttn a = {};
  a.s = s;
  a.v = v;
  a.probs = ops[1].out - v.a.base;  // (the kernel adds v.a's offsets)
  int used = 3;
  if (left > 3 && ops[3].kind == GraphOp::COPY) {
    // the copy walks the result's batches, rows and columns, in whatever order
    const CopyArgs &c = ops[3].copy;
    int axis[3] = {-1, -1, -1};  // batch, row, column
    const int64_t want_ext[3] = {nb, s.M, v.N}, want_st[3] = {(int64_t)v.M * v.N, v.c.si, v.c.sj};
    bool ok = c.in == v.C + v.c.base && v.c.si == v.N && v.c.sj == 1 &&
              (v.nb[2] == 1 || v.c.sb[2] == want_st[0]) && (v.nb[1] == 1 || v.c.sb[1] == v.nb[2] * want_st[0]) && (v.nb[0] == 1 || v.c.sb[0] == (int64_t)v.nb[1] * v.nb[2] * want_st[0]);
    bool taken[3] = {false, false, false};
    for (int w = 0; w < 3 && ok; w++) {
      for (int q = 0; q < 3; q++)
        if (!taken[q] && c.ext[q] == want_ext[w] && (c.is[q] == want_st[w] || want_ext[w] == 1)) {
          axis[w] = q;
          taken[q] = true;
          break;
        }
      ok = axis[w] >= 0;
    }
    const Span co = copy_span(c, true);
    for (const Span &in : ins) ok = ok && (!in.lo || apart(co, in));
    for (const Span &o : outs) ok = ok && apart(co, o);
    if (ok) {
      a.copy = c.out;
      a.cb = c.os[axis[0]];
      a.ci = c.os[axis[1]];
      a.cj = c.os[axis[2]];
      used = 4;
    }
  }
  if (npre) {
    // what they write may be read by the chain as keys and values, in whole pieces of four; nothing else may meet it
    for (int q = 0; q < npre; q++) {
      const CopyArgs &c = pre[q].copy;
      if (c.ext[0] != 1 || c.ext[1] != 1 || c.os[2] != 1 || c.is[2] != 1 || c.ext[2] % 4 || (((uintptr_t)c.out | (uintptr_t)c.in) & 15)) return 0;
      const Span w = copy_span(c, true), r = copy_span(c, false);
      for (const Span &o : outs)
        if (!apart(o, w) || !apart(o, r)) return 0;
      if (used == 4) {
        const Span o = copy_span(ops[3].copy, true);
        if (!apart(o, w) || !apart(o, r)) return 0;
      }
      if (!apart(w, ins[0]) || (ins[3].lo && !apart(w, ins[3])) || (ins[4].lo && !apart(w, ins[4]))) return 0;
      for (int p = 0; p < npre; p++)
        if (!apart(w, copy_span(pre[p].copy, false)) || (p < q && !apart(w, copy_span(pre[p].copy, true)))) return 0;
      a.pre_out[q] = c.out;
      a.pre_in[q] = c.in;
      a.pre_n[q] = c.ext[2];
    }
  }
  hipLaunchKernelGGL(k_graph_attn, dim3(s.M, (unsigned)nb), dim3(256), 0, state().stream, a);
  const hipError_t e = hipGetLastError();
  rc = e == hipSuccess ? 0 : fail((int)e, "graph: launch -> %s", hipGetErrorString(e));
  return npre + used;
}

// LayerNorm at ops[0], the Linear over its (few) rows at ops[1]
static bool run_norm_linear(const GraphOp *ops, int left, int &rc) {
  if (left < 2 || ops[0].kind != GraphOp::LAYERNORM || ops[1].kind != GraphOp::LINEAR) return false;
  const GraphOp &n = ops[0], &l = ops[1];
  if (l.x != n.out || l.rows != n.rows || l.n != n.n || l.rows < 1 || l.rows > 2 || n.n % 4 || n.n > 4096 || (!l.bias && !l.resid)) return false;
  WMat w = {};
  w.type = CTHIP_F32;
  w.rows = l.cols;
  w.cols = l.n;
  w.q = const_cast<float *>(l.w);
  w.q_bytes = (int64_t)l.cols * l.n * 4;
  if (!gemv_norm_out_ok(&w)) return false;
  for (const void *p : {(const void *)n.x, (const void *)n.g, (const void *)n.b, (const void *)n.out})
    if ((uintptr_t)p & 15) return false;
  const Span y = rows_span(l.out, l.rows, l.cols), no = rows_span(n.out, n.rows, n.n), x = rows_span(n.x, n.rows, n.n);
  if (!apart(y, no) || !apart(y, x) || !apart(no, x)) return false;
  const Span reads[5] = {n.g ? rows_span(n.g, 1, n.n) : x, n.b ? rows_span(n.b, 1, n.n) : x, rows_span(l.w, l.cols, l.n), l.bias ? rows_span(l.bias, 1, l.cols) : x,
                         l.resid ? rows_span(l.resid, l.rows, l.cols) : x};
  for (int q = 0; q < 5; q++)
    if (!apart(no, reads[q]) || (q < 4 && !apart(y, reads[q]))) return false;  // (a residual may be the result itself)
  GemvArgs a = {};
  a.y = l.out;
  a.x = n.x;
  a.bias = l.bias;
  a.residual = l.resid;
  a.act = l.act;
  a.pro = CTHIP_PRO_LAYERNORM;
  a.norm_g = n.g;
  a.norm_b = n.b;
  a.eps = n.eps;
  a.norm_out = n.out;
  a.x_stride = l.n;
  a.y_stride = l.cols;
  rc = launch_gemv(&w, a, (int)l.rows);
  return true;
}

static int run_one(const GraphOp &op) {
  switch (op.kind) {
    case GraphOp::BMM: return launch_bmm(op.bmm);
    case GraphOp::SOFTMAX: return cthip_softmax(op.out, op.x, op.rows, op.n);
    case GraphOp::LAYERNORM: return cthip_layernorm(op.out, op.x, op.g, op.b, op.eps, op.rows, op.n);
    case GraphOp::LINEAR: return matmul_routed(op.out, op.x, op.w, (int)op.rows, op.cols, op.n, op.act, op.bias, op.resid, true);
    case GraphOp::COPY: return run_copies(&op, 1);
  }
  return fail(CTHIP_E_STATE, "graph: unknown operation");
}

int graph_ops_flush() {
  if (!t_queue || t_queue->empty()) return 0;
  std::vector<GraphOp> ops;
  ops.swap(*t_queue);
  int rc = 0;
  for (size_t k = 0; k < ops.size() && !rc;) {
    const int left = (int)(ops.size() - k);
    const int used = run_attention(&ops[k], left, rc);
    if (used) {
      k += used;
    } else if (run_norm_linear(&ops[k], left, rc)) {
      k += 2;
    } else if (ops[k].kind == GraphOp::COPY) {
      int n = 1;
      for (; n < left && n < kMaxCopies && ops[k + n].kind == GraphOp::COPY; n++) {
        bool ok = true;
        const Span o = copy_span(ops[k + n].copy, true), i = copy_span(ops[k + n].copy, false);
        for (int q = 0; q < n && ok; q++)
          ok = apart(o, copy_span(ops[k + q].copy, true)) && apart(o, copy_span(ops[k + q].copy, false)) && apart(i, copy_span(ops[k + q].copy, true));
        if (!ok) break;
      }
      rc = run_copies(&ops[k], n);
      k += n;
    } else {
      rc = run_one(ops[k]);
      k++;
    }
  }
  ops.clear();
  if (t_queue->capacity() == 0) t_queue->swap(ops);  // keep the storage
  return rc;
}
int graph_op(const GraphOp &op) {
  if (!t_queue) return run_one(op);
  t_queue->push_back(op);
  // issue while the walk goes on: nothing that could join a chain is pending behind the last of these
  const bool open = op.kind == GraphOp::LAYERNORM || op.kind == GraphOp::BMM || op.kind == GraphOp::SOFTMAX || op.kind == GraphOp::COPY;
  return open && t_queue->size() < 16 ? 0 : graph_ops_flush();
}

}  // namespace cthip
