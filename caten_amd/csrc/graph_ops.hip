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
#include "graph_plan.h"

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
// (What the kernel is told is what it needs and no more: a round of scalar loads is 0.2 us in front of everything else, and two descriptions of whole products were
// eight of them.)
struct GraphRows {  // where an operand's row of a batch begins: elements per step of a batch axis, per row
  int64_t at, sb[3], si;
};
struct GraphAttn {
  const float *Q, *K, *V, *M0, *M1;  // M0, M1: addends of the scores (none: the queries' first element, with strides of 0)
  GraphRows q, k, v, m0, m1;
  int64_t k_sj, v_sk, m0_sj, m1_sj;
  int N, Kd, Nv;             // keys, elements of a key, of a value
  int nb1;
  unsigned inv_nb1;          // 2^32 / nb1, rounded up: quotients of numbers below 2^16
  bool has0, has1;
  float s_alpha, v_alpha;
  float *S, *probs, *C;
  GraphRows s, p, c;
  int64_t c_sj;
  float *copy;               // null: no copy behind it
  int64_t cb, ci, cj;        // its strides per batch, row, column
  // copies of a contiguous row in front (a step's new key and value rows): the workgroups share them, and whoever needs a
  // key of the copied row reads it at its source
  float *pre_out[2];
  const float *pre_in[2];
  int pre_n[2];
};
constexpr int kGraphAttnMaxKeys = 2048;
__global__ __launch_bounds__(kGraphAttnThreads) void k_graph_attn(GraphAttn a) {
  __shared__ float sc[kGraphAttnMaxKeys];
  __shared__ float4 part[16][16];
  __shared__ float red[8];
  const int tid = threadIdx.x, i = blockIdx.x, lane = tid & 63, wv = tid >> 6, c = tid & 15, g = tid >> 4;
  const int b2 = blockIdx.y, b0 = a.nb1 > 1 ? (int)__umulhi(blockIdx.z, a.inv_nb1) : (int)blockIdx.z, b1 = (int)blockIdx.z - b0 * a.nb1;
  auto off = [&](const GraphRows &o) { return o.at + (int64_t)b0 * o.sb[0] + (int64_t)b1 * o.sb[1] + (int64_t)b2 * o.sb[2] + (int64_t)i * o.si; };
  // (one wait for all of what the first loads' addresses are made of)
  const float *Qp = a.Q, *Kp = a.K, *Vp = a.V;
  GraphRows rq = a.q, rk = a.k, rv = a.v;
  int64_t k_sj = a.k_sj, v_sk = a.v_sk;
  int N = a.N, K = a.Kd, Nv = a.Nv;
  asm volatile(""
               : "+s"(Qp), "+s"(Kp), "+s"(Vp), "+s"(rq.at), "+s"(rq.sb[0]), "+s"(rq.sb[1]), "+s"(rq.sb[2]), "+s"(rq.si), "+s"(rk.at), "+s"(rk.sb[0]), "+s"(rk.sb[1]),
                 "+s"(rk.sb[2]), "+s"(rv.at), "+s"(rv.sb[0]), "+s"(rv.sb[1]), "+s"(rv.sb[2]), "+s"(k_sj), "+s"(v_sk), "+s"(N), "+s"(K), "+s"(Nv));
  typedef const __attribute__((address_space(1))) float *gfloat;
  typedef float f4 __attribute__((ext_vector_type(4)));
  typedef const __attribute__((address_space(1))) f4 *gfloat4;
  const gfloat A = (gfloat)(Qp + off(rq)), KB = (gfloat)(Kp + off(rk)), VB = (gfloat)(Vp + off(rv));
  // what belongs at p, from where it can be read now.  (Selects, not branches: behind a branch every load was waited for by itself, eight round trips in front
  // of the first score; a launch of a 12-head step at position 27, 8.5 -> 5 us.)
  const uint64_t o0 = (uint64_t)a.pre_out[0], o1 = (uint64_t)a.pre_out[1], m0 = (uint64_t)a.pre_in[0] - o0, m1 = (uint64_t)a.pre_in[1] - o1;
  const uint64_t n0 = 4ull * a.pre_n[0], n1 = 4ull * a.pre_n[1];
  auto at = [&](gfloat p) __attribute__((always_inline)) {
    const uint64_t x = (uint64_t)p;
    const bool in0 = x - o0 < n0, in1 = x - o1 < n1;
    const uint64_t lo = in0 ? m0 : in1 ? m1 : 0;
    const f4 t = *(gfloat4)(x + lo);
    return make_float4(t[0], t[1], t[2], t[3]);
  };
  // Asked for in front of any arithmetic, in the order of use: four passes of 16 keys together (64-wide heads: one piece of each key per lane), the addends, the
  // same keys' values, and one piece a thread of the copies in front, the workgroups in turn.
  const gfloat p0 = (gfloat)(a.M0 + off(a.m0)), p1 = (gfloat)(a.M1 + off(a.m1));
  float *Crow = a.S + off(a.s);
  float4 kw[4], vw[4], cw[2];
  float e0[4], e1[4];
  auto addends = [&](int j0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int j = min(j0 + 16 * u + g, N - 1);
      e0[u] = p0[j * a.m0_sj];
      e1[u] = p1[j * a.m1_sj];
    }
  };
  auto keys = [&](int j0, int k0, float4 *w) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4; u++) w[u] = at(KB + (int64_t)min(j0 + 16 * u + g, N - 1) * k_sj + k0);
  };
  const int kc = 4 * c < K ? 4 * c : 0;
  const GraphShare mine = graph_share(((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x, (int64_t)gridDim.x * gridDim.y * gridDim.z, tid);
  const f4 x0 = *(gfloat4)(A + kc);
  keys(0, kc, kw);
  __builtin_amdgcn_sched_barrier(0);
  addends(0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < 4; u++) vw[u] = at(VB + (int64_t)min(g + 16 * u, N - 1) * v_sk + (4 * c < Nv ? 4 * c : 0));
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const f4 t = *(gfloat4)(mine.first < a.pre_n[q] ? (gfloat)a.pre_in[q] + mine.first : A);
    cw[q] = make_float4(t[0], t[1], t[2], t[3]);
  }
  __builtin_amdgcn_sched_barrier(0);
  auto pass = [&](int j0) __attribute__((always_inline)) {
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    auto dot = [&](const f4 &x, const float4 *w) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < 4; u++) {
        acc[u] = fmaf(x.x, w[u].x, acc[u]);
        acc[u] = fmaf(x.y, w[u].y, acc[u]);
        acc[u] = fmaf(x.z, w[u].z, acc[u]);
        acc[u] = fmaf(x.w, w[u].w, acc[u]);
      }
    };
    if (4 * c < K) dot(x0, kw);
    for (int k0 = 4 * c + 64; k0 < K; k0 += 64) {
      float4 w[4];
      keys(j0, k0, w);
      const f4 x = *(gfloat4)(A + k0);
      dot(x, w);
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int j = j0 + 16 * u + g;
      acc[u] = row16_sum(acc[u]);
      if (c == 0 && j < N) {
        float v = a.s_alpha * acc[u];
        if (a.has0) v += e0[u];
        if (a.has1) v += e1[u];
        Crow[j] = v;
        sc[j] = v;
      }
    }
  };
  pass(0);  // (not in the loop: at its top the wait for the first keys would be one for everything that has been asked for)
  for (int j0 = 64; j0 < N; j0 += 64) {
    keys(j0, kc, kw);
    addends(j0);
    pass(j0);
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
  float *P = a.probs + off(a.p);
  for (int j = tid; j < N; j += 256) {
    const float p = sc[j] * inv;
    sc[j] = p;
    P[j] = p;
  }
  __syncthreads();
  float *C = a.C + off(a.c);
  float *Y = a.copy ? a.copy + (int64_t)(blockIdx.z * gridDim.y + blockIdx.y) * a.cb + (int64_t)i * a.ci : nullptr;
  for (int d0 = 0; d0 < Nv; d0 += 64) {
    const int j4 = d0 + 4 * c;
    const bool live = j4 < Nv;
    const int jc = live ? j4 : 0;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int k0 = g; k0 < N; k0 += 64) {
      float4 w[4];
      if (k0 == g && d0 == 0) {
#pragma unroll
        for (int u = 0; u < 4; u++) w[u] = vw[u];
      } else {
#pragma unroll
        for (int u = 0; u < 4; u++) w[u] = at(VB + (int64_t)min(k0 + 16 * u, N - 1) * v_sk + jc);
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
        const float v = a.v_alpha * o[q];
        C[(int64_t)(j4 + q) * a.c_sj] = v;
        if (Y) Y[(int64_t)(j4 + q) * a.cj] = v;
      }
    }
    __syncthreads();
  }
  // (the copies' first pieces, one to a thread and the workgroups in turn, were asked for with the first values: a round trip to memory less at the end)
#pragma unroll
  for (int q = 0; q < 2; q++) {
    if (mine.first < a.pre_n[q]) *(float4 *)(a.pre_out[q] + mine.first) = cw[q];
    for (int64_t t = mine.first + mine.step; t < a.pre_n[q]; t += mine.step) *(float4 *)(a.pre_out[q] + t) = *(const float4 *)(a.pre_in[q] + t);
  }
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
  auto rows_of = [](const BmmOperand &o) { return GraphRows{o.base, {o.sb[0], o.sb[1], o.sb[2]}, o.si}; };
  auto whole = [&](const BmmOperand &o) {  // (all rows of a batch are read)
    GraphRows r = rows_of(o);
    r.si = 0;
    return r;
  };
  a.Q = s.A, a.K = s.B, a.V = v.B, a.S = s.C, a.C = v.C;
  a.q = rows_of(s.a), a.k = whole(s.b), a.v = whole(v.b), a.s = rows_of(s.c), a.p = rows_of(v.a), a.c = rows_of(v.c);
  a.k_sj = s.b.sj, a.v_sk = v.b.sk, a.c_sj = v.c.sj;
  a.has0 = s.pre0 != nullptr, a.has1 = s.pre1 != nullptr;
  a.M0 = a.has0 ? s.pre0 : s.A, a.M1 = a.has1 ? s.pre1 : s.A;
  if (a.has0) a.m0 = rows_of(s.p0), a.m0_sj = s.p0.sj;
  else a.m0.at = s.a.base;
  if (a.has1) a.m1 = rows_of(s.p1), a.m1_sj = s.p1.sj;
  else a.m1.at = s.a.base;
  a.N = s.N, a.Kd = s.K, a.Nv = v.N, a.s_alpha = s.alpha, a.v_alpha = v.alpha;
  a.nb1 = s.nb[1], a.inv_nb1 = s.nb[1] > 1 ? (unsigned)((0x100000000ull + s.nb[1] - 1) / s.nb[1]) : 0u;
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
  hipLaunchKernelGGL(k_graph_attn, dim3(s.M, (unsigned)s.nb[2], (unsigned)(s.nb[0] * s.nb[1])), dim3(kGraphAttnThreads), 0, state().stream, a);
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
