// Single-row Linear on 4-bit quantised rows, multiplied as integers on the matrix cores.
//
// The vector kernels (gemv_kernels.h, gemv_wide.hip) spend 2.4 - 7.8 vector instructions on a weight -- a conversion, a
// multiply-add, their share of the prologue -- which at one wavefront per SIMD is as much time as the weights take to arrive.
// Here the input vector is written as four signed base-256 digits per element (30 bits below the largest value of its chunk, the block of 32
// that meets 16 bytes of weights, with a power of two for each; all bits there are where fewer than 30 lie above the smallest float), nibbles go to v_mfma_i32_16x16x64_i8 as bytes (one or two
// bit operations per four of them), and the products and their sums over a chunk are exact integers:
//   sum q x = 2^e (((i0 256 + i1) 256 + i2) 256 + i3),  i_r = sum over the chunk of q * digit r.
// Digits are the rows of the first operand, weight rows the columns of the second: lane l holds 16 bytes of weight row l % 16, the (l / 16)-th chunk of
// an instruction, and only rows 4 (l / 16) + r of that chunk's k carry digit r (the other twelve are zeros), so that lane l of the
// result holds the four digit sums of its own row and chunk -- the chunk whose scale it has fetched.  25 vector instructions per
// 2048 weights.  (8-bit rows arrive no faster than the vector kernels multiply them: 12288 x 4096 15.0 us this way, 14.4 theirs.)
//
// K is shared among the ks wavefronts of a workgroup (a unit of 128 bytes of each of 16 rows at a time, whole cache lines of
// a row), rgp such sets work on neighbouring groups of 16 rows; a workgroup goes over its groups with PD units in flight per
// wavefront and meets once, for the sums of them all.  What bounds it: the weights, behind 3 us of launch, the vector's way into LDS and the meeting at
// the end (22016 x 4096, 50.7 MB: 12.9 us, 4096 x 11008, 25.4 MB: 8.6, 4096 x 4096, 9.4 MB: 5.4).  Everything in front of the stream is instructions that sixteen wavefronts share four
// issue slots for, and any wait there is one in front of the weights: with addresses per lane, divisions for the share of the rows and a common block of zeros whose address had to
// be fetched for every unit, the three were 13.3, 10.4 and 6.2 us.  Errors against 64 bits, 4096 columns: 0.6 - 1.2e-7; the vector kernels, which take nibbles times
// inputs less eight times the inputs' sum, 2 - 5e-7.
#include "common.h"
#include "gemv_int.h"
#include "gemv_kernels.h"
#include "gemv_plan.h"

namespace cthip {

struct GemvIntShape {
  int upw, ks, rgp;        // units per wavefront and group; wavefronts sharing a group; groups a workgroup works on together
  int inv_ks, inv_rows;    // 65536 / ks, 65536 / (16 rgp), rounded up: quotients of numbers below 1024
  int grid, full, rest;    // workgroups; every one goes over `full` groups of 16 rgp rows, the first `rest` over one more
};

// CENTRED: the mean of a LayerNorm comes off the vector before its digits are made, not off the sums behind them
template <int PRO, bool CENTRED, bool NT>
__global__ __launch_bounds__(1024) void k_gemv_int(GemvArgs a, GemvIntShape sh) {
  constexpr int PD = 2;              // units in flight per wavefront (four: no faster stream, 0.8 us more code to get through)
  constexpr bool RMS = PRO == CTHIP_PRO_RMSNORM, LAYERNORM = PRO == CTHIP_PRO_LAYERNORM;
  constexpr int CB = 128;            // bytes of digits per chunk: [half of its k][digit][16 bytes]
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, i = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), sub = (wv * sh.inv_ks) >> 16, wk = wv - sub * sh.ks, nw = sh.ks * sh.rgp, nthr = 64 * nw;
  const int nchunks = a.cols >> 5, n4 = a.cols >> 2;
  const int cpad = sh.ks * sh.upw * 8;  // chunks that the wavefronts go over: zeros past the row
  // LDS: 256 bytes of zeros, digits, a scale per chunk, reductions, the groups' partial sums
  unsigned char *dig = smem + 256;
  float *sx = (float *)(dig + (size_t)cpad * CB), *red = sx + cpad, *ps = red + 32;
  const int m = blockIdx.y;
  const float *__restrict__ x = a.x + (int64_t)m * a.x_stride;
  const int rows_sg = 16 * sh.rgp, iters = sh.full + ((int)blockIdx.x < sh.rest ? 1 : 0);

  // ---- the row this thread finishes (the plan: no more of them than threads), and what it needs for that ----
  const int oj = (tid * sh.inv_rows) >> 16, oi = tid - oj * rows_sg, orow = ((int)blockIdx.x + oj * sh.grid) * rows_sg + oi;
  const int orc = min(orow, a.rows - 1);

  // ---- the input vector is asked for, then the first units of weights ----
  constexpr int SB = 3;
  const float4 *x4 = (const float4 *)x;
  const float4 *u4 = (RMS || LAYERNORM) && a.norm_g ? (const float4 *)a.norm_g : x4;
  float4 xv[SB], uv[SB];
#pragma unroll
  for (int b = 0; b < SB; b++) {
    const unsigned k = 16u * (unsigned)min(tid + nthr * b, n4 - 1);
    xv[b] = *(const float4 *)((const char *)x4 + k);
    if (RMS || LAYERNORM) uv[b] = *(const float4 *)((const char *)u4 + k);
  }
  // (what is not there is read as the vector's first element and counts as nothing.  Not a block of zeros of the program's: its address comes out of memory by itself, and
  // a wavefront that picks between that and another stands still for it -- in front of the first weights and again at every unit: see `request`)
  typedef const __attribute__((address_space(1))) float *gfloat;  // (a flat load would be waited for with everything behind it)
  auto opt = [&](const float *p, int64_t off) __attribute__((always_inline)) { return ((p ? (gfloat)p : (gfloat)x) + (p ? off : 0))[p ? (unsigned)orc : 0u]; };
  const float rb = opt(a.bias, 0), rr = opt(a.residual, (int64_t)m * a.y_stride), rf = LAYERNORM ? opt(a.fold_s, 0) : 0.0f;

  uint4 wt[PD][2];
  unsigned st[PD];  // the scales of both chunks
  const int nu = iters * sh.upw;  // units of this wavefront
  int rq_j = 0, rq_u = 0;         // the next one to ask for
  auto request = [&](int p) __attribute__((always_inline)) {
    const bool past = rq_j >= iters;  // (uniform) nothing left: the matrix's first bytes, never used
    const int row0 = past ? 0 : min(((int)blockIdx.x + rq_j * sh.grid) * rows_sg + 16 * sub, a.rows - 1);
    // chunks 2g and 2g + 1 of the unit: both loads of a wavefront touch the same lines, the scales are one load
    // (nchunks is even; past the row: its last two chunks again, against zeros)
    const int c0 = min((wk * sh.upw + rq_u) * 8 + 2 * g, nchunks - 2);
    // offsets from the group's first row, which is the same for the wavefront: 16 rows of at most 2^20 columns
    const unsigned off = past ? 0u : (unsigned)(min(i, a.rows - 1 - row0) * nchunks + c0);
    const char *q0 = (const char *)a.q + (int64_t)row0 * nchunks * 16, *d0 = (const char *)a.d + (int64_t)row0 * nchunks * 2;
#pragma unroll
    for (int s = 0; s < 2; s++) wt[p][s] = load_chunk<NT>((const uint4 *)(q0 + 16u * off) + s);
    st[p] = *(const unsigned *)(d0 + 2u * off);
    if (++rq_u == sh.upw) rq_u = 0, rq_j++;
  };
#pragma unroll
  for (int p = 0; p < PD; p++) request(p);
  __builtin_amdgcn_sched_barrier(0);
  const int posv = a.pos ? a.pos[0] : 0;

  // ---- digits ----
  float s1 = 0.0f, mu = 0.0f, rstd = 1.0f;
  if (tid < 64) ((unsigned *)smem)[tid] = 0u;
  auto of_all = [&](const float *p, int stride, int n) __attribute__((always_inline)) {  // p[0] + p[stride] + ..., n <= 16, all asked for together
    float t[16], v = 0.0f;
#pragma unroll
    for (int w = 0; w < 16; w++) t[w] = p[min(w, n - 1) * stride];
#pragma unroll
    for (int w = 0; w < 16; w++) v += w < n ? t[w] : 0.0f;
    return v;
  };
  if (CENTRED) {
    auto add = [&](const float4 &t) __attribute__((always_inline)) { s1 += (t.x + t.y) + (t.z + t.w); };
#pragma unroll
    for (int b = 0; b < SB; b++)
      if (tid + nthr * b < n4) add(xv[b]);
    for (int k = tid + nthr * SB; k < n4; k += nthr) add(x4[k]);
    s1 = wave_sum(s1);
    if (lane == 0) red[wv] = s1;
    __syncthreads();
    mu = of_all(red, 1, nw) / (float)a.cols;
    s1 = 0.0f;
  }
  auto put = [&](int k, const unsigned *w, float down) __attribute__((always_inline)) {  // digits of k = 4 k .. + 3: [16 k][digit][16 bytes]
    int_digits_put(dig, sx, k, w, down);
  };
  for (int k = n4 + tid; k < cpad * 8; k += nthr) {  // past the row
    const unsigned z[4] = {0u, 0u, 0u, 0u};
    put(k, z, 0.0f);
  }
  auto piece = [&](int k, const float4 &x0, const float4 &u0) __attribute__((always_inline)) {  // (a chunk's lanes stay together: n4 is a multiple of eight)
    float v[4] = {x0.x, x0.y, x0.z, x0.w};
    const float u[4] = {u0.x, u0.y, u0.z, u0.w};
#pragma unroll
    for (int e = 0; e < 4; e++) {
      if (CENTRED) v[e] -= mu;
      else if (LAYERNORM) s1 += v[e];
      if (RMS || CENTRED) s1 = fmaf(v[e], v[e], s1);
      if ((RMS || LAYERNORM) && a.norm_g) v[e] *= u[e];
    }
    unsigned w[4];
    const float down = int_digits(v, w);
    put(k, w, down);
  };
  // (what has been asked for stays out of the loop over the rest: behind a way back the wait for it would be one for the weights as well)
#pragma unroll
  for (int b = 0; b < SB; b++)
    if (tid + nthr * b < n4) piece(tid + nthr * b, xv[b], uv[b]);
  for (int k = tid + nthr * SB; k < n4; k += nthr) {
    const float4 t = x4[k];
    piece(k, t, RMS || LAYERNORM ? u4[k] : t);
  }
  if (RMS || LAYERNORM) {
    s1 = wave_sum(s1);
    if (lane == 0) red[CENTRED ? 16 + wv : wv] = s1;
  }
  __syncthreads();
  if (LAYERNORM && !CENTRED) {  // the deviations from the mean: the vector once more (it is in the caches; the weights are on their way)
    mu = of_all(red, 1, nw) / (float)a.cols;
    float q = 0.0f;
    for (int k = tid; k < n4; k += nthr) {
      const float4 t = x4[k];
      const float d0 = t.x - mu, d1 = t.y - mu, d2 = t.z - mu, d3 = t.w - mu;
      q = fmaf(d0, d0, fmaf(d1, d1, fmaf(d2, d2, fmaf(d3, d3, q))));
    }
    q = wave_sum(q);
    if (lane == 0) red[16 + wv] = q;  // (read behind the barrier after the stream)
  }

  // ---- stream ----
  const bool act = (i >> 2) == g;  // this lane's row of the first operand belongs to its own chunk of k
  const unsigned char *dl = act ? dig + g * (2 * CB) + (i & 3) * 16 : smem + (lane < 32 ? 192 : 64);
  const int dunit = act ? 8 * CB : 0, dchunk = act ? CB : 0, dhalf = act ? 64 : 0;
  float acc = 0.0f;
  auto consume = [&](int p, int unit) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const uint4 q = wt[p][s];
      const unsigned char *da = dl + unit * dunit + s * dchunk;
      const float f = int_chunk(q, *(const v4i *)da, *(const v4i *)(da + dhalf));
      const float d = half_bits_to_float((unsigned short)(s ? st[p] >> 16 : st[p])) * sx[unit * 8 + 2 * g + s];
      acc = fmaf(d, f, acc);
    }
  };
  int j = 0, u = 0;
  auto step = [&](int p) __attribute__((always_inline)) {
    consume(p, wk * sh.upw + u);
    if (++u == sh.upw) {  // (uniform) the group's share is complete
      u = 0;
      acc += __shfl_xor(acc, 16, 64);
      acc += __shfl_xor(acc, 32, 64);
      if (lane < 16) ps[(j * nw + wv) * 16 + lane] = acc;
      acc = 0.0f;
      j++;
    }
  };
  int t = 0;
  for (; t + PD <= nu; t += PD) {
#pragma unroll
    for (int p = 0; p < PD; p++) {
      step(p);
      request(p);
    }
  }
#pragma unroll
  for (int p = 0; p < PD; p++)
    if (t + p < nu) step(p);  // (uniform)
  __syncthreads();

  // ---- the sums of the wavefronts, in their order, and the epilogue ----
  const float ob = a.bias ? rb : 0.0f, orr = a.residual ? rr : 0.0f, of = LAYERNORM && a.fold_s ? rf : 0.0f;
  if (RMS || LAYERNORM) rstd = 1.0f / sqrtf(of_all(LAYERNORM ? red + 16 : red, 1, nw) / (float)a.cols + a.eps);
  float best = -INFINITY;
  int besti = 0x7fffffff;
  if (oj < iters && orow < a.rows) {
    const float *p = ps + ((size_t)oj * nw + (oi >> 4) * sh.ks) * 16 + (oi & 15);
    float v = of_all(p, 16, sh.ks);
    if (LAYERNORM && !CENTRED) v -= mu * of;
    if (RMS || LAYERNORM) v *= rstd;
    if (a.pair_swiglu) {  // rows 2r, 2r + 1 are a (gate, up) pair, in neighbouring threads (rows are even)
      const float full = v + ob, up = __shfl_xor(full, 1, 64);
      if (!(oi & 1)) a.y[(int64_t)m * a.y_stride + (orow >> 1)] = ct_silu(full) * up;
    } else {
      best = gemv_store(a, m, orow, v, posv, ob, orr);
      besti = orow;
    }
  }
  if (a.am_val) {
    __syncthreads();
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) argmax_merge(best, besti, __shfl_xor(best, o, 64), __shfl_xor(besti, o, 64));
    if (lane == 0) red[wv] = best, ((int *)red)[16 + wv] = besti;
    __syncthreads();
    if (tid == 0) {
      for (int w = 1; w < nw; w++) argmax_merge(best, besti, red[w], ((int *)red)[16 + w]);
      a.am_val[blockIdx.x] = best;
      a.am_idx[blockIdx.x] = besti;
    }
  }
}

bool gemv_int_supported(const WMat *w, const GemvArgs &a) {
  if (a.norm_out || a.pro == CTHIP_PRO_SWIGLU || (a.pro == CTHIP_PRO_LAYERNORM && !a.fold_s) || (a.pro == CTHIP_PRO_RMSNORM && a.norm_b)) return false;
  if (a.pair_swiglu && ((w->rows & 1) || a.am_val || a.residual || a.act != CTHIP_ACT_NONE || (a.split1 > 0 && a.split1 != (int)w->rows))) return false;
  return gemv_int_plan(w->type, w->rows, w->cols, state().compute_units).ok;
}

int launch_gemv_int(const WMat *w, GemvArgs a, int m, int *am_parts) {
  State &s = state();
  const GemvIntPlan p = gemv_int_plan(w->type, w->rows, w->cols, s.compute_units);
  if (!p.ok) return fail(CTHIP_E_UNSUPPORTED, "gemv: no integer launch for a (%lld, %lld) matrix of type %d", (long long)w->rows, (long long)w->cols, w->type);
  a.q = w->q;
  a.d = (const unsigned short *)w->d;
  a.rows = (int)w->rows;
  a.cols = (int)w->cols;
  if (a.split1 <= 0) a.split1 = a.split2 = a.rows;
  // A LayerNorm folded through the product loses what the mean takes off behind it.  Without a bias or a residual of the launch's own (a model's head), where the
  // vector kernels normalise their copy of the vector, the mean comes off the vector here too, one barrier ahead: error against 64 bits,
  // 50257 x 1280, mean of 3 / 30 / 300 deviations 3.5e-7 / 3.5e-6 / 3.3e-5 -> 1.4e-7 / 1.5e-6 / 6e-6 (vector kernels 4e-7 / 1e-6 / 1.6e-5; what is left is the mean's own rounding), in as much time (10.5 us).
  const bool centred = a.pro == CTHIP_PRO_LAYERNORM && !a.bias0 && !a.residual;
  // A line asked for with the hint is fetched a second time for its second chunk, which costs 4 - 7 % of a stream; keeping the weights from
  // pushing each other out of the cache is worth more until they are many times its size (us per step, with the hint / without: 36 layers of 1280, 0.46 GB 1040 / 1100;
  // 48 of 1600, 0.87 GB 1560 / 1560; 32 of 4096, 3.7 GB 1617 / 1549).
  const bool nt = s.gemv_stream < 0 ? w->stream && !w->stream_far : s.gemv_stream != 0;
  typedef void (*int_fn)(GemvArgs, GemvIntShape);
#define PICK(PRO, CENTRED) (nt ? k_gemv_int<PRO, CENTRED, true> : k_gemv_int<PRO, CENTRED, false>)
  int_fn fn = a.pro == CTHIP_PRO_RMSNORM ? PICK(CTHIP_PRO_RMSNORM, false) : a.pro != CTHIP_PRO_LAYERNORM ? PICK(CTHIP_PRO_NONE, false)
              : centred ? PICK(CTHIP_PRO_LAYERNORM, true) : PICK(CTHIP_PRO_LAYERNORM, false);
#undef PICK
  if (p.lds > 64 * 1024) {
    CTHIP_CHECK(hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kGemvIntMaxLdsBytes));
  }
  const long long nsg = (w->rows + 16 * p.rgp - 1) / (16 * p.rgp);
  hipLaunchKernelGGL(fn, dim3(p.grid, (unsigned)m), dim3(64 * p.ks * p.rgp), p.lds, s.stream, a, GemvIntShape{p.upw, p.ks, p.rgp, (65536 + p.ks - 1) / p.ks, (65536 + 16 * p.rgp - 1) / (16 * p.rgp), (int)p.grid, (int)(nsg / p.grid), (int)(nsg % p.grid)});
  CTHIP_LAUNCH_CHECK();
  *am_parts = (int)p.grid;
  return 0;
}

}  // namespace cthip
