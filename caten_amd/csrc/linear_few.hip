// Linear over a handful of rows: the projections of a short prompt, or of the next turn of a conversation.  Two ways:
//  - 8 .. 64 rows that lie in memory as operands of two bf16 terms (store_operands4 in planes.h), packed weights of up to 2048 columns, ALL of K in a
//    workgroup, the result finished here (launch_linear_few);
//  - X32: 8 .. 32 rows as they are, split by every workgroup, packed weights of any number of columns; K is shared among gridDim.y workgroups, whose partial sums go to memory
//    for the pass behind that adds up and normalises (launch_linear_few_shares; one share is finished here).
//
// The tiles of matmul.hip give such a product to a whole chip only by splitting K, which leaves partial tiles in memory and a
// second launch that adds them up.  Here a workgroup owns 16 NB output columns and all of K (or its share): its eight wavefronts take an eighth of it each,
// fetch their pieces of the weights and of the rows straight into operand registers (v_mfma_f32_16x16x32_bf16, lane l: row l % 16, k = 8 (l / 16) .. + 7 of a
// block of 32), BATCH blocks asked for together, and meet once in LDS.  A workgroup reads nothing twice; the rows are read by all of them, out of L2,
// and lie as the wavefronts hold them, whole cache lines to a request (as rows of terms, 16 half lines a request: 9.2 us for 37 rows of 1024 x 4096 fp16, 7.6 this
// way; by tiles 7.9 and 3.3 for their sums).  What bounds it: a launch, one round trip for a batch, and what a compute unit pulls out of
// L2 (all rows and its columns: 220 KB there).
// Products as in the tiles: the integers of a quantised weight are exact in bf16, their block's scale is applied to the block's
// sum; an fp16 weight is two terms, and the product of both lower terms is left out.  Error against 64 bits the same (2.5e-6, fp16 3.7e-6).
#include <algorithm>

#include "common.h"
#include "planes.h"

namespace cthip {

struct FewArgs {
  const unsigned char *A;    // the rows as operands of two terms (store_operands4)
  const unsigned char *W;    // N rows of packed weights, wpitch bytes apart
  const unsigned short *wd;  // scales, nkb a row
  int wpitch;
  int nkb;                   // blocks of 32 k
  const float *X;            // the rows as they are (X32)
  float *ws;                 // several shares of K (gridDim.y): their sums, [share][row][column]
  PlaneGemmArgs e;           // M, N and what happens to the result
};

enum { FW_Q8 = 0, FW_Q4 = 1, FW_F16 = 2 };
typedef float v4f_few __attribute__((ext_vector_type(4)));
constexpr int kFewWaves = 8;

template <int SRC, int MB, int NB, int BATCH, bool X32>
__global__ __launch_bounds__(64 * kFewWaves, MB * NB <= 2 && BATCH <= 5 ? 4 : 2) void k_linear_few(FewArgs a) {
  constexpr int NPB = SRC == FW_F16 ? 2 : 1, ROWS = 16 * MB, COLS = 16 * NB;
  extern __shared__ __align__(16) float red[];  // [wavefront][row][column]
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, col = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.x * COLS, M = a.e.M, N = a.e.N;
  const int share = X32 ? uniform_div(a.nkb + gridDim.y - 1, gridDim.y) : a.nkb, s0 = blockIdx.y * share, s1 = min(a.nkb, s0 + share);
  const int per = (share + kFewWaves - 1) / kFewWaves, kb0 = s0 + wv * per, kb1 = min(s1, kb0 + per);
  const unsigned char *ap = a.A + lane * 16;
  const float *xp[MB];
  if constexpr (X32) {
#pragma unroll
    for (int i = 0; i < MB; i++) xp[i] = a.X + (int64_t)min(16 * i + col, M - 1) * (32 * a.nkb) + 8 * g;  // rows past the end repeat the last one
  }
  const unsigned char *wp[NB];
  const unsigned short *dp[NB];
  v4f_few acc[MB][NB];
#pragma unroll
  for (int j = 0; j < NB; j++) {
    const int n = min(n0 + 16 * j + col, N - 1);  // columns past the end repeat the last one
    // 8 k of a block: 8 bytes of Q8_0; the low (k < 16) or high nibbles of 8 bytes of Q4_0; 16 bytes of fp16
    wp[j] = a.W + (int64_t)n * a.wpitch + (SRC == FW_Q8 ? 8 * g : SRC == FW_Q4 ? 8 * (g & 1) : 16 * g);
    dp[j] = SRC == FW_F16 ? nullptr : a.wd + (int64_t)n * a.nkb;
#pragma unroll
    for (int i = 0; i < MB; i++) acc[i][j] = v4f_few{0.0f, 0.0f, 0.0f, 0.0f};
  }
  // what a thread's first four results are added to, asked for with the first weights (at the end it was a round trip to memory: 1024 x 3072 f16 over 40 rows,
  // 7.6 us in place of 7.0); whole quads of columns, and the weights' first bytes where there is nothing
  const int f0c = 4 * (tid % (COLS / 4)), f0m = tid / (COLS / 4);
  float4 bb0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), rr0 = bb0;
  if constexpr (!X32) {
    bb0 = *(const float4 *)(a.e.bias ? a.e.bias + min(n0 + f0c, N - 4) : (const float *)a.A);
    rr0 = *(const float4 *)(a.e.residual ? a.e.residual + (int64_t)min(f0m, M - 1) * N + min(n0 + f0c, N - 4) : (const float *)a.A);
  }
  for (int b0 = kb0; b0 < kb1; b0 += BATCH) {
    // every request of the batch, none behind a branch: blocks past the share repeat its last one and are not multiplied
    uint4 w[BATCH][NB];
    unsigned d[BATCH][NB];
    uint4 af[BATCH][MB][2];  // two terms of 8 k, or 8 floats
#pragma unroll
    for (int b = 0; b < BATCH; b++) {
      const int kb = min(b0 + b, kb1 - 1);
#pragma unroll
      for (int j = 0; j < NB; j++) {
        if constexpr (SRC == FW_F16) {
          w[b][j] = *(const uint4 *)(wp[j] + kb * 64);
        } else {
          const uint2 t = *(const uint2 *)(wp[j] + kb * (SRC == FW_Q8 ? 32 : 16));
          w[b][j].x = t.x, w[b][j].y = t.y;
          d[b][j] = dp[j][kb];
        }
      }
#pragma unroll
      for (int q = 0; q < 2; q++)
#pragma unroll
        for (int i = 0; i < MB; i++) af[b][i][q] = X32 ? *(const uint4 *)(xp[i] + kb * 32 + 4 * q) : *(const uint4 *)(ap + ((kb * 2 + q) * MB + i) * 1024);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < BATCH; b++) {
      if (b0 + b >= kb1) break;  // (uniform)
      v8bf at[MB][2];
#pragma unroll
      for (int i = 0; i < MB; i++) {
        uint4 pl[2] = {af[b][i][0], af[b][i][1]};
        if constexpr (X32) {
          const float4 lo = __builtin_bit_cast(float4, pl[0]), hi = __builtin_bit_cast(float4, pl[1]);
          const float x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
          split8_planes<2>(x, pl);
        }
        at[i][0] = __builtin_bit_cast(v8bf, pl[0]), at[i][1] = __builtin_bit_cast(v8bf, pl[1]);
      }
#pragma unroll
      for (int j = 0; j < NB; j++) {
        v8bf bf[NPB];
        const uint4 v = w[b][j];
        if constexpr (SRC == FW_F16) {
          const unsigned h[4] = {v.x, v.y, v.z, v.w};
          float x[8];
#pragma unroll
          for (int e = 0; e < 4; e++) x[2 * e] = half_bits_to_float((unsigned short)(h[e] & 0xffff)), x[2 * e + 1] = half_bits_to_float((unsigned short)(h[e] >> 16));
          uint4 pl[2];
          split8_planes<2>(x, pl);
          bf[0] = __builtin_bit_cast(v8bf, pl[0]);
          bf[NPB - 1] = __builtin_bit_cast(v8bf, pl[1]);
        } else if constexpr (SRC == FW_Q8) {
          bf[0] = bf_of_q8(v.x, v.y);
        } else {
          const int sh = 4 * (g >> 1);
          const unsigned lo = (((v.x >> sh) & 0x0f0f0f0fu) + 0x78787878u) ^ 0x80808080u, hi = (((v.y >> sh) & 0x0f0f0f0fu) + 0x78787878u) ^ 0x80808080u;  // nibble - 8 as int8
          bf[0] = bf_of_q8(lo, hi);
        }
#pragma unroll
        for (int i = 0; i < MB; i++) {
          if constexpr (SRC == FW_F16) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(at[i][1], bf[0], acc[i][j], 0, 0, 0);  // smallest products first
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(at[i][0], bf[NPB - 1], acc[i][j], 0, 0, 0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(at[i][0], bf[0], acc[i][j], 0, 0, 0);
          } else {
            v4f_few t = {0.0f, 0.0f, 0.0f, 0.0f};
            t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(at[i][1], bf[0], t, 0, 0, 0);
            t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(at[i][0], bf[0], t, 0, 0, 0);
            const float dd = half_bits_to_float((unsigned short)d[b][j]);
#pragma unroll
            for (int r = 0; r < 4; r++) acc[i][j][r] = fmaf(dd, t[r], acc[i][j][r]);
          }
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < MB; i++)
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) red[(wv * ROWS + 16 * i + 4 * g + r) * COLS + 16 * j + col] = acc[i][j][r];
  __syncthreads();
#pragma unroll 1
  for (int f = tid; f < M * (COLS / 4); f += 64 * kFewWaves) {
    const int m = f / (COLS / 4), c = 4 * (f % (COLS / 4));
    if (n0 + c >= N) continue;
    float4 t[kFewWaves], v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int w = 0; w < kFewWaves; w++) t[w] = *(const float4 *)(red + (w * ROWS + m) * COLS + c);
#pragma unroll
    for (int w = 0; w < kFewWaves; w++) v.x += t[w].x, v.y += t[w].y, v.z += t[w].z, v.w += t[w].w;
    if (a.ws) {
      *(float4 *)(a.ws + ((int64_t)blockIdx.y * M + m) * N + n0 + c) = v;
    } else {
      PlaneStore store(a.e, PlaneStore::Late());
      // (anew in every pass: known to be the same, they have the loop copied for each of their cases)
      asm volatile("" : "+s"(store.act), "+s"(store.pairs), "+s"(store.routed));
      if (X32 || f != tid) {
        if (store.bias) bb0 = *(const float4 *)(store.bias + n0 + c);
        if (store.residual) rr0 = *(const float4 *)(store.residual + (int64_t)m * N + n0 + c);
      }
      plane_gemm_finish(store, N, m, n0 + c, v, bb0, rr0);
    }
  }
}

// Against a launch of tiles, for the most part with a second one for their sums; us, m = 8 / 17 / 40 / 64, the norm in front included:
//   Q8_0 768 x 2304 10.9 / 11.1 / 11.7 / 12.0 -> 7.0 / 7.3 / 8.1 / 8.8, 1280 x 5120 13.0 / 13.3 / 14.9 / 16.0 -> 9.5 / 10.5 / 11.7 / 13.0; Q4_0 alike;
//   f16 1024 x 4096 11.1 / 11.4 / 12.4 / 13.7 -> 6.8 / 7.3 / 8.5 / 9.2, 2048 x 11264 m = 17 / 40 / 64 30.9 / 31.9 / 34.8 -> 19.7 / 21.6 / 24.7.
// Short rows of many columns and long rows of few are where it loses (256 x 8192 m = 64 8.9 -> 9.4, 2048 x 256 m = 64 12.1 -> 12.8).  Where the rows are not
// passed over anyway its operands are a launch of their own, 2.5 us: 1024 x 4096 f16 8.5 / 8.9 / 9.8 / 10.8 -> 6.4 / 7.0 / 8.0 / 8.7, but 2048 x 768
// 8.1 / 8.1 / 8.5 / 8.9 -> 7.7 / 9.1 / 10.7 / 12.4, 256 x 768 5.7 / 5.8 / 5.8 / 6.2 -> 5.9 / 6.2 / 6.8 / 7.3.
bool linear_few_pays(const WMat *w, int m, int precision, bool norm) {
  if (precision != GEMM_BF16X3 || m < 8 || m > 64 || w->cols % 32 || w->cols > 2048 || w->rows % 4 || w->rows > 48ll * state().compute_units) return false;
  if (w->type != CTHIP_Q8_0 && w->type != CTHIP_Q4_0 && w->type != CTHIP_F16) return false;
  if (norm) return w->cols < 512 ? w->rows <= (m > 32 ? 4096 : 8192) : !(m > 32 && w->cols > 1280 && w->rows < 512);
  return w->cols >= 512 && w->rows <= 8192 && (w->cols <= 1280 ? m <= 32 || w->rows >= 512 : m <= 16);
}

template <int SRC, int MB, int NB>
static int few_launch(const FewArgs &a) {
  const dim3 grid((unsigned)((a.e.N + 16 * NB - 1) / (16 * NB))), block(64 * kFewWaves);
  constexpr size_t lds = (size_t)kFewWaves * 16 * MB * 16 * NB * 4;
  const int per = (a.nkb + kFewWaves - 1) / kFewWaves;  // blocks of a wavefront: in one batch where registers hold them
  if constexpr (NB == 3) {
    if (lds > 64 * 1024) CTHIP_CHECK(hipFuncSetAttribute((const void *)k_linear_few<SRC, MB, 3, (MB <= 2 ? 4 : 2), false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((k_linear_few<SRC, MB, 3, (MB <= 2 ? 4 : 2), false>), grid, block, lds, state().stream, a);
    CTHIP_LAUNCH_CHECK();
    return 0;
  }
  constexpr int kLong = MB <= 2 ? 8 : 4;
  if (per <= 4) hipLaunchKernelGGL((k_linear_few<SRC, MB, NB, 4, false>), grid, block, lds, state().stream, a);
  else if (per == 5) hipLaunchKernelGGL((k_linear_few<SRC, MB, NB, 5, false>), grid, block, lds, state().stream, a);
  else hipLaunchKernelGGL((k_linear_few<SRC, MB, NB, kLong, false>), grid, block, lds, state().stream, a);
  CTHIP_LAUNCH_CHECK();
  return 0;
}

template <int SRC, int MB>
static int few_launch32(const FewArgs &a, int shares) {
  const dim3 grid((unsigned)((a.e.N + 15) / 16), (unsigned)shares), block(64 * kFewWaves);
  constexpr size_t lds = (size_t)kFewWaves * 16 * MB * 16 * 4;
  const int share = (a.nkb + shares - 1) / shares, per = (share + kFewWaves - 1) / kFewWaves;
  if (per <= 2) hipLaunchKernelGGL((k_linear_few<SRC, MB, 1, 2, true>), grid, block, lds, state().stream, a);
  else if (per <= 4) hipLaunchKernelGGL((k_linear_few<SRC, MB, 1, 4, true>), grid, block, lds, state().stream, a);
  else hipLaunchKernelGGL((k_linear_few<SRC, MB, 1, 6, true>), grid, block, lds, state().stream, a);
  CTHIP_LAUNCH_CHECK();
  return 0;
}

static FewArgs few_args(float *y, const WMat *w, int m, const float *bias, const float *residual, int act) {
  FewArgs a = {};
  a.nkb = (int)(w->cols / 32);
  a.W = (const unsigned char *)w->q;
  a.wd = (const unsigned short *)w->d;
  a.wpitch = (int)(w->type == CTHIP_Q8_0 ? w->cols : w->type == CTHIP_Q4_0 ? w->cols / 2 : 2 * w->cols);
  a.e.C = y;
  a.e.M = m, a.e.N = (int)w->rows;
  a.e.bias = bias, a.e.residual = residual;
  a.e.act = act;
  return a;
}

// The Linears in front of a norm of a short prompt (projection, second of the MLP), which adds shares of K up on its way: rows as they are, which every
// workgroup splits into their two terms (as many bytes either way), shares to fill the chip once, twice as many where a wavefront
// would have more than four blocks.  A prompt of gpt2 q8_0, 9 / 14 rows 543 / 550 -> 486 / 493 us, q4_0 28 rows 630 -> 605, gpt2-medium q8_0 22 rows 1125 -> 1067,
// gpt2-large f16 12 rows 1664 -> 1560, llama-1.1b f16 9 rows 1472 -> 1384; more rows are as fast in tiles (gpt2-medium 37: 1220, 1224; llama-1.1b f16 17:
// 1496, 1517) or faster (gpt2-large 52 rows 2116, 2277 this way), and
// so are 4096 output columns (llama-7b 12 rows 3960, 4199).
bool linear_few_shares_pays(const WMat *w, int m, int precision) {
  if (precision != GEMM_BF16X3 || m < 8 || w->cols % 32 || w->rows % 4 || w->rows > 8ll * state().compute_units) return false;
  if (w->type != CTHIP_Q8_0 && w->type != CTHIP_Q4_0 && w->type != CTHIP_F16) return false;
  return m <= 16 || (m <= 32 && w->rows <= 1024);
}
// y (m, rows) = x W^T + bias + residual, or defer's shares of x W^T (to be added up and freed by the caller); all on 16 bytes
int launch_linear_few_shares(float *y, const WMat *w, const float *x, int m, const float *bias, const float *residual, GemmDeferred *defer) {
  FewArgs a = few_args(y, w, m, bias, residual, CTHIP_ACT_NONE);
  a.X = x;
  int shares = std::max(1, std::min(state().compute_units / ((a.e.N + 15) / 16), a.nkb / kFewWaves));
  if (a.nkb > 4 * kFewWaves * shares) shares *= 2;
  shares = std::min(shares, 16);
  const int share = (a.nkb + shares - 1) / shares;
  shares = (a.nkb + share - 1) / share;
  if (shares > 1) {
    const int rc = alloc_scratch((void **)&a.ws, sizeof(float) * (size_t)shares * m * a.e.N);  // fully written
    if (rc) return rc;
  }
  const int rc = w->type == CTHIP_Q8_0   ? (m <= 16 ? few_launch32<FW_Q8, 1>(a, shares) : few_launch32<FW_Q8, 2>(a, shares))
                 : w->type == CTHIP_Q4_0 ? (m <= 16 ? few_launch32<FW_Q4, 1>(a, shares) : few_launch32<FW_Q4, 2>(a, shares))
                                         : (m <= 16 ? few_launch32<FW_F16, 1>(a, shares) : few_launch32<FW_F16, 2>(a, shares));
  if (rc && a.ws) cthip_free(a.ws);
  else if (a.ws) defer->ws = a.ws, defer->ksplit = shares;
  return rc;
}

// y (m, rows) = act(x W^T + bias) + residual; act may be kActSwigluPairs, route as for launch_linear_gemm.
// Call only where linear_few_pays; y, bias and residual on 16 bytes.
int launch_linear_few(float *y, const WMat *w, const void *operands, int m, const float *bias, const float *residual, int act, const GemmRoute *route) {
  FewArgs a = few_args(y, w, m, bias, residual, act);
  a.A = (const unsigned char *)operands;
  if (act == kActSwigluPairs) {
    if (residual || route) return fail(CTHIP_E_BAD_ARG, "launch_linear_few: paired SwiGLU epilogue with a residual or a route");
    a.e.act = CTHIP_ACT_NONE;
    a.e.pairs = 1;
  }
  if (route) {
    a.e.routed = 1;
    a.e.route = *route;
  }
  const int nb = (a.e.N + 16 * state().compute_units - 1) / (16 * state().compute_units);  // 16 columns a workgroup, 32 or 48 where that is the one round over the chip
#define FEW2(SRC, MB) return nb == 1 ? few_launch<SRC, MB, 1>(a) : nb == 2 ? few_launch<SRC, MB, 2>(a) : few_launch<SRC, MB, 3>(a)
#define FEW(SRC)               \
  do {                         \
    if (m <= 16) FEW2(SRC, 1); \
    if (m <= 32) FEW2(SRC, 2); \
    if (m <= 48) FEW2(SRC, 3); \
    FEW2(SRC, 4);              \
  } while (0)
  if (w->type == CTHIP_Q8_0) FEW(FW_Q8);
  if (w->type == CTHIP_Q4_0) FEW(FW_Q4);
  FEW(FW_F16);
#undef FEW
#undef FEW2
}

}  // namespace cthip
