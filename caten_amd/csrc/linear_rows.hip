// Linear over a few rows (2 .. 32: a handful of sequences decoded together, a short prompt, the next turn of a
// conversation) on packed weights.  What such a launch cannot do without is ONE read of the weights; a
// single-row kernel per row reads them once for each, and a GEMM tile of 64 rows spends its time converting operands it
// uses once.
//
// A wavefront owns NS x 16 weight rows and multiplies them with all input rows on the matrix cores
// (v_mfma_f32_16x16x32).  Its weights come straight from memory into a ring of its own in LDS, whole cache lines of a row
// at a time, PD units (4 - 8 KB) in flight per wavefront and no barrier in the loop.  The input rows, split into 16-bit
// terms by a small launch in front (k_rows_planes, which also applies the norm or SwiGLU), wait in LDS for the workgroup's
// share of k.  (Every workgroup splitting its own share of the rows saved that launch and cost 5 us per workgroup.)
//
// Terms are bf16: they have the range of a float, so that an input keeps its bits whatever the largest of its row is (a row of a
// model with outlier channels spans more than the 2^39 of scaled fp16 terms).  Three of them hold all 24 bits.  A quantised
// weight is an integer, exact in bf16, times its block's scale, which is applied to the block's partial sum; an fp16 weight
// is two terms, exact; an fp32 weight three.  Products of terms below 2^-24 of the leading one are left out.
// An infinity or a NaN stands in the last term, which meets the leading term of a weight only (infinity times a lower
// term of zero would be NaN): it comes out as it does of fp32 products.  Matrix cores take a term below 2^-126 for zero: a
// row of nothing above 2^-32 goes in times the power of two that takes it to 2^-16.
// Three terms per input, two where "gemm_precision" asks for operands rounded to bf16.
//
// K is shared among as many workgroups as fill the chip; a share leaves its partial sums in memory and draws a ticket, the
// last one of a column group adds them in share order and stores the result (bias, activation, residual, routes).
#include "common.h"
#include "planes.h"

namespace cthip {

struct RowsGemmArgs {
  const unsigned char *A;    // planes of the input rows: [M][nkb][NPA][32], nkb = whole units (zeros past K)
  const float *rscale;       // per input row: what undoes its power of two
  int nkb;
  const unsigned char *W;    // N rows of packed weights, wpitch = wbytes apart
  const unsigned short *wd;  // scales, dpitch apart
  int wbytes, dpitch;
  int kblocks, kper;         // blocks of 32 k per weight row, per workgroup (whole units)
  float *parts;              // [column groups][shares][M][columns of a group]; null: one share
  PlaneGemmArgs e;           // M, N and what happens to the result
};

template <bool SIGNED>  // 8 int8 -> bf16 (SIGNED), or 8 nibbles (a byte each) - 8
__device__ __forceinline__ v8bf bf_of_bytes(unsigned a, unsigned b) {
  if (!SIGNED) a = (a + 0x78787878u) ^ 0x80808080u, b = (b + 0x78787878u) ^ 0x80808080u;  // per byte: nibble - 8 as int8 (no carry leaves a byte)
  return bf_of_q8(a, b);
}
// 8 floats -> NP terms, each of what the terms before it miss
template <int NP>
__device__ __forceinline__ void split8_rows(const float *v, uint4 *pl) {
  constexpr float kLargest = 3.38953139e38f;  // of bf16: what a float above it has more goes to the next term
  float r[8], t[8];
#pragma unroll
  for (int e = 0; e < 8; e++) r[e] = fabsf(v[e]) < INFINITY ? v[e] : 0.0f;
#pragma unroll
  for (int p = 0; p < NP; p++) {
    unsigned w[4];
#pragma unroll
    for (int e = 0; e < 8; e++) t[e] = p == 0 ? fminf(fmaxf(r[e], -kLargest), kLargest) : p + 1 == NP && !(fabsf(v[e]) < INFINITY) ? v[e] : r[e];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      w[e] = pack_bf16_pl(t[2 * e], t[2 * e + 1]);
      r[2 * e] -= __uint_as_float(w[e] << 16);  // exact: the difference of a float and its own leading bits
      r[2 * e + 1] -= __uint_as_float(w[e] & 0xffff0000u);
    }
    pl[p] = make_uint4(w[0], w[1], w[2], w[3]);
  }
}
typedef float v4f __attribute__((ext_vector_type(4)));
__device__ __forceinline__ v4f mma_rows(v8bf a, v8bf b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

enum { RW_Q8 = 1, RW_Q4 = 2, RW_F16 = 3, RW_F32 = 4 };

constexpr int kRowsMax = 32, kRowsGroups = 4096;  // input rows, column groups
__device__ __forceinline__ static int *rows_tickets() {  // zero between launches (inside a function its address is known without a trip to memory)
  static __device__ int tickets[kRowsGroups];
  return tickets;
}

// Bytes of a weight row in a unit, and blocks of 32 k: whole cache lines.  (Requests that cover 32 bytes of a row each, as
// operand registers would ask for them, are bound by the tag lookups of the compute unit's cache: 2.4 TB/s of Q8_0 and
// 1.5 TB/s of Q4_0 weights, most of it for the scales.)
constexpr int rows_unit_blocks(int src) { return src == RW_Q8 ? 4 : src == RW_Q4 ? 8 : 2; }
constexpr int rows_unit_bytes(int src) { return src == RW_F32 ? 256 : 128; }
constexpr bool rows_quant(int src) { return src == RW_Q8 || src == RW_Q4; }
// What the launcher instantiates: 16 NS weight rows a wavefront, 4 MB wavefronts, rings of PD units
constexpr int kRowsNS = 2, kRowsPD = 2;
constexpr int rows_columns(int mb) { return 16 * kRowsNS * 4 * mb; }  // of the result, per workgroup
constexpr int rows_slot(int src, bool wide_d) {  // bytes of a unit in a ring: weights, scales (whole load instructions)
  return 16 * kRowsNS * rows_unit_bytes(src) + (rows_quant(src) ? 16 * kRowsNS * rows_unit_blocks(src) / (wide_d ? 2 : 1) / 64 * 256 : 0);
}

// A wavefront: NS x 16 weight rows against MB x 16 input rows, v_mfma_f32_16x16x32 (lane l: row l % 16 of its operand, k =
// 8 (l / 16) .. + 7 of the block; result row 4 (l / 16) + r, column l % 16).  WIDE_D: a row's scales start at a multiple of four bytes, two of them are fetched as one dword
template <int SRC, int NPA, int MB, int NS, int NW, int PD, bool WIDE_D>
__global__ __launch_bounds__(64 * NW, 2) void k_linear_rows(RowsGemmArgs a) {
  constexpr bool QUANT = rows_quant(SRC);
  constexpr int NPB = QUANT ? 1 : SRC == RW_F16 ? 2 : NPA;
  constexpr int UB = rows_unit_blocks(SRC), CPW = rows_unit_bytes(SRC) / 16;  // blocks, 16-byte chunks of a row per unit
  constexpr int NR = 16 * NS;                                                     // weight rows of a wavefront
  constexpr int IW = NR * CPW / 64, ID = !QUANT ? 0 : NR * UB / (WIDE_D ? 2 : 1) / 64;  // load instructions per unit: weights, scales
  constexpr int WBYTES = NR * CPW * 16, SLOT = WBYTES + ID * 256;
  static_assert(NS == kRowsNS && PD == kRowsPD && SLOT == rows_slot(SRC, WIDE_D), "the LDS that rows_share counts");
  constexpr int NT = NR * NW, T = 64 * NW;  // columns of a workgroup, threads
  extern __shared__ __align__(16) unsigned char smem[];
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)smem;
  const int tid = threadIdx.x, lane = tid & 63, grp = lane >> 4, col = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = (blockIdx.x * NW + wave) * NR;
  const int M = a.e.M, N = a.e.N;
  const int kb0 = blockIdx.y * a.kper, units = (min(a.kblocks - kb0, a.kper) + UB - 1) / UB, kbs = units * UB;  // blocks of this share

  // ---- this wavefront's ring: unit u in slot u % PD, row r's chunk c at r * CPW + (c ^ (r & 7)) ----
  const unsigned ring = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)wave * (PD * SLOT));
  const unsigned char *wbase = uniform(a.W + (int64_t)min(n0, N - 1) * a.wbytes);
  const unsigned char *dbase = QUANT ? uniform((const unsigned char *)(a.wd + (int64_t)min(n0, N - 1) * a.dpitch)) : nullptr;
  const int last = N - 1 - min(n0, N - 1);  // rows past the end repeat the last one
  int wrow[IW], wch[IW];
#pragma unroll
  for (int j = 0; j < IW; j++) {
    const int s = j * 64 + lane, r = s / CPW;
    wrow[j] = min(r, last) * a.wbytes;
    wch[j] = ((s % CPW) ^ (r & 7)) * 16;
  }
  auto request = [&](int u) __attribute__((always_inline)) {
    const unsigned slot = ring + (unsigned)(u % PD) * SLOT;
    u = min(u, units - 1);  // past the end: the last unit again (never read), so that the counts stay the same
    const int at = (kb0 / UB + u) * (CPW * 16);
    // chunks past the end of a row repeat its last one (and meet zeros of the input)
#pragma unroll
    for (int j = 0; j < IW; j++) dma16(wbase, (unsigned)(wrow[j] + min(at + wch[j], a.wbytes - 16)), slot + j * 1024);
#pragma unroll
    for (int j = 0; j < ID; j++) {  // scale (pair) i of row r at dword i * NR + r
      const int s = j * 64 + lane, r = min(s % NR, last) * a.dpitch, kb = kb0 + u * UB;
      if (WIDE_D) dma4(dbase, 2u * (unsigned)(r + min(kb + 2 * (s / NR), a.kblocks - 2)), slot + WBYTES + j * 256);
      else dma2(dbase, 2u * (unsigned)(r + min(kb + s / NR, a.kblocks - 1)), slot + WBYTES + j * 256);
    }
  };
  // ---- the share of the input rows -> LDS behind the rings: row r's chunk c (16 bytes) at r * cpr + (c ^ (r & 7)) ----
  __shared__ int s_ticket;
  __shared__ float s_scale[64];  // of the rows (requested here: read from memory at the end it cost every launch 3 us)
  if (wave == 0) dma4(a.rscale, (unsigned)lane * 4u, (unsigned)(size_t)(__attribute__((address_space(3))) float *)s_scale);
  const unsigned char *As = smem + NW * PD * SLOT;
  const int cpr = kbs * 4 * NPA;
  for (int r = wave; r < M; r += NW) {
    const unsigned char *src = uniform(a.A + ((int64_t)r * a.nkb + kb0) * (64 * NPA));
    for (int c0 = 0; c0 < cpr; c0 += 64)
      if (c0 + lane < cpr)
        dma16(src, (unsigned)((c0 + lane) ^ (r & 7)) * 16u, __builtin_amdgcn_readfirstlane(lds0 + NW * PD * SLOT + (unsigned)(r * cpr + c0) * 16u));
  }
#pragma unroll
  for (int p = 0; p < PD; p++) request(p);
  wait_barrier<PD *(IW + ID)>();  // the rows are there, the weights on their way

  v4f acc[MB][NS];
#pragma unroll
  for (int i = 0; i < MB; i++)
#pragma unroll
    for (int j = 0; j < NS; j++) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  // Chunk of an input row's share: 4 (NPA kb + q) + grp for block kb, term q.  Its place differs from it in the low three
  // bits only, which take two values a lane (blocks come in pairs: 8 NPA chunks).
  const unsigned char *arow[MB][2];
#pragma unroll
  for (int i = 0; i < MB; i++) {
    const int r = min(16 * i + col, M - 1);
#pragma unroll
    for (int t = 0; t < 2; t++) arow[i][t] = As + (r * cpr + ((4 * t + grp) ^ (r & 7))) * 16;
  }
  const unsigned char *wown = smem + wave * (PD * SLOT);
  auto pair = [&](const unsigned char *slot, int bp, int kb) __attribute__((always_inline)) {  // blocks 2 bp, 2 bp + 1 of the unit = kb, kb + 1 of the share
    // All operand reads of the pair first, then (behind a scheduling fence) the conversions, which hide them: left alone
    // the compiler reads each operand right before its matrix instruction and waits out an LDS round trip every time.
    constexpr int NV = SRC == RW_F32 ? 2 : 1;
    uint4 w[NS][2][NV];
    unsigned dv[NS][2];
#pragma unroll
    for (int j = 0; j < NS; j++) {
      const int r = 16 * j + col;
      auto at = [&](int ch) { return slot + (r * CPW + (ch ^ (r & 7))) * 16; };
#pragma unroll
      for (int b = 0; b < 2; b++) {
        if constexpr (SRC == RW_Q8) {
          const uint2 t = *(const uint2 *)(at(2 * (2 * bp + b) + (grp >> 1)) + 8 * (grp & 1));
          w[j][b][0].x = t.x, w[j][b][0].y = t.y;
        } else if constexpr (SRC == RW_Q4) {
          const uint2 t = *(const uint2 *)(at(2 * bp + b) + 8 * (grp & 1));
          w[j][b][0].x = t.x, w[j][b][0].y = t.y;
        } else if constexpr (SRC == RW_F16) {
          w[j][b][0] = *(const uint4 *)at(4 * b + grp);
        } else {
          w[j][b][0] = *(const uint4 *)at(8 * b + 2 * grp);
          w[j][b][NV - 1] = *(const uint4 *)at(8 * b + 2 * grp + 1);
        }
      }
      if constexpr (QUANT) {
        const unsigned *D = (const unsigned *)(slot + WBYTES);
        if (WIDE_D) dv[j][0] = D[bp * NR + r];
        else dv[j][0] = D[2 * bp * NR + r], dv[j][1] = D[(2 * bp + 1) * NR + r];
      }
    }
    v8bf af[MB][2][NPA];
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
      for (int b = 0; b < 2; b++)
#pragma unroll
        for (int q = 0; q < NPA; q++) {
          const int c4 = NPA * b + q;  // in units of four chunks
          af[i][b][q] = __builtin_bit_cast(v8bf, *(const uint4 *)(arow[i][c4 & 1] + kb * (NPA * 64) + (c4 >> 1) * 128));
        }
    __builtin_amdgcn_sched_barrier(0);
    v8bf bf[NS][2][NPB];
#pragma unroll
    for (int j = 0; j < NS; j++)
#pragma unroll
      for (int b = 0; b < 2; b++) {
        const uint4 v = w[j][b][0];
        if constexpr (SRC == RW_Q8) {
          bf[j][b][0] = bf_of_bytes<true>(v.x, v.y);
        } else if constexpr (SRC == RW_Q4) {  // k 0..15 of a block are the low nibbles of its bytes, 16..31 the high ones
          bf[j][b][0] = bf_of_bytes<false>((v.x >> (4 * (grp >> 1))) & 0x0f0f0f0fu, (v.y >> (4 * (grp >> 1))) & 0x0f0f0f0fu);
        } else {
          float x[8];
          if constexpr (SRC == RW_F16) {
            const unsigned h[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < 4; e++) x[2 * e] = half_bits_to_float((unsigned short)(h[e] & 0xffff)), x[2 * e + 1] = half_bits_to_float((unsigned short)(h[e] >> 16));
          } else {
            const uint4 u = w[j][b][NV - 1];
            const unsigned f[8] = {v.x, v.y, v.z, v.w, u.x, u.y, u.z, u.w};
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = __uint_as_float(f[e]);
          }
          uint4 pl[NPB];
          split8_planes<NPB>(x, pl);
#pragma unroll
          for (int q = 0; q < NPB; q++) bf[j][b][q] = __builtin_bit_cast(v8bf, pl[q]);
        }
      }
    // a block's (quantised) or the pair's sum by itself: it is scaled before it is added, and one chain of matrix
    // instructions over thousands of k would round five times as much
    if constexpr (QUANT) {
      float dd[NS][2];
#pragma unroll
      for (int j = 0; j < NS; j++) {
        dd[j][0] = half_bits_to_float((unsigned short)(dv[j][0] & 0xffff));
        dd[j][1] = half_bits_to_float((unsigned short)(WIDE_D ? dv[j][0] >> 16 : dv[j][1]));
        asm("" : "+v"(dd[j][0]), "+v"(dd[j][1]));  // as floats: a multiply-add that converts its fp16 operand runs at half rate
      }
#pragma unroll
      for (int i = 0; i < MB; i++) {
        v4f tmp[NS][2];
#pragma unroll
        for (int q = NPA - 1; q >= 0; q--)
#pragma unroll
          for (int j = 0; j < NS; j++)
#pragma unroll
            for (int b = 0; b < 2; b++) tmp[j][b] = mma_rows(af[i][b][q], bf[j][b][0], q == NPA - 1 ? v4f{0.0f, 0.0f, 0.0f, 0.0f} : tmp[j][b]);
#pragma unroll
        for (int j = 0; j < NS; j++)
#pragma unroll
          // the pair's two meet first: half the roundings at the size of the total (Q8_0, 4096 columns: error 1.17e-7 -> 1.10e-7)
          for (int r = 0; r < 4; r++) acc[i][j][r] += fmaf(dd[j][0], tmp[j][0][r], dd[j][1] * tmp[j][1][r]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < MB; i++) {
        v4f tmp[NS];
#pragma unroll
        for (int j = 0; j < NS; j++) tmp[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        // pairs of terms above 2^-8(terms) of the leading product, the smallest first: only the two leading ones round at the
        // size of the sum (fp16 weights, 5 rows of 4096: error 1.26e-7 -> 1.1e-7 of the result, block after block -> this)
#pragma unroll
        for (int t = NPA - 1; t >= 0; t--)
#pragma unroll
          for (int q = 0; q <= t; q++)
            if (t - q < NPB)
#pragma unroll
              for (int b = 0; b < 2; b++)
#pragma unroll
                for (int j = 0; j < NS; j++) tmp[j] = mma_rows(af[i][b][q], bf[j][b][t - q], tmp[j]);
#pragma unroll
        for (int j = 0; j < NS; j++) acc[i][j] += tmp[j];
      }
    }
  };
  // Unit u has landed when at most the requests of the PD - 1 units behind it are outstanding.  Its slot is asked for again
  // when its last reads are done: no other wavefront looks into this ring, so there is no barrier.
  for (int u = 0; u < units; u++) {
    wait_loads<(PD - 1) * (IW + ID)>();
    const unsigned char *slot = wown + (u % PD) * SLOT;
#pragma unroll
    for (int bp = 0; bp < UB / 2; bp++) pair(slot, bp, u * UB + 2 * bp);
    wait_lds();
    request(u + PD);
  }
  wait_barrier<0>();  // (the last requests have landed: the memory is free for other things)

  // ---- the result: this share's partial sums, and behind the group's last ticket their sum ----
  const bool shares = a.parts != nullptr;
  float *mine = shares ? a.parts + ((int64_t)blockIdx.x * gridDim.y + blockIdx.y) * M * NT : (float *)smem;
#pragma unroll
  for (int i = 0; i < MB; i++)
#pragma unroll
    for (int j = 0; j < NS; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int m = 16 * i + 4 * grp + r;
        if (m >= M) continue;
        float *o = mine + m * NT + wave * NR + 16 * j + col;
        const float v = acc[i][j][r] * s_scale[m];
        if (shares) __hip_atomic_store(o, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else *o = v;
      }
  if (shares) {
    // a share's sums are device-scope stores that have reached memory before its ticket is drawn (a fence would write
    // back and invalidate the whole L2 of the XCD); the counters are left at zero for the next launch
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) s_ticket = __hip_atomic_fetch_add(rows_tickets() + blockIdx.x, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (s_ticket != (int)gridDim.y - 1) return;
    if (tid == 0) __hip_atomic_store(rows_tickets() + blockIdx.x, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    __syncthreads();
  }
  const float *all = shares ? a.parts + (int64_t)blockIdx.x * gridDim.y * M * NT : (const float *)smem;
  for (int f = tid; f < M * (NT / 4); f += T) {
    const int m = f / (NT / 4), c = 4 * (f % (NT / 4));
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (shares) {
      for (int z0 = 0; z0 < (int)gridDim.y; z0 += 8) {  // eight shares requested together, added in order
        unsigned long long t[8][2];
#pragma unroll
        for (int z = 0; z < 8; z++) {
          const unsigned long long *src = (const unsigned long long *)(all + ((int64_t)min(z0 + z, (int)gridDim.y - 1) * M + m) * NT + c);
          t[z][0] = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          t[z][1] = __hip_atomic_load(src + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int z = 0; z < 8; z++)
          if (z0 + z < (int)gridDim.y) {
            v.x += __uint_as_float((unsigned)t[z][0]), v.y += __uint_as_float((unsigned)(t[z][0] >> 32));
            v.z += __uint_as_float((unsigned)t[z][1]), v.w += __uint_as_float((unsigned)(t[z][1] >> 32));
          }
      }
    } else {
      v = *(const float4 *)(all + m * NT + c);
    }
    plane_gemm_store(a.e, m, blockIdx.x * NT + c, v);
  }
}

// ---- input rows -> planes, with what the Linear has in front ----
// One block per row, held in registers (VPL pieces of 8 floats per thread).  ROWS: terms for k_linear_rows, else for
// gemm_planes.hip.  kbp: blocks of 32 k per row of planes (zeros past K).
// A few rows are a few blocks on cold compute units: what bounds those is the fetch of their own unrolled code and one wavefront's
// chain, so a block has as many threads as its row has pieces (up to 1024).  5 rows of 11008 with SwiGLU, 256 threads of 8 pieces -> 1024
// of 2: 9.5 -> 6.4 us.  What is left there is one compute unit's vector instructions, 1000 for each of 16 wavefronts; without a norm a piece needs nothing of the others but
// whether the row is one of small numbers, so gridDim.y blocks of 256 pieces share a row: 6.9 -> 4.8 us.
struct RowsPlanesArgs {
  uint4 *out;
  float *rscale;  // ROWS: what undoes a row's power of two
  const float *x;
  int64_t stride;
  int K, kbp;
  const float *g, *b;
  float eps;
  int row_blocks;  // not ROWS: as matrix operands of that many blocks of 16 rows (store_operands4), 0 = as planes
};
template <int PRO, int NP, bool ROWS, int NT, int VPL>
__global__ __launch_bounds__(NT) void k_rows_planes(RowsPlanesArgs a) {
  constexpr int NW = NT / 64;
  __shared__ float red[3][NW];
  const int tid = threadIdx.x, K = a.K;
  const float *xr = a.x + blockIdx.x * a.stride;
  constexpr bool NORM = PRO == CTHIP_PRO_LAYERNORM || PRO == CTHIP_PRO_RMSNORM;
  float v[VPL][8];
  const int first = NORM ? tid : tid + NT * VPL * (int)blockIdx.y;  // this thread's first piece
  auto ld8 = [&](const float *p, int j, float *o) __attribute__((always_inline)) {  // K % 4 == 0: four floats are inside the row or past it
    const int k = 8 * (first + NT * j);
    const float4 t0 = *(const float4 *)(p + min(k, K - 4)), t1 = *(const float4 *)(p + min(k + 4, K - 4));
    o[0] = t0.x, o[1] = t0.y, o[2] = t0.z, o[3] = t0.w, o[4] = t1.x, o[5] = t1.y, o[6] = t1.z, o[7] = t1.w;
  };
  auto in = [&](int j, int e) { return 8 * (first + NT * j) + e < K; };
#pragma unroll
  for (int j = 0; j < VPL; j++) ld8(xr, j, v[j]);
  if (PRO == CTHIP_PRO_SWIGLU) {
#pragma unroll
    for (int j = 0; j < VPL; j++) {
      float u[8];
      ld8(xr + K, j, u);
#pragma unroll
      for (int e = 0; e < 8; e++) v[j][e] = ct_silu(v[j][e]) * u[e];
    }
  }
  auto block_sum = [&](int slot, float s) {
    s = wave_sum(s);
    if ((tid & 63) == 0) red[slot][tid >> 6] = s;
    __syncthreads();
    s = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; w += 2) s += red[slot][w] + red[slot][w + 1];
    return s;
  };
  if (NORM) {
    const float inv_n = 1.0f / (float)K;
    float mean = 0.0f, q = 0.0f;
    if (PRO == CTHIP_PRO_LAYERNORM) {
      float s = 0.0f;
#pragma unroll
      for (int j = 0; j < VPL; j++)
#pragma unroll
        for (int e = 0; e < 8; e++) s += in(j, e) ? v[j][e] : 0.0f;
      mean = block_sum(0, s) * inv_n;
    }
#pragma unroll
    for (int j = 0; j < VPL; j++)
#pragma unroll
      for (int e = 0; e < 8; e++) {
        v[j][e] -= mean;
        q += in(j, e) ? v[j][e] * v[j][e] : 0.0f;
      }
    const float rstd = 1.0f / sqrtf(block_sum(1, q) * inv_n + a.eps);
#pragma unroll
    for (int j = 0; j < VPL; j++) {
      float g[8], b[8];
      if (a.g) ld8(a.g, j, g);
      if (a.b) ld8(a.b, j, b);
#pragma unroll
      for (int e = 0; e < 8; e++) {
        v[j][e] *= rstd;
        if (a.g) v[j][e] *= g[e];
        if (a.b) v[j][e] += b[e];
      }
    }
  }
  auto emit = [&](float up) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < VPL; j++) {
      const int c = first + NT * j;
      if (c >= 4 * a.kbp) continue;
      float t[8];
#pragma unroll
      for (int e = 0; e < 8; e++) t[e] = in(j, e) ? v[j][e] * up : 0.0f;
      uint4 pl[NP];
      if (ROWS) split8_rows<NP>(t, pl);
      else split8_planes<NP>(t, pl);
#pragma unroll
      for (int q = 0; q < NP; q++)
        if (!ROWS && a.row_blocks) a.out[((int64_t)((c >> 2) * NP + q) * a.row_blocks + (blockIdx.x >> 4)) * 64 + 16 * (c & 3) + (blockIdx.x & 15)] = pl[q];
        else a.out[((int64_t)blockIdx.x * a.kbp + (c >> 2)) * (4 * NP) + 4 * q + (c & 3)] = pl[q];
    }
  };
  emit(1.0f);
  if (ROWS) {  // behind the stores, which then need not wait for the whole row: one of small numbers is stored again
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < VPL; j++)
#pragma unroll
      for (int e = 0; e < 8; e++) m = in(j, e) && fabsf(v[j][e]) < INFINITY ? fmaxf(m, fabsf(v[j][e])) : m;
    m = wave_max(m);
    if ((tid & 63) == 0) red[2][tid >> 6] = m;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; w++) m = fmaxf(m, red[2][w]);
    if (!NORM && gridDim.y > 1 && m < 0x1p-32f) {  // (uniform) nothing here says that the row is not one of small numbers: all of it, in every block alike
      for (int c = tid; 8 * c < K; c += NT) {
        float o[8];
        ld8(xr, c / NT - (first - tid) / NT, o);
        if (PRO == CTHIP_PRO_SWIGLU) {
          float u[8];
          ld8(xr + K, c / NT - (first - tid) / NT, u);
#pragma unroll
          for (int e = 0; e < 8; e++) o[e] = ct_silu(o[e]) * u[e];
        }
#pragma unroll
        for (int e = 0; e < 8; e++) m = 8 * c + e < K && fabsf(o[e]) < INFINITY ? fmaxf(m, fabsf(o[e])) : m;
      }
      m = wave_max(m);
      __syncthreads();
      if ((tid & 63) == 0) red[2][tid >> 6] = m;
      __syncthreads();
#pragma unroll
      for (int w = 0; w < NW; w++) m = fmaxf(m, red[2][w]);
    }
    const bool small = m < 0x1p-32f;
    // to 2^-16: 110 bits above what the matrix cores take for zero, and 2^15 finite weights times it have a finite sum
    const int e = small ? 111 - max((int)(__float_as_uint(m) >> 23), 1) : 0;
    if (small) emit(__uint_as_float((unsigned)(127 + e) << 23));
    if (tid == 0 && blockIdx.y == 0) a.rscale[blockIdx.x] = __uint_as_float((unsigned)(127 - e) << 23);
  }
}
constexpr int kRowsPlanesMaxK = 8 * 1024 * 4;  // widest row the largest instantiation holds

// How many workgroups share K, as units per share, and the LDS such a workgroup asks for.  Every compute unit holds `resident`
// workgroups (LDS) at a time; a round of them costs its units at the rate of the compute unit (about 0.85 us per 16 KB of weights
// and workgroup, 30 % more per further 16 input rows) and about 1.5 us of its own, a share costs its partial sums.
// At most 32 shares, one where there are more column groups than tickets: wide rows then fit no workgroup (per = 0).
struct RowsShare {
  int per = 0;
  size_t lds = 0;
};
static RowsShare rows_share(int src, int terms, int mb, bool wide_d, int M, int N, int kblocks) {
  const int ub = rows_unit_blocks(src), nt = rows_columns(mb), cus = state().compute_units;
  const int groups = (N + nt - 1) / nt, units = (kblocks + ub - 1) / ub;
  RowsShare best;
  double best_us = 0;
  for (int ks = 1; ks <= 32 && ks <= units; ks++) {
    const int per = (units + ks - 1) / ks;
    if ((units + per - 1) / per != ks || (ks > 1 && groups > kRowsGroups)) continue;
    size_t lds = (size_t)4 * mb * kRowsPD * rows_slot(src, wide_d) + (size_t)M * per * ub * 64 * terms;
    if (lds < (size_t)M * nt * 4) lds = (size_t)M * nt * 4;
    if (lds > 156 * 1024) continue;
    const int resident = lds <= 78 * 1024 ? 2 : 1;
    const double tu = 0.85 * rows_unit_bytes(src) / 128 * mb * (1 + 0.3 * (mb - 1));
    const int64_t wgs = (int64_t)groups * ks;
    const int64_t full = wgs / (cus * resident), left = wgs - full * cus * resident;
    double t = full * (resident * per * tu + 1.5);
    if (left) t += (left > cus ? 2 : 1) * per * tu + 1.5;
    t += ks > 1 ? 1.0 + (double)ks * M * N * 8 / 4e6 : 0.0;
    if (best.per == 0 || t < best_us) best_us = t, best.per = per, best.lds = lds;
  }
  return best;
}

template <int SRC, int NPA, int MB, bool WIDE_D>
static int rows_launch(RowsGemmArgs a, bool *done) {
  constexpr int NS = kRowsNS, NW = 4 * MB, PD = kRowsPD, NT = rows_columns(MB), T = 64 * NW, UB = rows_unit_blocks(SRC);
  const int M = a.e.M, N = a.e.N, groups = (N + NT - 1) / NT, units = (a.kblocks + UB - 1) / UB;
  const RowsShare share = rows_share(SRC, NPA, MB, WIDE_D, M, N, a.kblocks);
  if (share.per == 0) return fail(CTHIP_E_STATE, "linear rows: no share of (%d, %d, %d blocks) fits", M, N, a.kblocks);
  a.kper = share.per * UB;
  const int ks = (units + share.per - 1) / share.per;
  a.parts = nullptr;
  if (ks > 1 && alloc_scratch((void **)&a.parts, sizeof(float) * (size_t)groups * ks * M * NT)) return 0;
  *done = true;
  static bool big_lds = false;
  auto fn = k_linear_rows<SRC, NPA, MB, NS, NW, PD, WIDE_D>;
  if (!big_lds) {
    CTHIP_CHECK(hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, 157 * 1024));
    big_lds = true;
  }
  hipLaunchKernelGGL(fn, dim3(groups, ks), dim3(T), share.lds, state().stream, a);
  const hipError_t e = hipGetLastError();
  const int rc = a.parts ? cthip_free(a.parts) : 0;  // stream-ordered: handed out again only to later work on this stream
  if (e != hipSuccess) return fail((int)e, "linear rows: launch -> %s", hipGetErrorString(e));
  return rc;
}

template <int PRO, int NP, bool ROWS>
static void rows_planes_launch(const RowsPlanesArgs &a, int m) {
  const int pieces = a.kbp * 4;
  const int blocks = (pieces + 255) / 256;
  // several blocks to a row while they find compute units of their own; past that they only take turns
  if (PRO != CTHIP_PRO_LAYERNORM && PRO != CTHIP_PRO_RMSNORM && blocks > 1 && (int64_t)m * blocks <= state().compute_units) {
    hipLaunchKernelGGL((k_rows_planes<PRO, NP, ROWS, 256, 1>), dim3(m, blocks), dim3(256), 0, state().stream, a);
    return;
  }
#define RP(NT, V) hipLaunchKernelGGL((k_rows_planes<PRO, NP, ROWS, NT, V>), dim3(m), dim3(NT), 0, state().stream, a)
  if (pieces <= 256) RP(256, 1);
  else if (pieces <= 512) RP(512, 1);
  else if (pieces <= 1024) RP(1024, 1);
  else if (pieces <= 2048) RP(1024, 2);
  else RP(1024, 4);
#undef RP
}

static int rows_source(const WMat *w) { return w->type == CTHIP_Q8_0 ? RW_Q8 : w->type == CTHIP_Q4_0 ? RW_Q4 : w->type == CTHIP_F16 ? RW_F16 : RW_F32; }
// terms per input: all 24 bits, or 16 where operands rounded to bf16 are asked for
static int rows_terms(int m, int precision) { return m >= 8 && precision == GEMM_BF16 ? 2 : 3; }
static bool rows_wide_scales(const WMat *w) { return w->cols / 32 % 2 == 0 && rows_quant(rows_source(w)); }

// Whether this is the launch to take: the operands are laid out for it, a share of it fits a workgroup, and it is the faster one.
// Fewer than 8 rows: against the single-row kernels, one pass over the weights per row.  They cost about 3 us + m weights
// at 4.3 (quantised), 2.7 (fp16) or 2.0 (fp32) per ns, the two launches here 9.5 us + the weights once at 3.2 / 2.3 / 1.15.
//   us, m = 3 / 5 / 7, weights not in any cache:  22016 x 4096 Q8_0 49 / 73 / 98 -> 31 / 33 / 33, fp32 158 / 261 / 368 -> 86 / 89 / 103;
//   4096 x 4096 Q8_0 m = 5 / 7 23 / 29 -> 13 / 13;  4096 x 11008 Q4_0 m = 5 44 -> 20;  768 x 3072 stays there at 5 / 7 (6 / 7; 11 here)
// 8 rows and more: against a GEMM tile of 64 rows, which is as fast on small matrices and where the tile fills up:
//   22016 x 4096 m = 12: Q8_0 51 -> 38, Q4_0 52 -> 36, fp16 74 -> 49;  fp16 m = 24 / 32 74 / 74 -> 61 / 73;
//   11264 x 2048 m = 12: Q8_0, Q4_0, fp16 20, 20, 26 -> 16, 16, 19;  4096 x 4096 m = 12: 15, 14, 18 -> 14, 14, 16.
// Of 14 - 16 rows as long as 11008 a workgroup's memory holds a share too small for one round over the chip: Q8_0 m = 14 / 16
// 25 / 26 -> 22 / 28; they are taken for their bits (the tiles' error is 2.4e-6 there, 1.3e-7 here).
bool linear_rows_pays(const WMat *w, const float *x, int64_t x_stride, int m, int precision, const float *g, const float *b) {
  if (m < 2 || m > kRowsMax || precision == GEMM_FP32) return false;  // (fp32 operands asked for: the single-row kernels')
  if (w->cols % (w->type == CTHIP_F16 ? 8 : 4) || w->cols < 64 || w->cols > kRowsPlanesMaxK - 256) return false;  // whole 16-byte pieces
  auto al = [](const void *p) { return (uintptr_t)p % 16 == 0; };
  if (x_stride % 4 || !al(x) || !al(g) || !al(b)) return false;
  const double weights = (double)w->rows * w->cols * 1e-3;
  const bool quant = w->type == CTHIP_Q8_0 || w->type == CTHIP_Q4_0;
  if (m < 8) {
    const double each = quant ? 4.3 : w->type == CTHIP_F16 ? 2.7 : 2.0, once = quant ? 3.2 : w->type == CTHIP_F16 ? 2.3 : 1.15;
    if (3000 + m * weights / each <= 9500 + weights / once) return false;
  } else if (w->type == CTHIP_F32 || (m <= 16 ? weights < (quant ? 22e3 : 20e3) : quant || weights < 60e3)) {
    return false;
  }
  return rows_share(rows_source(w), rows_terms(m, precision), m <= 16 ? 1 : 2, rows_wide_scales(w), m, (int)w->rows, (int)((w->cols + 31) / 32)).per > 0;
}

// rows with what a Linear has in front of it as bf16 planes for gemm_planes.hip (x on 16 bytes, K % 32 == 0)
bool rows_planes_supported(int K) { return K % 32 == 0 && K <= kRowsPlanesMaxK; }
int launch_rows_planes(void *planes, const float *x, int m, int K, int pro, const float *g, const float *b, float eps, int terms) {
  const RowsPlanesArgs pa = {(uint4 *)planes, nullptr, x, K, K, K / 32, g, b, eps, terms == kTermsOperands ? (m + 15) / 16 : 0};
  if (pro == CTHIP_PRO_LAYERNORM) rows_planes_launch<CTHIP_PRO_LAYERNORM, 2, false>(pa, m);
  else if (pro == CTHIP_PRO_RMSNORM) rows_planes_launch<CTHIP_PRO_RMSNORM, 2, false>(pa, m);
  else rows_planes_launch<CTHIP_PRO_NONE, 2, false>(pa, m);
  CTHIP_LAUNCH_CHECK();
  return 0;
}

// y (m, rows) = act(prologue(x) @ W^T + bias) + residual for a few rows; act may be kActSwigluPairs, route as for
// launch_linear_gemm.  Call only where linear_rows_pays; *done stays false where there is no scratch to be had.
int launch_linear_rows(float *y, const WMat *w, const float *x, int64_t x_stride, int m, const float *bias, const float *residual, int act,
                       int pro, const float *norm_g, const float *norm_b, float eps, int precision, const GemmRoute *route, bool *done) {
  const int terms = rows_terms(m, precision);
  const int ub = rows_unit_blocks(rows_source(w));
  RowsGemmArgs a = {};
  a.kblocks = (int)((w->cols + 31) / 32);
  a.nkb = (a.kblocks + ub - 1) / ub * ub;
  a.W = (const unsigned char *)w->q;
  a.wd = (const unsigned short *)w->d;
  a.dpitch = (int)(w->cols / 32);
  a.wbytes = (int)(w->type == CTHIP_Q8_0 ? w->cols : w->type == CTHIP_Q4_0 ? w->cols / 2 : w->type == CTHIP_F16 ? 2 * w->cols : 4 * w->cols);
  a.e.C = y;
  a.e.M = m;
  a.e.N = (int)w->rows;
  a.e.bias = bias;
  a.e.residual = residual;
  a.e.act = act;
  if (act == kActSwigluPairs) {
    if (a.e.N % 4 || residual || route) return fail(CTHIP_E_BAD_ARG, "launch_linear_rows: paired SwiGLU epilogue with %d rows, a residual or a route", a.e.N);
    a.e.act = CTHIP_ACT_NONE;
    a.e.pairs = 1;
  }
  if (route) {
    a.e.routed = 1;
    a.e.route = *route;
  }
  unsigned char *planes = nullptr;
  const size_t plane_bytes = (size_t)m * a.nkb * 64 * terms;
  if (stream_capturing() || alloc_scratch((void **)&planes, plane_bytes + sizeof(float) * 64)) return 0;  // fully written by the first launch
  float *rscale = (float *)(planes + plane_bytes);
  a.rscale = rscale;
  int rc = 0;
  a.A = planes;
  const RowsPlanesArgs pa = {(uint4 *)planes, rscale, x, x_stride, (int)w->cols, a.nkb, norm_g, pro == CTHIP_PRO_LAYERNORM || m >= 8 ? norm_b : nullptr, eps, 0};
#define RP2(PRO)                                              \
  do {                                                        \
    if (terms == 3) rows_planes_launch<PRO, 3, true>(pa, m);  \
    else rows_planes_launch<PRO, 2, true>(pa, m);             \
  } while (0)
  switch (pro) {
    case CTHIP_PRO_LAYERNORM: RP2(CTHIP_PRO_LAYERNORM); break;
    case CTHIP_PRO_RMSNORM: RP2(CTHIP_PRO_RMSNORM); break;
    case CTHIP_PRO_SWIGLU: RP2(CTHIP_PRO_SWIGLU); break;
    default: RP2(CTHIP_PRO_NONE); break;
  }
#undef RP2
  const bool wide = rows_wide_scales(w);
#define RL(SRC, MB, WD)                                 \
  do {                                                  \
    if (terms == 3) rc = rows_launch<SRC, 3, MB, WD>(a, done); \
    else rc = rows_launch<SRC, 2, MB, WD>(a, done);           \
  } while (0)
  if (w->type == CTHIP_Q8_0 && wide) RL(RW_Q8, 1, true);
  else if (w->type == CTHIP_Q8_0) RL(RW_Q8, 1, false);
  else if (w->type == CTHIP_Q4_0 && wide) RL(RW_Q4, 1, true);
  else if (w->type == CTHIP_Q4_0) RL(RW_Q4, 1, false);
  else if (w->type == CTHIP_F32) rc = rows_launch<RW_F32, 3, 1, false>(a, done);
  else if (m <= 16) RL(RW_F16, 1, false);
  else RL(RW_F16, 2, false);
#undef RL
  const int rf = cthip_free(planes);  // stream-ordered: handed out again only to later work on this stream
  return rc ? rc : rf;
}

}  // namespace cthip
