// MFMA GEMM over operands that lie in memory as bf16 terms ("planes"), for products large enough to fill the chip:
// prompts, Linears over many rows and big matmuls.  The small ones stay with matmul.hip.
//
// matmul.hip converts fp32 operands on their way into LDS, once per tile: every tile of a row of tiles repeats the
// conversion of the same rows, a third of a workgroup's wavefronts do nothing else, and a 64 x 64 (64 x 128) tile asks the
// caches for 64 bytes per matrix instruction.  Here an operand is split ONCE (by k_planes_rows / k_planes_cols or by
// the kernel that produces it) and the GEMM kernel only moves and multiplies: global memory -> LDS by the load path that
// bypasses registers, LDS -> operand registers, matrix cores.
//
// Layout of a plane operand: row-major, a row is a sequence of blocks of 32 consecutive k, a block is NP runs of 32
// bf16 (term 0 = bf16(x), term p = bf16 of what terms 0..p-1 miss).  A K-step of a row is one contiguous piece of NP * 64
// bytes: whole cache lines for NP = 2.
#include <mutex>
#include <unordered_set>

#include "common.h"
#include "digits.h"
#include "gemm_plan.h"

namespace cthip {

// 16-byte chunk c of row r of an LDS tile with CPR chunks per row is kept at chunk r * CPR + (c ^ swz<CPR>(r)).  A 16-byte read
// is served sixteen lanes at a time over 64 banks (256 bytes): of lanes 0 .. 31, each reading the same chunk of its own row,
// {0-3, 12-15, 20-27} and then {4-11, 16-19, 28-31}, and the same of lanes 32 .. 63 (timed on the card).  With SPREAD the sixteen rows of
// such a set lie in sixteen different columns of the banks; without, which is right for eight consecutive rows over 128 bytes, a read
// takes twice its cycles.
template <int CPR, bool SPREAD>
__device__ __forceinline__ int swz(int r) {
  static_assert(CPR % 4 == 0, "whole blocks of 32 k");
  if (SPREAD) return CPR % 8 == 0 ? ((r >> 1) & 7) : ((r >> 2) & 3);
  return CPR % 8 == 0 ? (r & 7) : ((r >> 1) & 3);
}

// SRC: how B lies in memory: PL_PLANES, or PL_INT, one plane of the integers of a quantised matrix (exact in bf16) with an
// fp16 scale per block of 32, which is applied to the block's partial sum (acc += d * sum a q).
// MB x NB blocks of 32 x 32 per wavefront, WM x WN wavefronts, NBUF LDS buffers; a step is a block of 32 k.
//
// What bounds it: the matrix cores ask LDS for an operand per instruction and block edge, so a wavefront's piece wants to be
// large (64 x 64: 16 reads for 24 instructions at two terms); two workgroups of four wavefronts per compute unit fill each
// other's waits (reading a step's operands under the step before it instead, two sets of registers, measured the same or
// slower; so did deeper rings than the launcher's).  4096^3, two terms: 284 us without the passes in front = 484 TFLOP/s of
// results, 1.45 PFLOP/s of matrix instructions (the library's bf16 product reaches 1.2 - 1.5 on the card), against 180 with the operands converted per tile.
// (3000 x 4100 x 5000, 256 x 256 tiles: matrix cores busy 54 % of the cycles that the counters show, 1.9 GHz.)  Integers need two products instead of three but 16 multiply-adds per lane and block for
// the scales: 1900 x 11264 x 2048 194 us (operands converted per tile: 340), 1900 x 2048 x 5632 117 us (149).
template <int NPA, int SRC, int NPB, int MB, int NB, int WM, int WN, int NBUF>
__global__ __launch_bounds__(64 * WM * WN, 2) void k_gemm_planes(PlaneGemmArgs a) {
  constexpr int NW = WM * WN, BM = 32 * MB * WM, BN = 32 * NB * WN;
  constexpr int CA = 4 * NPA, CB = 4 * NPB;  // chunks per row and step
  // Reads without conflicts are the faster ones (4096^3, two terms, 256 x 256 tiles: 354 -> 346 us; 128 x 128 of eight wavefronts: 392 -> 376; integers,
  // 1900 x 2048 x 5632: 126 -> 117) but in two tiles of four wavefronts, two workgroups to a compute unit, for a reason no counter shows: 64 x 64 a wavefront
  // at two terms (4096^3 357 -> 390, 3000 x 4100 x 5000 391 -> 435) and 64 x 32 at three (700 x 4500 x 800 49.9 -> 51.1).
  constexpr bool SPREAD = !(SRC == PL_PLANES && NW == 4 && MB == 2 && ((NPA == 2 && NB == 2) || (NPA == 3 && NB == 1)));
  constexpr int ABYTES = BM * CA * 16, BBYTES = BN * CB * 16, SBYTES = SRC == PL_PLANES ? 0 : BN * 4;
  constexpr int BUF = ABYTES + BBYTES + SBYTES;
  constexpr int IA = (BM * CA / 64 + NW - 1) / NW, IB = (BN * CB / 64 + NW - 1) / NW;  // load instructions per wavefront and step
  constexpr int IS = SRC == PL_PLANES ? 0 : (BN / 64 + NW - 1) / NW;
  constexpr int LOADS = IA + IB + IS;
  static_assert(BM * CA % 64 == 0 && BN * CB % 64 == 0, "whole load instructions");
  extern __shared__ __align__(16) unsigned char smem[];
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)smem;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave / WN, wn = wave % WN;
  // tiles in bands of `band` rows of tiles, column by column within a band; each XCD takes an equal run of that order
  const int tile = (blockIdx.x & 7) * a.chunk + (blockIdx.x >> 3);
  if (tile >= a.tm * a.tn) return;
  const int b0 = tile / (a.band * a.tn), inb = tile - b0 * a.band * a.tn, height = min(a.band, a.tm - b0 * a.band);
  const int mi = b0 * a.band + inb % height, ni = inb / height;
  const int m0 = mi * BM, n0 = ni * BN;
  const int nsteps = a.nkb;
  const PlaneStore store(a);

  // where this lane's pieces of a step lie, as offsets from the step's bases; rows past the end repeat the last one
  unsigned avo[IA], bvo[IB], svo[IS > 0 ? IS : 1];
#pragma unroll
  for (int j = 0; j < IA; j++) {
    const int s = ((j * NW + wave) * 64 + lane) % (BM * CA), r = s / CA, c = (s % CA) ^ swz<CA, SPREAD>(r);
    avo[j] = (unsigned)(min(r, a.M - 1 - m0) * a.apitch + c * 16);
  }
#pragma unroll
  for (int j = 0; j < IB; j++) {
    const int s = ((j * NW + wave) * 64 + lane) % (BN * CB), r = s / CB, c = (s % CB) ^ swz<CB, SPREAD>(r);
    bvo[j] = (unsigned)(min(r, a.N - 1 - n0) * a.bpitch + c * 16);
  }
#pragma unroll
  for (int j = 0; j < IS; j++) {
    const int s = ((j * NW + wave) * 64 + lane) % BN;
    svo[j] = (unsigned)(min(s, a.N - 1 - n0) * a.dpitch) * 2u;
  }
  const unsigned char *ab = a.A + (int64_t)m0 * a.apitch;  // of the next step to ask for
  const unsigned char *bb = a.B + (int64_t)n0 * a.bpitch;
  const unsigned char *sb = SRC == PL_PLANES ? nullptr : (const unsigned char *)(a.bd + (int64_t)n0 * a.dpitch);
  unsigned al[IA], bl[IB], sl[IS > 0 ? IS : 1];  // where its pieces go, in the first buffer
#pragma unroll
  for (int j = 0; j < IA; j++) al[j] = lds0 + ((j * NW + wave) * 1024) % ABYTES;
#pragma unroll
  for (int j = 0; j < IB; j++) bl[j] = lds0 + ABYTES + ((j * NW + wave) * 1024) % BBYTES;
#pragma unroll
  for (int j = 0; j < IS; j++) sl[j] = lds0 + ABYTES + BBYTES + ((j * NW + wave) * 256) % (SBYTES ? SBYTES : 1);
  int left = nsteps;  // steps to ask for
  auto issue = [&](int buf) __attribute__((always_inline)) {
    const unsigned char *as = uniform(ab), *bs = uniform(bb);
#pragma unroll
    for (int j = 0; j < IA; j++) dma16(as, avo[j], al[j] + buf * BUF);
#pragma unroll
    for (int j = 0; j < IB; j++) dma16(bs, bvo[j], bl[j] + buf * BUF);
#pragma unroll
    for (int j = 0; j < IS; j++) dma2(uniform(sb), svo[j], sl[j] + buf * BUF);
    if (--left > 0) ab += CA * 16, bb += CB * 16, sb += 2;  // past the end: the last step again, so that the counts stay the same
  };

  v16f acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; i++)
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][b][r] = 0.0f;

  const int half = lane >> 5, col = lane & 31;
  constexpr bool EARLY = MB * NB < 8;  // (registers for it)
  float4 bias;
  if (EARLY) bias = plane_gemm_bias<NB>(store, n0 + 32 * NB * wn, lane);
  // k of the matrix instructions of a block: slice s, lane half h take k = 16 h + 8 s .. +7 (the same for A and B)
  v16f tmp[2][SRC == PL_INT ? MB : 1] = {};  // PL_INT: partial sums of a block of 32 k, unscaled
  float dlast = 0.0f;
  auto mul = [&](int buf) __attribute__((always_inline)) {
    const unsigned char *At = smem + buf * BUF, *Bt = At + ABYTES;
    const int ra = 32 * MB * wm + col, rb = 32 * NB * wn + col;
    auto lda = [&](int i, int ch) { return *(const uint4 *)(At + ((ra + 32 * i) * CA + (ch ^ swz<CA, SPREAD>(ra))) * 16); };
    auto ldb = [&](int b, int ch) { return *(const uint4 *)(Bt + ((rb + 32 * b) * CB + (ch ^ swz<CB, SPREAD>(rb))) * 16); };
    // The operands of a slice are read before the slice in front of it is multiplied, behind a scheduling fence: left alone
    // the compiler puts every LDS read right in front of its use, and each pair of matrix instructions waits out an LDS
    // round trip.
    v8bf af[2][MB][NPA], bf[2][NB][NPB];
    auto ld = [&](int s) __attribute__((always_inline)) {
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int p = 0; p < NPB; p++) bf[s][b][p] = __builtin_bit_cast(v8bf, ldb(b, p * 4 + 2 * half + s));
#pragma unroll
      for (int i = 0; i < MB; i++)
#pragma unroll
        for (int p = 0; p < NPA; p++) af[s][i][p] = __builtin_bit_cast(v8bf, lda(i, p * 4 + 2 * half + s));
    };
    ld(0);
    ld(1);
    if constexpr (SRC == PL_PLANES) {
#pragma unroll
      for (int s = 0; s < 2; s++) {
        __builtin_amdgcn_sched_barrier(0);
        // every pair of terms whose product is above 2^-8(terms) of the leading one, smallest first
#pragma unroll
        for (int t = (NPA > NPB ? NPA : NPB) - 1; t >= 0; t--)
#pragma unroll
          for (int p = 0; p <= t; p++)
            if (p < NPA && t - p < NPB)
#pragma unroll
              for (int i = 0; i < MB; i++)
#pragma unroll
                for (int b = 0; b < NB; b++) acc[i][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[s][i][p], bf[s][b][t - p], acc[i][b], 0, 0, 0);
      }
    } else {
      float d[NB];
#pragma unroll
      for (int b = 0; b < NB; b++) d[b] = half_bits_to_float((unsigned short)((const unsigned *)(Bt + BBYTES))[rb + 32 * b]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < NB; b++) asm("" : "+v"(d[b]));  // as a float: a multiply-add that converts its fp16 operand runs at half rate
      // The partial sums of one column block are scaled under the matrix instructions of the next one (of the next step's
      // first one for the last), a few multiply-adds behind each, which run while it occupies the matrix core.  An odd NB
      // carries nothing into the next step: its buffers would change places.
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const int pb = (b + NB - 1) % NB;
        const float dp = b ? d[b - 1] : dlast;
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
          for (int r = 0; r < 16; r++) tmp[b & 1][i][r] = 0.0f;
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
          for (int p = NPA - 1; p >= 0; p--)
#pragma unroll
            for (int i = 0; i < MB; i++) tmp[b & 1][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[s][i][p], bf[s][b][0], tmp[b & 1][i], 0, 0, 0);
        if (b > 0 || NB % 2 == 0)
#pragma unroll
          for (int i = 0; i < MB; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][pb][r] = fmaf(dp, tmp[(b & 1) ^ 1][i][r], acc[i][pb][r]);
#pragma unroll
        for (int q = 0; q < 2 * NPA * MB; q++) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x2, 8 / NPA, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      dlast = d[NB - 1];
      if (NB % 2)
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
          for (int r = 0; r < 16; r++) acc[i][NB - 1][r] = fmaf(dlast, tmp[0][i][r], acc[i][NB - 1][r]);
    }
  };

  if (nsteps > 0) {
#pragma unroll
    for (int s = 0; s < NBUF - 1; s++) issue(s);
    // Its buffer known to the compiler, a step has fewer instructions: where an LDS instruction's offset reaches all of them (256 x 256 at two terms: 362 us rolled, 398 not).
    constexpr bool UNROLL = NBUF * BUF <= 80 * 1024;
    int b0 = 0;
    for (int i = 0; i < nsteps;)
#pragma unroll
      for (int b1 = 0; b1 < (UNROLL ? NBUF : 1); b1++) {
        const int buf = UNROLL ? b1 : b0;
        wait_barrier<LOADS *(NBUF - 2)>();  // step i has landed; nobody reads the buffer of step i - 1 any more
        issue(buf == 0 ? NBUF - 1 : buf - 1);
        mul(buf);
        b0 = b0 + 1 == NBUF ? 0 : b0 + 1;
        if (++i == nsteps) break;
      }
  }
  wait_barrier<0>();
  if (SRC == PL_INT && NB % 2 == 0)
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][NB - 1][r] = fmaf(dlast, tmp[1][SRC == PL_INT ? i : 0][r], acc[i][NB - 1][r]);

  // ---- acc[i][b][r] is row 8 (r / 4) + 4 half + r % 4, column `col` of its block.  A wavefront turns its blocks around
  // in a piece of LDS of its own (no barrier) and stores rows of 32 NB columns, 16 bytes per lane.
  if (!EARLY) bias = plane_gemm_bias<NB>(store, n0 + 32 * NB * wn, lane);
  constexpr int LDC = 32 * NB + 4;
  float *Cs = (float *)smem + wave * 32 * LDC;
#pragma unroll
  for (int i = 0; i < MB; i++) {
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int r = 0; r < 16; r++) Cs[(8 * (r >> 2) + 4 * half + (r & 3)) * LDC + 32 * b + col] = acc[i][b][r];
    __builtin_amdgcn_wave_barrier();
    plane_gemm_store_rows<NB, EARLY ? 4 : 1>(store, Cs, m0 + 32 * (MB * wm + i), n0 + 32 * NB * wn, lane, bias);
    __builtin_amdgcn_wave_barrier();
  }
}

// ---- operands -> planes ----
// fp32 / fp16 rows (R, K) with pitch ld: a thread takes 8 consecutive k.  kbp: blocks of a plane row (k past K are zeros)
template <int NP, typename T, bool VEC>
__global__ __launch_bounds__(256) void k_planes_rows(uint4 *__restrict__ out, const T *__restrict__ x, int64_t R, int K, int64_t ld, int kbp) {
  const int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int per = kbp * 4;
  if (u >= R * per) return;
  const int64_t row = u / per;
  const int c = (int)(u - row * per), k = 8 * c;
  float v[8];
  const T *p = x + row * ld + k;
  if (VEC) {
    if (k < K) {
      if constexpr (sizeof(T) == 4) {
        const float4 t0 = *(const float4 *)p, t1 = *(const float4 *)(p + 4);
        v[0] = t0.x, v[1] = t0.y, v[2] = t0.z, v[3] = t0.w, v[4] = t1.x, v[5] = t1.y, v[6] = t1.z, v[7] = t1.w;
      } else {
        const uint4 t = *(const uint4 *)p;
        const unsigned w[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
        for (int j = 0; j < 4; j++) v[2 * j] = half_bits_to_float((unsigned short)(w[j] & 0xffff)), v[2 * j + 1] = half_bits_to_float((unsigned short)(w[j] >> 16));
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; j++) v[j] = 0.0f;
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = k + j < K ? (float)p[j] : 0.0f;
  }
  uint4 pl[NP];
  split8_planes<NP>(v, pl);
#pragma unroll
  for (int q = 0; q < NP; q++) out[(row * kbp + (c >> 2)) * (4 * NP) + 4 * q + (c & 3)] = pl[q];
}

// (K, N) row-major -> planes of its columns (N rows of K): a workgroup turns 64 k x 64 n around in LDS
template <int NP, bool VEC>
__global__ __launch_bounds__(256) void k_planes_cols(uint4 *__restrict__ out, const float *__restrict__ x, int K, int N, int kbp) {
  __shared__ float T[64][65];
  const int k0 = blockIdx.y * 64, n0 = blockIdx.x * 64, tid = threadIdx.x;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int k = k0 + (tid >> 4) + 16 * j, n = n0 + 4 * (tid & 15);
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (k < K) {
      const float *p = x + (int64_t)k * N + n;
      if (VEC) {
        if (n < N) v = *(const float4 *)p;
      } else {
        if (n < N) v.x = p[0];
        if (n + 1 < N) v.y = p[1];
        if (n + 2 < N) v.z = p[2];
        if (n + 3 < N) v.w = p[3];
      }
    }
    float *t = &T[(tid >> 4) + 16 * j][4 * (tid & 15)];
    t[0] = v.x, t[1] = v.y, t[2] = v.z, t[3] = v.w;
  }
  __syncthreads();
  const int n = tid >> 2;
  if (n0 + n >= N) return;
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int c = 2 * (tid & 3) + j;  // chunk of 8 k within the 64
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = T[8 * c + e][n];
    uint4 pl[NP];
    split8_planes<NP>(v, pl);
    if (k0 / 32 + (c >> 2) < kbp)
#pragma unroll
      for (int q = 0; q < NP; q++) out[((int64_t)(n0 + n) * kbp + k0 / 32 + (c >> 2)) * (4 * NP) + 4 * q + (c & 3)] = pl[q];
  }
}

// quant plane of a Q8_0 / Q4_0 matrix -> one plane of its integers: a thread takes 8 consecutive k
template <bool Q4>
__global__ __launch_bounds__(256) void k_planes_int(uint4 *__restrict__ out, const unsigned char *__restrict__ q, int64_t n8) {
  const int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;  // rows are whole blocks: the planes are as contiguous as the quants
  if (u >= n8) return;
  unsigned a, b;
  if (Q4) {
    const uint2 t = *(const uint2 *)(q + (u >> 2) * 16 + 8 * (u & 1));
    const int sh = (u & 2) ? 4 : 0;  // k 0..15 of a block are the low nibbles of its bytes, 16..31 the high ones
    a = (((t.x >> sh) & 0x0f0f0f0fu) + 0x78787878u) ^ 0x80808080u;  // per byte: nibble - 8 as int8 (no carry leaves a byte)
    b = (((t.y >> sh) & 0x0f0f0f0fu) + 0x78787878u) ^ 0x80808080u;
  } else {
    const uint2 t = *(const uint2 *)(q + u * 8);
    a = t.x, b = t.y;
  }
  out[u] = __builtin_bit_cast(uint4, bf_of_q8(a, b));
}

template <int NPA, int SRC, int NPB, int MB, int NB, int WM, int WN, int NBUF>
static int planes_launch(PlaneGemmArgs a) {
  constexpr int BM = 32 * MB * WM, BN = 32 * NB * WN;
  constexpr size_t buf = (size_t)BM * 64 * NPA + (size_t)BN * 64 * NPB + (SRC == PL_PLANES ? 0 : BN * 4);
  constexpr size_t turn = (size_t)WM * WN * 32 * (32 * NB + 4) * 4;
  constexpr size_t lds = NBUF * buf > turn ? NBUF * buf : turn;
  static_assert(lds <= 160 * 1024, "LDS");
  a.tm = (a.M + BM - 1) / BM;
  a.tn = (a.N + BN - 1) / BN;
  a.chunk = (a.tm * a.tn + 7) / 8;
  double best = -1.0;
  for (int bands = 1; bands <= 8 && bands <= a.tm; bands++) {  // the band height for the least operand bytes per L2
    const int h = (a.tm + bands - 1) / bands;
    const double score = (double)h * BM * NPA + ((double)a.chunk / h + 1.0) * BN * NPB;
    if (best < 0 || score < best) best = score, a.band = h;
  }
  auto fn = k_gemm_planes<NPA, SRC, NPB, MB, NB, WM, WN, NBUF>;
  static bool big_lds = false;
  if (!big_lds && lds > 64 * 1024) {
    CTHIP_CHECK(hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    big_lds = true;
  }
  hipLaunchKernelGGL(fn, dim3(8u * a.chunk), dim3(64 * WM * WN), lds, state().stream, a);
  CTHIP_LAUNCH_CHECK();
  return 0;
}

// A x B^T for operands in planes.  terms: of A; a.bd non-null: B is one plane of integers with scales, else terms_b planes.
static int planes_gemm(const PlaneGemmArgs &a, int terms, int terms_b) {
  const bool q = a.bd != nullptr;
  const int pick = plane_pick(a.M, a.N, a.nkb, terms, q, state().compute_units).tile;
#define T(NPA, SRC, NPB, MB, NB, WM, WN) return planes_launch<NPA, SRC, NPB, MB, NB, WM, WN, 2>(a)
#define T3(NPA, SRC, NPB, MB, NB, WM, WN) return planes_launch<NPA, SRC, NPB, MB, NB, WM, WN, 3>(a)
#define TILES(NPA)                                  \
  switch (pick) {                                   \
    case 0: T(NPA, PL_PLANES, NPA, 1, 1, 2, 2);     \
    case 1: T(NPA, PL_PLANES, NPA, 2, 1, 2, 2);     \
    case 2: T(NPA, PL_PLANES, NPA, 2, 1, 2, 4);     \
    case 3: T(NPA, PL_PLANES, NPA, 2, 2, 2, 2);     \
    case 4: T(NPA, PL_PLANES, NPA, 4, 2, 2, 4);     \
  }
#define QTILES(NPA)                                    \
  switch (pick) {                                      \
    case 0: T3(NPA, PL_INT, 1, 1, 1, 2, 2);            \
    case 1: T3(NPA, PL_INT, 1, 2, 2, 2, 2);            \
    case 2: T(NPA, PL_INT, 1, 2, 3, 2, 2);             \
  }
  if (q) {
    if (terms == 2) QTILES(2)
    else QTILES(1)
  } else if (terms == 3 && terms_b == 2) {
    switch (pick) {
      case 0: T(3, PL_PLANES, 2, 1, 1, 2, 2);
      case 1: T(3, PL_PLANES, 2, 2, 1, 2, 2);
      case 2: T(3, PL_PLANES, 2, 2, 2, 2, 4);
    }
  } else if (terms == 3) {
    switch (pick) {
      case 0: T(3, PL_PLANES, 3, 1, 1, 2, 2);
      case 1: T(3, PL_PLANES, 3, 2, 1, 2, 2);
      case 2: T(3, PL_PLANES, 3, 2, 2, 2, 4);
    }
  } else if (terms == 2) {
    TILES(2)
  } else {
    TILES(1)
  }
#undef T
#undef T3
#undef QTILES
#undef TILES
  return fail(CTHIP_E_STATE, "gemm planes: no tile (%d terms)", terms);
}

template <typename T>
static int planes_rows(unsigned char *out, const T *x, int64_t rows, int K, int64_t ld, int terms) {
  const int kbp = (K + 31) / 32;
  const int64_t blocks = (rows * kbp * 4 + 255) / 256;
  if (blocks > 0x7fffffff) return fail(CTHIP_E_BAD_ARG, "gemm planes: operand too large");
  const bool vec = K % 8 == 0 && ld % 8 == 0 && (uintptr_t)x % 16 == 0;
#define PR(NP)                                                                                                                             \
  do {                                                                                                                                     \
    if (vec) hipLaunchKernelGGL((k_planes_rows<NP, T, true>), dim3((unsigned)blocks), dim3(256), 0, state().stream, (uint4 *)out, x, rows, K, ld, kbp); \
    else hipLaunchKernelGGL((k_planes_rows<NP, T, false>), dim3((unsigned)blocks), dim3(256), 0, state().stream, (uint4 *)out, x, rows, K, ld, kbp);    \
  } while (0)
  if (terms == 3) PR(3);
  else if (terms == 2) PR(2);
  else PR(1);
#undef PR
  CTHIP_LAUNCH_CHECK();
  return 0;
}

static void planes_operands(PlaneGemmArgs &a, int K, int terms, int terms_b) {
  a.nkb = (K + 31) / 32;
  a.apitch = a.nkb * 64 * terms;
  a.bpitch = a.nkb * 64 * terms_b;
}

// C = act(A . B + bias) + residual with B (K, N) row-major.  *done stays false, and the caller takes the other path, where the
// results do not lie on 16 bytes or there is no memory for the terms.
int launch_matmul_planes(float *C, const float *A, const float *B, int M, int N, int K, int act, const float *bias, const float *residual, int precision,
                         bool *done) {
  if (N % 4 == 0 && (((uintptr_t)C | (uintptr_t)bias | (uintptr_t)residual) & 15)) return 0;
  const int terms = plane_terms(precision);
  PlaneGemmArgs a = {};
  a.C = C;
  a.M = M, a.N = N;
  a.act = act;
  a.bias = bias, a.residual = residual;
  planes_operands(a, K, terms, terms);
  unsigned char *pa = nullptr;
  const size_t abytes = (size_t)M * a.apitch, bbytes = (size_t)N * a.bpitch;
  if (stream_capturing() || alloc_scratch((void **)&pa, abytes + bbytes + 256)) return 0;  // fully written by the two passes
  *done = true;
  int rc = 0;
  unsigned char *pb = pa + (abytes + 255) / 256 * 256;
  rc = planes_rows<float>(pa, A, M, K, K, terms);
  if (!rc) {
    const dim3 grid((N + 63) / 64, (K + 63) / 64);
    const bool vec = N % 4 == 0 && (uintptr_t)B % 16 == 0;
#define PC(NP)                                                                                                             \
  do {                                                                                                                     \
    if (vec) hipLaunchKernelGGL((k_planes_cols<NP, true>), grid, dim3(256), 0, state().stream, (uint4 *)pb, B, K, N, a.nkb); \
    else hipLaunchKernelGGL((k_planes_cols<NP, false>), grid, dim3(256), 0, state().stream, (uint4 *)pb, B, K, N, a.nkb);    \
  } while (0)
    if (terms == 3) PC(3);
    else if (terms == 2) PC(2);
    else PC(1);
#undef PC
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) rc = fail((int)e, "gemm planes: launch -> %s", hipGetErrorString(e));
  }
  a.A = pa, a.B = pb;
  if (!rc) rc = planes_gemm(a, terms, terms);
  const int rf = cthip_free(pa);  // stream-ordered: handed out again only to later work on this stream
  return rc ? rc : rf;
}
bool matmul_planes_pay(int M, int N, int K, int precision) { return matmul_planes_faster(M, N, K, precision, state().compute_units); }

// ---- Linears over many rows ----
// A weight matrix as planes: one of integers for a quantised matrix (2 bytes per weight), two exact terms for fp16 (4).
// The first Linear that wants them makes them and they stay with the matrix, up to a limit for all matrices together
// (option "weight_planes"; what a 16-bit model of 16e9 weights takes, a ninth of the card), as long as a sixteenth of the card
// stays free; they go with the matrix, when an allocation fails, with cthip_cache_trim and with a lower limit.  Past that, for
// fp32 matrices and for a single term of an fp16 one they are made again by every call, 3 - 8 bytes of traffic per weight.
static std::mutex g_planes_mu;  // guards the fields planes* of every matrix, and:
static int64_t g_planes_limit = 32ll << 30, g_planes_bytes = 0;
static std::unordered_set<WMat *> g_planes_of;

static bool is_quant(const WMat *w) { return w->type == CTHIP_Q8_0 || w->type == CTHIP_Q4_0; }
static int weight_terms(const WMat *w, int terms) {
  if (w->type == CTHIP_Q4_0 && terms == 2) return kDigits;
  return is_quant(w) ? 1 : w->type == CTHIP_F16 && terms > 2 ? 2 : terms;
}
int linear_terms(const WMat *w, int precision) { return weight_terms(w, plane_terms(precision)) == kDigits ? kTermsDigits : kTermsPlanes; }
static int64_t weight_plane_bytes(const WMat *w, int terms_b) {
  return terms_b == kDigits ? digit_weight_bytes(w) : w->rows * ((w->cols + 31) / 32) * 64 * terms_b;
}
static bool weight_planes_stay(const WMat *w, int terms_b) { return is_quant(w) || (w->type == CTHIP_F16 && terms_b == 2); }

static int make_weight_planes(unsigned char *out, const WMat *w, int terms_b) {
  const int K = (int)w->cols;
  if (terms_b == kDigits) return make_weight_digits(out, w);
  if (w->type == CTHIP_F16) return planes_rows<_Float16>(out, (const _Float16 *)w->q, w->rows, K, K, terms_b);
  if (w->type == CTHIP_F32) return planes_rows<float>(out, (const float *)w->q, w->rows, K, K, terms_b);
  const int64_t n8 = w->rows * K / 8;
  if ((n8 + 255) / 256 > 0x7fffffff) return fail(CTHIP_E_BAD_ARG, "gemm planes: operand too large");
  const dim3 grid((unsigned)((n8 + 255) / 256));
  if (w->type == CTHIP_Q4_0) hipLaunchKernelGGL(k_planes_int<true>, grid, dim3(256), 0, state().stream, (uint4 *)out, (const unsigned char *)w->q, n8);
  else hipLaunchKernelGGL(k_planes_int<false>, grid, dim3(256), 0, state().stream, (uint4 *)out, (const unsigned char *)w->q, n8);
  CTHIP_LAUNCH_CHECK();
  return 0;
}
// A matrix of 4 bits is held in both of its forms where both are asked for (one term in bf16, two as digits); where there is room for one alone, the one that nobody uses goes.
static WMat::Form &form_of(const WMat *w, int terms_b) { return const_cast<WMat *>(w)->forms[terms_b == kDigits]; }
static int64_t form_spare(const WMat *w, int terms_b) {  // (with g_planes_mu held) bytes of the other form that can go
  const WMat::Form &o = w->forms[terms_b != kDigits];
  return o.p && !o.users ? o.bytes : 0;
}
// Whether they are there or the next call's stay (with g_planes_mu held)
static bool weight_planes_room(const WMat *w, int terms_b) {
  return weight_planes_stay(w, terms_b) && (form_of(w, terms_b).p || g_planes_bytes - form_spare(w, terms_b) + weight_plane_bytes(w, terms_b) <= g_planes_limit);
}
static bool weight_planes_kept(const WMat *w, int terms_b) {
  std::lock_guard<std::mutex> lk(g_planes_mu);
  return weight_planes_room(w, terms_b);
}
static void form_give_back(WMat::Form &f) {  // (stream-ordered: the block goes to later work on this stream only)
  cthip_free(f.p);
  g_planes_bytes -= f.bytes;
  f = {};
}
// The terms for one launch, null where there is no memory for them (or for terms that stay, where temp is null).  *temp:
// the caller frees them after its launch, else it calls weight_planes_release.
static const unsigned char *weight_planes(const WMat *w, int terms_b, bool *temp) {
  std::lock_guard<std::mutex> lk(g_planes_mu);
  WMat::Form &f = form_of(w, terms_b);
  const int64_t bytes = weight_plane_bytes(w, terms_b);
  const bool stay = weight_planes_room(w, terms_b);
  if (stay && f.p) {
    f.users++;
    if (temp) *temp = false;
    return (const unsigned char *)f.p;
  }
  if (!stay && !temp) return nullptr;
  if (stay && g_planes_bytes + bytes > g_planes_limit) form_give_back(const_cast<WMat *>(w)->forms[terms_b != kDigits]);
  unsigned char *p = nullptr;
  if (alloc_spare((void **)&p, (size_t)bytes)) return nullptr;
  if (make_weight_planes(p, w, terms_b)) {
    cthip_free(p);
    return nullptr;
  }
  if (stay) {
    f.p = p;
    f.bytes = bytes;
    f.users = 1;
    g_planes_bytes += bytes;
    g_planes_of.insert(const_cast<WMat *>(w));
  }
  if (temp) *temp = !stay;
  return p;
}
void weight_planes_release(const WMat *w, int precision) {
  std::lock_guard<std::mutex> lk(g_planes_mu);
  form_of(w, weight_terms(w, plane_terms(precision))).users--;
}
void wmat_drop_planes(WMat *w) {
  std::lock_guard<std::mutex> lk(g_planes_mu);
  for (WMat::Form &f : w->forms)
    if (f.p) form_give_back(f);
  g_planes_of.erase(w);
}
bool weight_planes_drop() {
  std::lock_guard<std::mutex> lk(g_planes_mu);
  bool any = false;
  for (auto it = g_planes_of.begin(); it != g_planes_of.end();) {
    bool left = false;
    for (WMat::Form &f : (*it)->forms) {
      if (f.p && !f.users) form_give_back(f), any = true;
      left = left || f.p;
    }
    it = left ? std::next(it) : g_planes_of.erase(it);
  }
  return any;
}
void weight_planes_limit(int64_t bytes) {
  bool over;
  {
    std::lock_guard<std::mutex> lk(g_planes_mu);
    g_planes_limit = bytes;
    over = g_planes_bytes > bytes;
  }
  if (over) weight_planes_drop();
}

bool linear_planes_pays(const WMat *w, int m, int precision, bool planes_in, bool prompt, bool shares) {
  if (precision == GEMM_FP32 || m < 64 || w->rows < 64 || w->cols < 64 || (!is_quant(w) && w->cols % 16)) return false;
  // (three terms against integers: registers for one 32-column block less per wavefront, no faster than the tiles)
  if (is_quant(w) && precision == GEMM_BF16X6) return false;
  const int terms = plane_terms(precision), terms_b = weight_terms(w, terms);
  const double w_bytes = weight_planes_kept(w, terms_b) ? 0.0 : (double)w->q_bytes + weight_plane_bytes(w, terms_b);
  const double x_bytes = planes_in ? 0.0 : (double)m * w->cols * (4 + 2 * terms);
  if (terms_b == kDigits) {
    if (!digits_fit((int)w->cols)) return false;
    // A prompt whose digits stay: always.  (Six layers, 65 / 256 / 950 rows, tiles alone and digits alone: 384 wide 347 / 364 / 434 and 307 / 325 / 419 us, GPT-2 small 403 / 405 / 701 and
    // 355 / 375 / 544, 1.1B shape 600 / 747 / 2032 and 528 / 615 / 1243, 7B shape 1452 / 2106 / 7201 and 1019 / 1384 / 3607; nowhere between 65 and 1900 rows are tiles the faster ones, and
    // chosen Linear by Linear the small models were up to 15 % slower than digits alone.)
    // Past the limit: memory that is only lent for a launch, where that is long.
    if (prompt && w_bytes == 0.0) return true;
    if (prompt && m < 512) return false;
    return linear_digits_faster(m, (int)w->rows, (int)w->cols, w->type, x_bytes, w_bytes, shares, state().compute_units);
  }
  return linear_planes_faster(m, (int)w->rows, (int)w->cols, precision, w->type, w_bytes + x_bytes, prompt, state().compute_units);
}
// ... and nothing can be in the way of it
bool linear_planes_ready(const WMat *w, int m, int precision) {
  return linear_planes_pays(w, m, precision, true, true) && weight_planes(w, weight_terms(w, plane_terms(precision)), nullptr);
}
int launch_linear_planes(float *y, const WMat *w, const float *x, const unsigned char *xplanes, int m, const float *bias, const float *residual, int act,
                         int precision, const GemmRoute *route, unsigned char *planes_out, int out_terms, bool prompt, GemmDeferred *defer, bool *done) {
  const int K = (int)w->cols, terms = plane_terms(precision), terms_b = weight_terms(w, terms);
  const bool digits = terms_b == kDigits;
  DigitGemmArgs a = {};
  a.C = y;
  a.M = m, a.N = (int)w->rows;
  a.bias = bias, a.residual = residual;
  a.act = act;
  uintptr_t at = (uintptr_t)y | (uintptr_t)bias | (uintptr_t)residual;
  if (act == kActSwigluPairs) {
    if (a.N % 4 || residual || route) return 0;
    a.act = CTHIP_ACT_NONE;
    a.pairs = 1;
  }
  if (route) {
    for (int i = 0; i < 3; i++)
      if (route->c0[i] != INT_MAX) at |= (uintptr_t)route->dst[i] | (route->c0[i] % 4 || route->ld[i] % 4 ? 1 : 0);
    if (route->c0[0] != 0 || residual || a.N % 4) return 0;
    a.routed = 1;
    a.route = *route;
  }
  if (a.N % 4 == 0 && (at & 15)) return 0;
  if (planes_out) {
    const int width = a.pairs ? a.N / 2 : a.N;
    if (terms != 2 || a.N % 4 || width % 32 || (out_terms == kTermsDigits && !digits)) return 0;
    if (out_terms == kTermsDigits) a.digits = planes_out;
    else a.planes = (unsigned short *)planes_out;
    a.pkb = width / 32;
  }
  planes_operands(a, K, terms, terms_b);
  if (is_quant(w) && !digits) {
    a.bd = (const unsigned short *)w->d;
    a.dpitch = a.nkb;
  }
  unsigned char *tmp = nullptr;
  if (stream_capturing() || (!xplanes && alloc_scratch((void **)&tmp, digits ? (size_t)digit_row_bytes(m, a.nkb) : (size_t)m * a.apitch)))
    return 0;  // written by the pass in front, but for rows that reach no result
  bool temp_b = false;
  const unsigned char *pb = weight_planes(w, terms_b, &temp_b);
  if (!pb) {
    cthip_free(tmp);
    return 0;
  }
  *done = true;
  int rc = xplanes ? 0 : digits ? launch_rows_digits(tmp, x, m, K, CTHIP_PRO_NONE, nullptr, nullptr, 0.0f) : planes_rows<float>(tmp, x, m, K, K, terms);
  a.A = xplanes ? xplanes : tmp, a.B = pb;
  if (!rc && digits) {
    // Shares of K: left to the caller, or added up (with bias and residual) by a launch of their own
    const bool plain = a.act == CTHIP_ACT_NONE && !a.pairs && !a.routed && !planes_out;
    const int out = !a.digits ? kDigitsPlain : a.pairs ? kDigitsOutPairs : kDigitsOut;
    DigitsPick pick = digits_pick(m, a.N, a.nkb, out, plain, defer != nullptr, state().compute_units);
    float *ws = nullptr;
    if (pick.ks > 1 && alloc_scratch((void **)&ws, sizeof(float) * (size_t)pick.ks * m * a.N)) pick = digits_pick(m, a.N, a.nkb, out, false, false, state().compute_units);
    if (ws) a.C = ws, a.bias = a.residual = nullptr;
    rc = digits_gemm(a, pick);
    if (ws && defer && !rc) {
      defer->ws = ws;
      defer->ksplit = pick.ks;
    } else if (ws) {
      if (!rc) rc = launch_splitk_reduce(y, ws, pick.ks, m, a.N, bias, residual);
      cthip_free(ws);  // stream-ordered: handed out again only to later work on this stream
    }
  } else if (!rc) {
    rc = planes_gemm(a, terms, terms_b);
  }
  cthip_free(tmp);  // stream-ordered: handed out again only to later work on this stream
  if (temp_b) cthip_free(const_cast<unsigned char *>(pb));
  else weight_planes_release(w, precision);
  return rc;
}

}  // namespace cthip
