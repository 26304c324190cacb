// MFMA GEMM over 6-bit digits: Linears over many rows on weights of 4 bits at two bf16 terms' precision.
//
// gemm_planes.hip multiplies the rows' two bf16 terms by the integers of a quantised matrix: four v_mfma_f32_32x32x16_bf16 (32 cycles each) per block of 32 x 32 results and
// 32 k.  An integer of 4 bits is also a float of 6 bits, and a value of a row is four such digits with a power of two each (digits.h).  v_mfma_scale_f32_32x32x64_f8f6f4
// multiplies them at four times the rate, K = 64 holding two digits of a block against the same weights twice, and applies the powers of two itself: two instructions
// of 38 cycles per block, 96 bytes per row and block instead of 128, 24 per column instead of 64.  The block's scale is one multiply-add per result, as there.
// What is lost: 2^-19 of a block's largest value, where two bf16 terms lose 2^-18 of each value.  Measured against 64 bits over rows of normal values 1.03e-6 (two terms:
// 2.46e-6), with every 37th column 100 times as large 2.1e-6 (2.3e-6), values of wide range, exp(2 x), 2.2 - 2.35e-6 (2.1 - 2.4e-6).  Results that the largest values do not reach would
// lose more: blocks with values far above the others have what three digits leave as two bf16 terms besides (digits.h: which, and what that leaves of the loss).
//
// us, operands in place / planes: 1900 x 11264 x 2048 134 / 194, 1900 x 2048 x 5632 71 / 117, 1900 x 2560 x 2048 38 / 70; prompt of 1900 rows, 1.1B shape, 10.9 -> 7.7 ms, of 300, 7B shape,
// 16.2 -> 8.7.  What bounds it: large products the power limit (a card at 1.5 - 1.8 GHz there; a step of two workgroups of 128 x 256 was 2550 cycles, of which the matrix
// cores were busy 1220 and the vector ALU 1024 with the scales; without the loads 160 us instead of 205 at 2.1 GHz, without the scales 91: variants with parts left
// out) and single wavefronts' instructions (a step with a seventh fewer of them was 5 - 15 % faster); small ones the latency of a step, 0.24 us, and a launch's ends, 5 us.
#include "common.h"
#include "digits.h"
#include "gemm_plan.h"

namespace cthip {

// MB x NB blocks of 32 x 32 per wavefront, WM x WN wavefronts, NBUF LDS buffers; a step is a block of 32 k.
// OUT: what becomes of the sums (gemm_plan.h).
template <int MB, int NB, int WM, int WN, int KB, int NBUF, int OUT>
__global__ __launch_bounds__(64 * WM * WN, MB * NB * KB <= 2 ? 4 : MB * NB <= 4 ? 3 : 2) void k_gemm_digits(DigitGemmArgs a) {
  constexpr int NW = WM * WN, BM = 32 * MB * WM, BN = 32 * NB * WN, NBLK = MB * NB;
  static_assert(NBLK * KB % 2 == 0, "the sums of a step's last block wait for the next step's first: two sets in turn");
  constexpr int ABYTES = BM * 96, BBYTES = BN * 32, SBYTES = BM * 4;
  constexpr int PART = ABYTES + BBYTES + SBYTES, BUF = KB * PART;
  constexpr int NA = ABYTES / 1024, NBL = BBYTES / 1024, NS = BM / 64;  // load instructions of a step
  constexpr int IA = (NA + NW - 1) / NW, IB = (NBL + NW - 1) / NW, IS = (NS + NW - 1) / NW;
  constexpr int LOADS = KB * (IA + IB + IS);
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
  const PlaneStore store(a);
  unsigned char *const digits = early(a.digits);
  const int nkb = a.nkb, k0 = blockIdx.y * a.kper, nsteps = min(a.kper, nkb - k0);  // of this share (none is empty)

  // where this lane's pieces of a step lie, as offsets from the step's bases; groups of rows past the end repeat the last one
  const int mg = (a.M + 31) / 32, ng = (a.N + 31) / 32;
  unsigned avo[IA], bvo[IB], svo[IS];
#pragma unroll
  for (int j = 0; j < IA; j++) {
    const int s = (j * NW + wave) % NA;
    avo[j] = (unsigned)min(s / 3, mg - 1 - m0 / 32) * (unsigned)(nkb * kDigitRecord) + (s % 3) * 1024 + lane * 16;
  }
#pragma unroll
  for (int j = 0; j < IB; j++) bvo[j] = (unsigned)min((j * NW + wave) % NBL, ng - 1 - n0 / 32) * (unsigned)(nkb * kDigitWRecord) + lane * 16;
#pragma unroll
  for (int j = 0; j < IS; j++) svo[j] = (unsigned)min(((j * NW + wave) % NS) * 64 + lane, mg * 32 - 1 - m0) * 4u;
  const unsigned char *ab = a.A + ((int64_t)(m0 / 32) * nkb + k0) * kDigitRecord;
  const unsigned char *bb = a.B + ((int64_t)(n0 / 32) * nkb + k0) * kDigitWRecord;
  const unsigned char *sb = a.A + (int64_t)mg * nkb * kDigitRecord + ((int64_t)k0 * mg * 32 + m0) * 4;
  unsigned al[IA], bl[IB], sl[IS];  // where they go, in the first buffer
#pragma unroll
  for (int j = 0; j < IA; j++) al[j] = lds0 + ((j * NW + wave) % NA) * 1024;
#pragma unroll
  for (int j = 0; j < IB; j++) bl[j] = lds0 + ABYTES + ((j * NW + wave) % NBL) * 1024;
#pragma unroll
  for (int j = 0; j < IS; j++) sl[j] = lds0 + ABYTES + BBYTES + ((j * NW + wave) % NS) * 256;
  int left = nsteps;  // steps to ask for
  auto issue = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < KB; k++) {
      const unsigned char *as = uniform(ab), *bs = uniform(bb), *ss = uniform(sb);
#pragma unroll
      for (int j = 0; j < IA; j++) dma16(as, avo[j], al[j] + buf * BUF + k * PART);
#pragma unroll
      for (int j = 0; j < IB; j++) dma16(bs, bvo[j], bl[j] + buf * BUF + k * PART);
#pragma unroll
      for (int j = 0; j < IS; j++) dma4(ss, svo[j], sl[j] + buf * BUF + k * PART);
      if (--left > 0) ab += kDigitRecord, bb += kDigitWRecord, sb += mg * 128;  // past the end: the last block again, so that the counts stay the same
    }
  };

  // (the bias is there long before it is needed)
  const int half = lane >> 5, col = lane & 31;
  float bias[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) bias[b] = a.col_bias ? a.col_bias[min(n0 + 32 * (NB * wn + b) + col, a.N - 1)] : 0.0f;
  v16f acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; i++)
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][b][r] = 0.0f;

  v16f tmp[2] = {};  // sums over a block of 32 k, unscaled
  float dlast = 0.0f;
  unsigned least[MB];  // of this lane's pairs of exponents: below 256 where the upper one is 0
#pragma unroll
  for (int i = 0; i < MB; i++) least[i] = 0xffffu;
  // both: the step has all of its KB blocks (an odd number of blocks: the last one's second half counts for nothing)
  auto mul = [&](int buf, bool both) __attribute__((always_inline)) {
    uint4 a16[KB][MB][2], b16[KB][NB];
    uint2 a8[KB][MB][2], b8[KB][NB];
    int sc[KB][MB];
    float d[KB][NB];
    // (behind a fence: left alone the compiler puts every LDS read right in front of its use)
#pragma unroll
    for (int k = 0; k < KB; k++) {
      const unsigned char *At = smem + buf * BUF + k * PART + MB * wm * kDigitRecord, *Bt = smem + buf * BUF + k * PART + ABYTES + NB * wn * kDigitWRecord;
      const unsigned char *St = smem + buf * BUF + k * PART + ABYTES + BBYTES + MB * wm * 128;
      auto lda = [&](int i) __attribute__((always_inline)) {
        sc[k][i] = *(const unsigned short *)(St + i * 128 + col * 4 + half * 2);
#pragma unroll
        for (int j = 1; j >= 0; j--) {
          a16[k][i][j] = *(const uint4 *)(At + i * kDigitRecord + j * 1024 + lane * 16);
          a8[k][i][j] = *(const uint2 *)(At + i * kDigitRecord + 2048 + j * 512 + lane * 8);
          asm volatile("" ::: "memory");  // (two 8-byte reads made one would not land behind their 16 bytes)
        }
      };
      auto ldb = [&](int b) __attribute__((always_inline)) {
        b16[k][b] = *(const uint4 *)(Bt + b * kDigitWRecord + col * 16);
        b8[k][b] = *(const uint2 *)(Bt + b * kDigitWRecord + 512 + col * 8);
        d[k][b] = *(const float *)(Bt + b * kDigitWRecord + 768 + col * 4);
        asm volatile("" ::: "memory");
      };
      lda(0);
      ldb(0);
#pragma unroll
      for (int i = 1; i < MB; i++) lda(i);
#pragma unroll
      for (int b = 1; b < NB; b++) ldb(b);
    }
    if (KB == 1) issue((buf + NBUF - 1) % NBUF);  // while they are on their way
    __builtin_amdgcn_sched_barrier(0);
    // the sums of a block are scaled under the matrix instructions of the next one (of the next step's first one for the last)
#pragma unroll
    for (int q = 0; q < KB * NBLK; q++) {
      const int k = q / NBLK, b = q % NBLK / MB, i = q % MB, prev = (q + KB * NBLK - 1) % (KB * NBLK), pk = prev / NBLK, pb = prev % NBLK / MB, pi = prev % MB;
      if (KB > 1 && k == KB - 1 && q % NBLK == 0)
#pragma unroll
        for (int n = 0; n < NB; n++) d[k][n] = both ? d[k][n] : 0.0f;
      const float dp = q ? d[pk][pb] : dlast;
      const v8i_dg bv = {(int)b16[k][b].x, (int)b16[k][b].y, (int)b16[k][b].z, (int)b16[k][b].w, (int)b8[k][b].x, (int)b8[k][b].y, 0, 0};
      v16f t;
#pragma unroll
      for (int r = 0; r < 16; r++) t[r] = 0.0f;
#pragma unroll
      for (int j = 1; j >= 0; j--) {  // the small digits first
        const v8i_dg av = {(int)a16[k][i][j].x, (int)a16[k][i][j].y, (int)a16[k][i][j].z, (int)a16[k][i][j].w, (int)a8[k][i][j].x, (int)a8[k][i][j].y, 0, 0};
        t = j ? __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv, t, 2, 2, 1, sc[k][i], 0, 127) : __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv, t, 2, 2, 0, sc[k][i], 0, 127);
      }
      tmp[q & 1] = t;
#pragma unroll
      for (int r = 0; r < 16; r++) acc[pi][pb][r] = fmaf(dp, tmp[(q & 1) ^ 1][r], acc[pi][pb][r]);
#pragma unroll
      for (int g = 0; g < 2; g++) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, 8, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    dlast = d[KB - 1][NB - 1];
#pragma unroll
    for (int k = 0; k < KB; k++)
#pragma unroll
      for (int i = 0; i < MB; i++) least[i] = min(least[i], (unsigned)sc[k][i]);
  };

#pragma unroll
  for (int s = 0; s < NBUF - 1; s++) issue(s);
  for (int i = 0; i < nsteps;)
#pragma unroll
    for (int buf = 0; buf < NBUF; buf++) {  // (its buffer known to the compiler, a step has a seventh fewer instructions)
      wait_barrier<LOADS *(NBUF - 2)>();  // step i has landed; nobody reads the buffer of step i - 1 any more
      if (KB > 1) issue((buf + NBUF - 1) % NBUF);  // (few workgroups: as early as can be)
      mul(buf, KB == 1 || i + KB <= nsteps);
      if ((i += KB) >= nsteps) break;
    }
  wait_barrier<0>();
#pragma unroll
  for (int r = 0; r < 16; r++) acc[MB - 1][NB - 1][r] = fmaf(dlast, tmp[1][r], acc[MB - 1][NB - 1][r]);

  // ---- what three digits left of blocks that have it as terms (digits.h), of this wavefront's own rows.  Rare: one look at a wavefront's exponents, and where one is 0 all of the
  // share's again, 32 blocks of k at a time; a block is the four instructions of two bf16 terms against the same weights.  (us with the pass that makes the digits, no such block / a
  // column of all of K / every block: 1900 x 11264 x 2048 150 / 158 / 400, 1900 x 2048 x 5632 92 / 95 / 235, 280 x 12288 x 4096 62 / 65 / 162; two bf16 terms in place, without their pass:
  // 194 and 117 for the first two.  Every block is 128 bytes a row for every tile of columns, by every wavefront for itself.)
  bool look = false, mine[MB];
#pragma unroll
  for (int i = 0; i < MB; i++) {
    mine[i] = m0 + 32 * (MB * wm + i) + col < a.M;
    look = look || __any(mine[i] && least[i] < 256u);
  }
  if (look) {
    const unsigned char *words = a.A + (int64_t)mg * nkb * kDigitRecord + (int64_t)k0 * mg * 128;
    const unsigned char *rests = a.A + (int64_t)mg * nkb * (kDigitRecord + kDigitScales) + (int64_t)k0 * kDigitRests + lane * 16;
    int group[MB];  // (past the end: not this wavefront's)
#pragma unroll
    for (int i = 0; i < MB; i++) group[i] = min(m0 / 32 + MB * wm + i, mg - 1);
    const unsigned upper = half ? ~0u : 0u;
    auto word_of = [&](int i, int kb) __attribute__((always_inline)) { return *(const unsigned *)(words + ((int64_t)kb * mg + group[i]) * 128 + col * 4); };
    auto terms_of = [&](int i, int kb, uint4 *t) __attribute__((always_inline)) {  // the small term first
      const uint4 *r = (const uint4 *)(rests + ((int64_t)group[i] * nkb + kb) * kDigitRests);
      t[0] = r[128], t[1] = r[192], t[2] = r[0], t[3] = r[64];
    };
    auto weights_of = [&](int b, int kb, uint4 &w16, uint2 &w8, float &dw) __attribute__((always_inline)) {
      const unsigned char *w = a.B + ((int64_t)min(n0 / 32 + NB * wn + b, ng - 1) * nkb + k0 + kb) * kDigitWRecord;
      w16 = *(const uint4 *)(w + col * 16);
      w8 = *(const uint2 *)(w + 512 + col * 8);
      dw = *(const float *)(w + 768 + col * 4);
    };
    auto own = [&](int i, unsigned word, uint4 *t) __attribute__((always_inline)) {  // (rows that have none: nothing was written there)
      const unsigned has = mine[i] & (word < 0x1000000u) ? ~0u : 0u;
#pragma unroll
      for (int q = 0; q < 4; q++) t[q].x &= has, t[q].y &= has, t[q].z &= has, t[q].w &= has;
    };
    auto add = [&](int b, const uint4 (*t)[4], uint4 w16, uint2 w8, float dw) __attribute__((always_inline)) {
      const v6u_dg six = {w16.x, w16.y, w16.z, w16.w, w8.x, w8.y};
      const auto all = __builtin_bit_cast(v16u_dg, __builtin_amdgcn_cvt_scalef32_pk32_bf16_fp6(six, 1.0f));
      unsigned mid[8];  // k 16 half .. + 15  (not a choice of two elements, which is made one of sixteen)
#pragma unroll
      for (int e = 0; e < 8; e++) mid[e] = all[e] ^ ((all[e] ^ all[8 + e]) & upper);
      const uint4 k8[2] = {make_uint4(mid[0], mid[1], mid[2], mid[3]), make_uint4(mid[4], mid[5], mid[6], mid[7])};
#pragma unroll
      for (int i = 0; i < MB; i++) {
        v16f p;
#pragma unroll
        for (int e = 0; e < 16; e++) p[e] = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; q++) p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, t[i][q]), __builtin_bit_cast(v8bf, k8[q & 1]), p, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 16; e++) acc[i][b][e] = fmaf(dw, p[e], acc[i][b][e]);
      }
    };
#pragma unroll 1
    for (int c = 0; c < nsteps; c += 32) {
      unsigned any = 0;
#pragma unroll
      for (int i = 0; i < MB; i++) {
        const int rows = a.M - 32 * (m0 / 32 + MB * wm + i) - 4 * (lane & 7);  // of the four whose exponents this lane looks at
        uint4 word[4];
#pragma unroll
        for (int u = 0; u < 4; u++) word[u] = *(const uint4 *)(words + ((int64_t)min(c + 8 * u + (lane >> 3), nsteps - 1) * mg + group[i]) * 128 + (lane & 7) * 16);
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const bool has = ((word[u].x < 0x1000000u) & (rows > 0)) | ((word[u].y < 0x1000000u) & (rows > 1)) | ((word[u].z < 0x1000000u) & (rows > 2)) | ((word[u].w < 0x1000000u) & (rows > 3));
          uint64_t t = __ballot(has & (c + 8 * u + (lane >> 3) < nsteps));  // eight lanes to a block of k
          t |= t >> 4, t |= t >> 2, t |= t >> 1;
          any |= (unsigned)((t & 0x0101010101010101ull) * 0x0102040810204080ull >> 56) << (8 * u);
        }
      }
      if constexpr (KB == 2) {
        // a block's loads asked for under the one before it, where there are registers for both (1900 x 2048 x 5632, every block, 285 -> 235 us)
        struct {
          unsigned word[MB];
          uint4 t[MB][4], w16[NB];
          uint2 w8[NB];
          float dw[NB];
        } now, next;
        auto ask = [&](int kb) __attribute__((always_inline)) {
#pragma unroll
          for (int i = 0; i < MB; i++) next.word[i] = word_of(i, kb), terms_of(i, kb, next.t[i]);
#pragma unroll
          for (int b = 0; b < NB; b++) weights_of(b, kb, next.w16[b], next.w8[b], next.dw[b]);
        };
        if (any) ask(c + __builtin_ctz(any));
#pragma unroll 1
        while (any) {
          now = next;
          any &= any - 1;
          if (any) ask(c + __builtin_ctz(any));
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < MB; i++) own(i, now.word[i], now.t[i]);
#pragma unroll
          for (int b = 0; b < NB; b++) add(b, now.t, now.w16[b], now.w8[b], now.dw[b]);
        }
      } else {
#pragma unroll 1
        for (; any; any &= any - 1) {
          const int kb = c + __builtin_ctz(any);
          unsigned word[MB];
          uint4 t[MB][4];
#pragma unroll
          for (int i = 0; i < MB; i++) word[i] = word_of(i, kb), terms_of(i, kb, t[i]);
#pragma unroll
          for (int i = 0; i < MB; i++) own(i, word[i], t[i]);
#pragma unroll
          for (int b = 0; b < NB; b++) {
            uint4 w16;
            uint2 w8;
            float dw;
            weights_of(b, kb, w16, w8, dw);
            add(b, t, w16, w8, dw);
          }
        }
      }
    }
  }

  // ---- acc[i][b][r] is row 8 (r / 4) + 4 half + r % 4, column `col` of its block.  A wavefront turns its blocks around in a piece of LDS of its own
  // (no barrier) and stores rows of 32 NB columns, 16 bytes per lane, or a block of 32 columns of a row per lane as digits.
  // (Small code: a launch of a few steps waits for its own instructions.)
  constexpr int LDC = 32 * NB + 4, C4 = 8 * NB;
  float *Cs = (float *)smem + wave * 32 * LDC;
  const int col0 = n0 + 32 * NB * wn, c4 = lane % C4, at = col0 + 4 * c4;  // a lane stores the same four columns of every 64 / C4-th row
#pragma unroll
  for (int i = 0; i < MB; i++) {
    const int row0 = m0 + 32 * (MB * wm + i);
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int r = 0; r < 16; r++) Cs[(8 * (r >> 2) + 4 * half + (r & 3)) * LDC + 32 * b + col] = acc[i][b][r] + bias[b];
    __builtin_amdgcn_wave_barrier();
    if constexpr (OUT == kDigitsOut || OUT == kDigitsOutPairs) {
      constexpr int PER = OUT == kDigitsOutPairs ? 2 : 1;  // columns per result
      static_assert(NB % PER == 0, "whole blocks of results");
#pragma unroll 1
      for (int u = lane; u < 32 * NB / PER; u += 64) {
        const int c = (u >> 5) * 32 * PER, row = row0 + col;
        if (col0 + c >= store.N) continue;  // (the same for a block's 32 lanes)
        const float *p = Cs + col * LDC + c;
        float v[32];
#pragma unroll
        for (int q = 0; q < 8 * PER; q++) {
          const float4 t = *(const float4 *)(p + 4 * q);
          if (PER == 2) v[2 * q] = ct_silu(t.x) * t.y, v[2 * q + 1] = ct_silu(t.z) * t.w;
          else v[4 * q] = t.x, v[4 * q + 1] = t.y, v[4 * q + 2] = t.z, v[4 * q + 3] = t.w;
        }
        if (PER == 1 && store.act == CTHIP_ACT_GELU) {
#pragma unroll
          for (int q = 0; q < 32; q++) v[q] = ct_gelu(v[q]);
        }
        const float m = digits_top(v);
        const bool rest = digits_uneven_columns(v, m, row < store.M) || digits_one_large(v, m);
        if (row < store.M) store_digits32(digits, (int64_t)mg * 32, store.pkb, row, (col0 + c) / (32 * PER), v, m, rest);
      }
    } else if constexpr (OUT == kDigitsPlain) {
      plane_gemm_store_rows<NB>(store, Cs, row0, col0, lane, make_float4(0.0f, 0.0f, 0.0f, 0.0f));
    } else {
#pragma unroll 1
      for (int r = lane / C4; r < 32; r += 64 / C4) {
        const int row = row0 + r;
        const float4 v = *(const float4 *)(Cs + r * LDC + 4 * c4);
        if (row >= store.M || at >= store.N) continue;
        float *p = store.C + ((int64_t)blockIdx.y * store.M + row) * store.N + at;
        if (store.N % 4 == 0) {
          *(float4 *)p = v;
        } else {
          p[0] = v.x;
          if (at + 1 < store.N) p[1] = v.y;
          if (at + 2 < store.N) p[2] = v.z;
          if (at + 3 < store.N) p[3] = v.w;
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// Q4_0 -> digits: a thread takes a block of a row
__global__ __launch_bounds__(256) void k_digits_q4(unsigned char *__restrict__ out, const unsigned char *__restrict__ q, const unsigned short *__restrict__ d, int64_t rows, int nkb) {
  const int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t rec = u >> 5, row = rec / nkb * 32 + (u & 31);
  const int kb = (int)(rec % nkb);
  if (rec >= (rows + 31) / 32 * nkb) return;
  unsigned w[6] = {};
  float s = 0.0f;
  if (row < rows) {
    const uint4 t = *(const uint4 *)(q + (row * nkb + kb) * 16);
    s = 2.0f * half_bits_to_float(d[row * nkb + kb]);
    const unsigned in[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
    for (int i = 0; i < 32; i++) {  // k 0 .. 15 of a block are the low nibbles of its bytes, 16 .. 31 the high ones
      const unsigned n = (in[(i & 15) >> 2] >> (8 * (i & 3) + (i >= 16 ? 4 : 0))) & 15u;
      // |n - 8| halves in six bits: 0, 4, 8, 12, 16, 18, 20, 22, 24
      const unsigned m = n < 8 ? 8 - n : n - 8, c = (m <= 4 ? 4 * m : 8 + 2 * m) | (n < 8 ? 32u : 0u);
      w[6 * i / 32] |= c << (6 * i % 32);
      if (6 * i % 32 > 26) w[6 * i / 32 + 1] |= c >> (32 - 6 * i % 32);
    }
  }
  unsigned char *r = out + rec * kDigitWRecord;
  *(uint4 *)(r + (u & 31) * 16) = make_uint4(w[0], w[1], w[2], w[3]);
  *(uint2 *)(r + 512 + (u & 31) * 8) = make_uint2(w[4], w[5]);
  *(float *)(r + 768 + (u & 31) * 4) = s;
}

int64_t digit_weight_bytes(const WMat *w) { return (w->rows + 31) / 32 * (w->cols / 32) * kDigitWRecord; }
int make_weight_digits(unsigned char *out, const WMat *w) {
  const int nkb = (int)(w->cols / 32);
  const int64_t blocks = ((w->rows + 31) / 32 * nkb * 32 + 255) / 256;
  if (blocks > 0x7fffffff) return fail(CTHIP_E_BAD_ARG, "gemm digits: operand too large");
  hipLaunchKernelGGL(k_digits_q4, dim3((unsigned)blocks), dim3(256), 0, state().stream, out, (const unsigned char *)w->q, (const unsigned short *)w->d, w->rows, nkb);
  CTHIP_LAUNCH_CHECK();
  return 0;
}

// ---- rows -> digits ----
// A workgroup takes eight blocks of 32 rows, a block of a row per thread, through LDS: a wavefront reads 1024 bytes of a row at a time, and neighbouring lanes hold the same block of
// neighbouring rows, whose 16-byte pieces of a digit lie side by side.
__global__ __launch_bounds__(256) void k_digits_rows(unsigned char *__restrict__ out, const float *__restrict__ x, int64_t rows, int K) {
  constexpr int PITCH = 36, BLOCK = 32 * PITCH + 32;  // floats between rows and blocks: no two of the 16 lanes of a 16-byte access meet in a bank
  __shared__ __align__(16) float turn[8 * BLOCK];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nkb = K >> 5;
  const int64_t row0 = (int64_t)blockIdx.x * 32;
  const int kb0 = blockIdx.y * 8, at = min(kb0 * 32 + 4 * lane, K - 4);
  f4_any v4[8];  // (rows at any alignment)
#pragma unroll
  for (int j = 0; j < 8; j++) v4[j] = *(const f4_any *)(x + min(row0 + wave + 4 * j, rows - 1) * K + at);
#pragma unroll
  for (int j = 0; j < 8; j++) *(f4_any *)&turn[(lane >> 3) * BLOCK + (wave + 4 * j) * PITCH + 4 * (lane & 7)] = v4[j];
  __syncthreads();
  const int r = tid & 31, kb = kb0 + (tid >> 5);
  if (kb >= nkb) return;  // (the same for a block's 32 lanes)
  float v[32];
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const float4 f = *(const float4 *)&turn[(tid >> 5) * BLOCK + r * PITCH + 4 * q];
    v[4 * q] = f.x, v[4 * q + 1] = f.y, v[4 * q + 2] = f.z, v[4 * q + 3] = f.w;
  }
  const float m = digits_top(v);
  const bool rest = digits_uneven_columns(v, m, row0 + r < rows) || digits_one_large(v, m);
  if (row0 + r < rows) store_digits32(out, (rows + 31) / 32 * 32, nkb, row0 + r, kb, v, m, rest);
}

// The same behind a norm, a wavefront per row (V4 float4 per lane) while it is normalised, four rows to a workgroup; then 64 blocks of the four rows at a time through LDS.
// (A row's blocks in its own wavefront's lanes, 16 bytes stored every 3072: 1900 rows of 2048 13.4 us.)
template <int PRO, int V4>
__global__ __launch_bounds__(256) void k_rows_digits(unsigned char *__restrict__ out, const float *__restrict__ x, int64_t rows, int K, const float *__restrict__ g,
                                                     const float *__restrict__ b, float eps) {
  constexpr int RS = 64 * 36 + 16;  // blocks 36 floats apart and rows 4 banks: no two of the 16 lanes of a 16-byte access meet in a bank
  __shared__ __align__(16) float turn[4 * RS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n4 = K >> 2, nkb = K >> 5;
  const int64_t row0 = (int64_t)blockIdx.x * 4;
  const float4 *xr = (const float4 *)(x + min(row0 + wave, rows - 1) * K);
  const int crow = threadIdx.x & 3, cblk = threadIdx.x >> 2;  // what this thread converts
  float4 v[V4], gm[V4], bt[PRO == CTHIP_PRO_LAYERNORM ? V4 : 1];
#pragma unroll
  for (int j = 0; j < V4; j++) v[j] = xr[min(lane + 64 * j, n4 - 1)];
#pragma unroll
  for (int j = 0; j < V4; j++) {
    gm[j] = ((const float4 *)(g ? g : x))[min(lane + 64 * j, n4 - 1)];
    if (PRO == CTHIP_PRO_LAYERNORM) bt[j] = ((const float4 *)(b ? b : x))[min(lane + 64 * j, n4 - 1)];
  }
  const float inv_n = 1.0f / (float)K;
  float mean = 0.0f, q = 0.0f;
  if (PRO == CTHIP_PRO_LAYERNORM) {
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < V4; j++) s += lane + 64 * j < n4 ? (v[j].x + v[j].y) + (v[j].z + v[j].w) : 0.0f;
    mean = wave_sum(s) * inv_n;
  }
#pragma unroll
  for (int j = 0; j < V4; j++) {
    v[j].x -= mean, v[j].y -= mean, v[j].z -= mean, v[j].w -= mean;
    q += lane + 64 * j < n4 ? (v[j].x * v[j].x + v[j].y * v[j].y) + (v[j].z * v[j].z + v[j].w * v[j].w) : 0.0f;
  }
  const float rstd = 1.0f / sqrtf(wave_sum(q) * inv_n + eps);
#pragma unroll
  for (int j = 0; j < V4; j++) {
    v[j].x *= rstd, v[j].y *= rstd, v[j].z *= rstd, v[j].w *= rstd;
    if (g) v[j].x *= gm[j].x, v[j].y *= gm[j].y, v[j].z *= gm[j].z, v[j].w *= gm[j].w;
    if (PRO == CTHIP_PRO_LAYERNORM && b) v[j].x += bt[j].x, v[j].y += bt[j].y, v[j].z += bt[j].z, v[j].w += bt[j].w;
  }
#pragma unroll
  for (int c = 0; c < V4; c += 8) {
    const int kb0 = 8 * c;
    if (kb0 >= nkb) break;
    if (c) __syncthreads();
#pragma unroll
    for (int j = 0; j < 8 && j < V4; j++) *(float4 *)&turn[wave * RS + (lane / 8 + 8 * j) * 36 + 4 * (lane % 8)] = make_float4(v[c + j].x, v[c + j].y, v[c + j].z, v[c + j].w);
    __syncthreads();
    if (kb0 + cblk < nkb && cblk < 8 * V4 && row0 + crow < rows) {
      float t[32];
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float4 f = *(const float4 *)&turn[crow * RS + cblk * 36 + 4 * i];
        t[4 * i] = f.x, t[4 * i + 1] = f.y, t[4 * i + 2] = f.z, t[4 * i + 3] = f.w;
      }
      const float m = digits_top(t);
      store_digits32(out, (rows + 31) / 32 * 32, nkb, row0 + crow, kb0 + cblk, t, m, digits_uneven(t, m) || digits_one_large(t, m));
    }
  }
}
// (K a multiple of 32; a norm: x, g and b on 16 bytes, K <= 8192)
int launch_rows_digits(void *digits, const float *x, int m, int K, int pro, const float *g, const float *b, float eps) {
  if (K % 32 || (pro != CTHIP_PRO_NONE && !rows_digits_supported(K))) return fail(CTHIP_E_BAD_ARG, "rows of %d as digits", K);
  const dim3 grid((m + 3) / 4);
#define RD(PRO, V4) hipLaunchKernelGGL((k_rows_digits<PRO, V4>), grid, dim3(256), 0, state().stream, (unsigned char *)digits, x, (int64_t)m, K, g, b, eps)
#define RDN(PRO)                      \
  do {                                \
    if (K <= 1024) RD(PRO, 4);        \
    else if (K <= 2048) RD(PRO, 8);   \
    else if (K <= 4096) RD(PRO, 16);  \
    else RD(PRO, 32);                 \
  } while (0)
  if (pro == CTHIP_PRO_LAYERNORM) RDN(CTHIP_PRO_LAYERNORM);
  else if (pro == CTHIP_PRO_RMSNORM) RDN(CTHIP_PRO_RMSNORM);
  else hipLaunchKernelGGL(k_digits_rows, dim3((m + 31) / 32, (K / 32 + 7) / 8), dim3(256), 0, state().stream, (unsigned char *)digits, x, (int64_t)m, K);
#undef RDN
#undef RD
  CTHIP_LAUNCH_CHECK();
  return 0;
}

template <int MB, int NB, int WM, int WN, int KB, int NBUF, int OUT>
static int digits_launch_as(DigitGemmArgs a, int ks) {
  constexpr int BM = 32 * MB * WM, BN = 32 * NB * WN;
  constexpr size_t buf = KB * ((size_t)BM * 100 + (size_t)BN * 32), turn = (size_t)WM * WN * 32 * (32 * NB + 4) * 4;
  constexpr size_t lds = NBUF * buf > turn ? NBUF * buf : turn;
  static_assert(lds <= 64 * 1024, "what a launch may ask for without an attribute, and two workgroups to a compute unit and more");
  a.col_bias = a.bias, a.bias = nullptr;
  a.tm = (a.M + BM - 1) / BM;
  a.tn = (a.N + BN - 1) / BN;
  a.chunk = (a.tm * a.tn + 7) / 8;
  a.kper = (a.nkb + ks - 1) / ks;
  double best = -1.0;
  for (int bands = 1; bands <= 8 && bands <= a.tm; bands++) {  // the band height for the least operand bytes per L2
    const int h = (a.tm + bands - 1) / bands;
    const double score = (double)h * BM * 100 + ((double)a.chunk / h + 1.0) * BN * 32;
    if (best < 0 || score < best) best = score, a.band = h;
  }
  auto fn = k_gemm_digits<MB, NB, WM, WN, KB, NBUF, OUT>;
  hipLaunchKernelGGL(fn, dim3(8u * a.chunk, (a.nkb + a.kper - 1) / a.kper), dim3(64 * WM * WN), lds, state().stream, a);
  CTHIP_LAUNCH_CHECK();
  return 0;
}
template <int MB, int NB, int WM, int WN, int KB, int NBUF>
static int digits_launch(const DigitGemmArgs &a, int ks) {
  if (ks > 1) return digits_launch_as<MB, NB, WM, WN, KB, NBUF, kDigitsShares>(a, ks);
  if (!a.digits) return digits_launch_as<MB, NB, WM, WN, KB, NBUF, kDigitsPlain>(a, 1);
  if constexpr (NB % 2 == 0)
    if (a.pairs) return digits_launch_as<MB, NB, WM, WN, KB, NBUF, kDigitsOutPairs>(a, 1);
  if (a.pairs || a.residual || a.routed || (a.act != CTHIP_ACT_NONE && a.act != CTHIP_ACT_GELU)) return fail(CTHIP_E_STATE, "gemm digits: no such epilogue in front of digits");
  return digits_launch_as<MB, NB, WM, WN, KB, NBUF, kDigitsOut>(a, 1);
}
// A x B^T for rows and weights as digits.  pick.ks > 1: raw sums, share after share, at a.C (no bias, activation, residual or other destination).
int digits_gemm(const DigitGemmArgs &a, const DigitsPick &pick) {
  if (pick.ks > 1 && (a.bias || a.residual || a.act != CTHIP_ACT_NONE || a.pairs || a.routed || a.planes || a.digits))
    return fail(CTHIP_E_STATE, "gemm digits: shares of K with an epilogue");
  if (pick.tile == 2) return digits_launch<2, 2, 2, 2, 1, 3>(a, pick.ks);
  if (pick.tile == 0) return digits_launch<1, 1, 2, 2, 2, 3>(a, pick.ks);
  // Up to two workgroups to a compute unit: two blocks of k a step, two steps ahead, for weights out of memory (280 x 12288 x 4096 58 -> 55 us, 1900 x 2048 x 5632 82 -> 71,
  // 100 x 3072 x 1024 13.8 -> 12.3).  More: four workgroups (1900 x 11264 x 2048 164 -> 133).
  if (pick.fullest <= 2) return digits_launch<1, 2, 2, 2, 2, 3>(a, pick.ks);
  return digits_launch<1, 2, 2, 2, 1, 3>(a, pick.ks);
}

}  // namespace cthip
