// Attention of a long prompt on bf16 matrix instructions, keys and values split into terms once.
//
// k_attn_mfma_bf (rowops.hip) converts every key / value tile it reads: 60 blocks of 32 query rows times 8 query heads of a group
// repeat the same conversions (4800 cycles of a 32 x 32 tile, 768 of them matrix instructions).  Here a small launch
// writes the keys as rows of two bf16 terms and the values transposed (32 keys of one element of the head side by side, in
// the order a lane supplies them to the second product); the attention kernel moves tiles of both to LDS by direct
// loads and spends its vector instructions on the softmax.  The same products as there: hi*hi + hi*lo + lo*hi.
//   S^T = K Q^T : lane l feeds K[key l%32][d = 16 s + 8 (l/32) .. +7] and Q[query l%32][the same d] (registers)
//   O^T += V^T P^T : registers 8 t .. 8 t + 7 of a lane are keys 16 t + 8 (e/4) + 4 (l/32) + e%4
// A wavefront owns 32 query rows of one head; a workgroup's wavefronts share a key / value head, so its tiles are read
// once for all of them.  What bounds it now: 24 matrix instructions and 210 vector instructions (the softmax and the split of P) a
// tile, which overlap little; interleaving the next tile's scores with a tile's exponentials, operands in registers a step
// early, and more or fewer wavefronts per SIMD all measured the same or slower.
// With the launch that splits: 1900 rows, 32 heads on 4 key / value heads of 64: 130 -> 66 us; 32 heads of 128: 234 -> 118 us.
#include "common.h"
#include "digits.h"

namespace cthip {

// ---- keys and values -> terms.  One workgroup per (block of 32 keys, key / value head). ----
template <int DH>
__global__ __launch_bounds__(256) void k_attn_split(unsigned short *__restrict__ kp, unsigned short *__restrict__ vp, const float *__restrict__ kc,
                                                    const float *__restrict__ vc, int T, int Hkv) {
  __shared__ float vt[32][DH + 1];
  const int kb = blockIdx.x, hk = blockIdx.y, tid = threadIdx.x, nkb = gridDim.x;
  const int64_t KD = (int64_t)Hkv * DH;
  const int64_t tile = ((int64_t)hk * nkb + kb) * (64 * DH);  // elements: 32 keys, 2 terms
  for (int f = tid; f < 8 * DH; f += 256) {
    const int key = f / (DH / 4), d = 4 * (f % (DH / 4)), row = 32 * kb + key;
    float4 k = make_float4(0.f, 0.f, 0.f, 0.f), v = k;
    if (row < T) {
      k = *(const float4 *)(kc + row * KD + hk * DH + d);
      v = *(const float4 *)(vc + row * KD + hk * DH + d);
    }
    uint2 pl[2];
    split4_planes<2>(k.x, k.y, k.z, k.w, pl);
    unsigned short *o = kp + tile + key * (2 * DH) + d;
    *(uint2 *)o = pl[0];
    *(uint2 *)(o + DH) = pl[1];
    vt[key][d] = v.x, vt[key][d + 1] = v.y, vt[key][d + 2] = v.z, vt[key][d + 3] = v.w;
  }
  __syncthreads();
  for (int f = tid; f < 4 * DH; f += 256) {  // eight keys of one element: chunk 2 t + half
    const int d = f % DH, c = f / DH;
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; e++) x[e] = vt[16 * (c >> 1) + 8 * (e >> 2) + 4 * (c & 1) + (e & 3)][d];
    uint4 pl[2];
    split8_planes<2>(x, pl);
    uint4 *o = (uint4 *)(vp + tile + d * 64) + c;
    o[0] = pl[0];
    o[4] = pl[1];
  }
}

struct AttnPlanesArgs {
  float *out;                  // (S, H, DH), or null:
  unsigned short *out_planes;  // rows of two terms for gemm_planes.hip
  unsigned char *out_digits;   // rows for gemm_digits.hip
  const float *q;              // (S, H, DH)
  const unsigned char *kp, *vp;
  int S, start, H, Hkv, nkb;   // nkb: blocks of 32 keys
  int units;                   // per key / value head: blocks of 32 rows x heads of the group
};

// NW units a workgroup, two wavefronts to each: one takes the even key tiles, the other the odd ones.  (With one wavefront per unit the longest
// workgroup is alone on its compute unit for half of its tiles, one wavefront per SIMD: 64 us.)
template <int DH, int NW>
__global__ __launch_bounds__(128 * NW) void k_attn_planes(AttnPlanesArgs a) {
  constexpr int NSL = DH / 16, DB = DH / 32;
  constexpr int KT = 128 * DH, BUF = 4 * KT, NBUF = DH == 64 ? 3 : 2;  // bytes of a key (value) tile; a step: two tiles of both
  constexpr int CK = DH / 4;                                           // 16-byte chunks of a key row (8 of a value row)
  constexpr int LD = BUF / 1024 / (2 * NW);                                  // load instructions per wavefront and tile
  static_assert(BUF % (2048 * NW) == 0 && KT % 1024 == 0, "whole load instructions");
  extern __shared__ __align__(16) unsigned char smem[];
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)smem;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, col = lane & 31, unit = wv % NW, odd = wv / NW;
  const int item = blockIdx.x;  // the longest first
  const int hk = item % a.Hkv, group = a.H / a.Hkv;
  const int u0 = max(0, a.units - NW * (item / a.Hkv + 1)), u = min(u0 + unit, a.units - 1);  // (the last one overlaps its neighbour)
  const int qb = u / group, h = hk * group + u % group, i0 = 32 * qb;
  const int ulast = min(u0 + NW - 1, a.units - 1);
  const int wg_tiles = (a.start + min(32 * (ulast / group) + 32, a.S) + 31) / 32;
  const int my_tiles = (a.start + min(i0 + 32, a.S) + 31) / 32;
  const int qrow = min(i0 + col, a.S - 1), Tq = a.start + qrow + 1;

  unsigned voff[LD];
  bool isv[LD];
#pragma unroll
  for (int j = 0; j < LD; j++) {
    const int p = (wv * LD + j) * 64 + lane;  // chunk of the buffer: keys of both tiles, then values of both
    isv[j] = wv * LD + j >= 2 * KT / 1024;
    const int pk = isv[j] ? p - 2 * KT / 16 : p, cpr = isv[j] ? 8 : CK, r = pk / cpr, c = pk % cpr;
    voff[j] = (unsigned)(r * cpr + (c ^ (isv[j] ? (r >> 1) & 7 : r & 15))) * 16u;  // (which lanes a read serves together: swz in gemm_planes.hip)
  }
  const unsigned char *kbase = a.kp + (int64_t)hk * a.nkb * KT, *vbase = a.vp + (int64_t)hk * a.nkb * KT;
  auto issue = [&](int t, int buf) __attribute__((always_inline)) {
    t = min(2 * t, (a.nkb - 1) & ~1);  // (an odd number of tiles: the launcher leaves room for one more)
    const unsigned char *ks = uniform(kbase + (int64_t)t * KT), *vs = uniform(vbase + (int64_t)t * KT);
    const unsigned base = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)(buf * BUF));
#pragma unroll
    for (int j = 0; j < LD; j++) dma16(isv[j] ? vs : ks, voff[j], base + (wv * LD + j) * 1024);
  };
#pragma unroll
  for (int s = 0; s < NBUF - 1; s++) issue(s, s);

  // the query rows, scaled by log2(e) / sqrt(DH): scores are exponents of two
  v8bf qh[NSL], ql[NSL];
  {
    const float scale = 1.4426950408889634f / sqrtf((float)DH);
    const float *qp = a.q + ((int64_t)qrow * a.H + h) * DH + 8 * half;
#pragma unroll
    for (int s = 0; s < NSL; s++) {
      const float4 t0 = *(const float4 *)(qp + 16 * s), t1 = *(const float4 *)(qp + 16 * s + 4);
      const float x[8] = {t0.x * scale, t0.y * scale, t0.z * scale, t0.w * scale, t1.x * scale, t1.y * scale, t1.z * scale, t1.w * scale};
      uint4 pl[2];
      split8_planes<2>(x, pl);
      qh[s] = __builtin_bit_cast(v8bf, pl[0]);
      ql[s] = __builtin_bit_cast(v8bf, pl[1]);
    }
  }
  float m = -INFINITY, l = 0.0f;
  v16f o[DB];
#pragma unroll
  for (int d = 0; d < DB; d++)
#pragma unroll
    for (int r = 0; r < 16; r++) o[d][r] = 0.0f;

  auto work = [&](int t, const unsigned char *Kt) __attribute__((always_inline)) {
    const unsigned char *Vt = Kt + 2 * KT;
    v16f s0, s1;
#pragma unroll
    for (int r = 0; r < 16; r++) s0[r] = s1[r] = 0.0f;
    auto kld = [&](int term, int s) { return __builtin_bit_cast(v8bf, *(const uint4 *)(Kt + (col * CK + ((term * (DH / 8) + 2 * s + half) ^ (col & 15))) * 16)); };
#pragma unroll
    for (int s = 0; s < NSL; s++) {
      const v8bf kh = kld(0, s), kl = kld(1, s);
      s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kl, qh[s], s1, 0, 0, 0);
      s0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kh, qh[s], s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kh, ql[s], s1, 0, 0, 0);
    }
    // register r: key 32 t + 8 (r/4) + 4 half + r%4 against query `col`
    float tmax = -INFINITY;
    if (32 * t + 31 >= a.start + i0 + 1) {  // (uniform) some query does not see all of the tile
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int key = 32 * t + 8 * (r >> 2) + 4 * half + (r & 3);
        s0[r] = key < Tq ? s0[r] + s1[r] : -INFINITY;
        tmax = fmaxf(tmax, s0[r]);
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; r++) {
        s0[r] += s1[r];
        tmax = fmaxf(tmax, s0[r]);
      }
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float m_new = fmaxf(m, tmax), m_use = m_new == -INFINITY ? 0.0f : m_new;  // (no key of these tiles visible to this query yet)
    if (__any(m_new > m)) {
      const float corr = __builtin_amdgcn_exp2f(m - m_use);
      l *= corr;
#pragma unroll
      for (int d = 0; d < DB; d++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[d][r] *= corr;
      m = m_new;
    }
    float p[16], ps[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int r = 0; r < 16; r++) {
      p[r] = __builtin_amdgcn_exp2f(s0[r] - m_use);
      ps[r & 3] += p[r];
    }
    l += (ps[0] + ps[1]) + (ps[2] + ps[3]);
#pragma unroll
    for (int t2 = 0; t2 < 2; t2++) {
      uint4 pl[2];
      split8_planes<2>(p + 8 * t2, pl);
      const v8bf ph = __builtin_bit_cast(v8bf, pl[0]), pw = __builtin_bit_cast(v8bf, pl[1]);
#pragma unroll
      for (int d = 0; d < DB; d++) {
        const int row = 32 * d + col;
        const v8bf vh = __builtin_bit_cast(v8bf, *(const uint4 *)(Vt + (row * 8 + ((2 * t2 + half) ^ ((row >> 1) & 7))) * 16));
        const v8bf vl = __builtin_bit_cast(v8bf, *(const uint4 *)(Vt + (row * 8 + ((4 + 2 * t2 + half) ^ ((row >> 1) & 7))) * 16));
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vl, ph, o[d], 0, 0, 0);
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vh, pw, o[d], 0, 0, 0);
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vh, ph, o[d], 0, 0, 0);
      }
    }
  };
  int buf = 0;
  for (int t = 0; 2 * t < wg_tiles; t++) {
    wait_barrier<LD *(NBUF - 2)>();  // step t has landed; nobody reads the buffer of step t - 1 any more
    issue(t + NBUF - 1, buf == 0 ? NBUF - 1 : buf - 1);
    if (2 * t + odd < my_tiles) work(2 * t + odd, smem + buf * BUF + odd * KT);
    buf = buf + 1 == NBUF ? 0 : buf + 1;
  }
  wait_barrier<0>();

  // the odd tiles' wavefront hands over (maximum, sum, unnormalised outputs)
  l += __shfl_xor(l, 32, 64);
  float *mine = (float *)smem + (unit * (16 * DB + 2)) * 64 + lane;
  if (odd) {
    mine[0] = m;
    mine[64] = l;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int r = 0; r < 16; r++) mine[(2 + 16 * d + r) * 64] = o[d][r];
  }
  __syncthreads();
  if (odd) return;
  {
    const float m1 = mine[0], M = fmaxf(m, m1);  // finite: this wavefront saw key 0
    const float e0 = __builtin_amdgcn_exp2f(m - M), e1 = __builtin_amdgcn_exp2f(m1 - M);
    l = l * e0 + mine[64] * e1;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int r = 0; r < 16; r++) o[d][r] = o[d][r] * e0 + mine[(2 + 16 * d + r) * 64] * e1;
  }
  const float inv = 1.0f / l;
  if (a.out_digits) {
    // a lane's halves of two blocks of 32 -> one whole block: lanes 0 .. 31 the even one, lanes 32 .. 63 the odd one
#pragma unroll
    for (int d = 0; d < DB; d += 2) {
      float v[32];
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(o[d][r] * inv), __float_as_uint(o[d + 1][r] * inv), false, false);
        v[8 * (r >> 2) + (r & 3)] = __uint_as_float(s[0]), v[8 * (r >> 2) + 4 + (r & 3)] = __uint_as_float(s[1]);
      }
      const float m = digits_top(v);
      const bool rest = digits_uneven_columns(v, m, i0 + col < a.S) || digits_one_large(v, m);
      if (i0 + col < a.S) store_digits32(a.out_digits, (int64_t)(a.S + 31) / 32 * 32, a.H * DH / 32, i0 + col, (h * DH >> 5) + d + half, v, m, rest);
    }
    return;
  }
  if (i0 + col >= a.S) return;
#pragma unroll
  for (int d = 0; d < DB; d++)
#pragma unroll
    for (int r = 0; r < 16; r += 4) {
      const int at = h * DH + 32 * d + 2 * r + 4 * half;  // r / 4 * 8
      const float v[4] = {o[d][r] * inv, o[d][r + 1] * inv, o[d][r + 2] * inv, o[d][r + 3] * inv};
      if (a.out_planes) store_planes4(a.out_planes, i0 + col, a.H * DH / 32, at, v);
      else *(float4 *)(a.out + (int64_t)(i0 + col) * a.H * DH + at) = make_float4(v[0], v[1], v[2], v[3]);
    }
}

// S rows behind `start` cached ones.  Tiles of 32 rows x 32 keys over 1024 SIMDs: 2 us each in k_attn_mfma_bf, which shares a block's
// keys among eight wavefronts; 0.75 us here, but half of a block's tiles follow one another, and a launch comes in front.
// (1000 rows of 32 heads on 4: 41 -> 32 us; 500 behind 1000: 38 against 42; 512 of 12 heads: 10 against 22.)
bool attn_planes_pays(int S, int start, int H, int Hkv, int DH) {
  if (S < 64 || (DH != 64 && DH != 128) || H % Hkv) return false;
  const double nqb = (S + 31) / 32, longest = (start + S + 31) / 32, tiles = H * nqb * (longest - (nqb - 1) / 2.0), f = DH / 64.0;
  const double before = 3.0 + f * 2.0 * tiles / (4.0 * state().compute_units);
  const double each = 0.75 * tiles / (4.0 * state().compute_units), chain = 0.75 * longest;
  return 10.0 + f * (each > chain ? each : chain) < before;
}
int launch_attn_planes(float *out, void *out_terms, int terms, const float *q, const float *kc, const float *vc, int S, int start, int H, int Hkv, int DH, bool *done) {
  if ((DH != 64 && DH != 128) || S < 1 || Hkv < 1 || H % Hkv) return fail(CTHIP_E_UNSUPPORTED, "attention: %d rows, %d heads on %d of %d", S, H, Hkv, DH);
  AttnPlanesArgs a = {};
  a.out = out;
  a.out_planes = terms == kTermsPlanes ? (unsigned short *)out_terms : nullptr;
  a.out_digits = terms == kTermsDigits ? (unsigned char *)out_terms : nullptr;
  a.q = q;
  a.S = S, a.start = start, a.H = H, a.Hkv = Hkv;
  const int T = start + S, group = H / Hkv;
  a.nkb = (T + 31) / 32;
  a.units = (S + 31) / 32 * group;
  constexpr int NW = 4;
  const int wgs = Hkv * ((a.units + NW - 1) / NW);
  unsigned char *planes = nullptr;
  const size_t bytes = (size_t)Hkv * a.nkb * 128 * DH;
  if (alloc_scratch((void **)&planes, 2 * bytes + 2 * 128 * DH)) return 0;  // fully written by the first launch
  *done = true;
  int rc = 0;
  a.kp = planes;
  a.vp = planes + bytes;  // (a tile behind either may be read, and is not looked at)
  const dim3 sgrid(a.nkb, Hkv);
  hipStream_t st = state().stream;
  const size_t lds = DH == 64 ? 3 * 512 * 64 : 2 * 512 * 128;
  static bool big_lds = false;
  if (!big_lds) {
    CTHIP_CHECK(hipFuncSetAttribute((const void *)k_attn_planes<64, NW>, hipFuncAttributeMaxDynamicSharedMemorySize, 3 * 512 * 64));
    CTHIP_CHECK(hipFuncSetAttribute((const void *)k_attn_planes<128, NW>, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * 512 * 128));
    big_lds = true;
  }
  if (DH == 64) {
    hipLaunchKernelGGL(k_attn_split<64>, sgrid, dim3(256), 0, st, (unsigned short *)a.kp, (unsigned short *)a.vp, kc, vc, T, Hkv);
    hipLaunchKernelGGL((k_attn_planes<64, NW>), dim3(wgs), dim3(128 * NW), lds, st, a);
  } else {
    hipLaunchKernelGGL(k_attn_split<128>, sgrid, dim3(256), 0, st, (unsigned short *)a.kp, (unsigned short *)a.vp, kc, vc, T, Hkv);
    hipLaunchKernelGGL((k_attn_planes<128, NW>), dim3(wgs), dim3(128 * NW), lds, st, a);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) rc = fail((int)e, "attention: launch -> %s", hipGetErrorString(e));
  const int rf = cthip_free(planes);  // stream-ordered: handed out again only to later work on this stream
  return rc ? rc : rf;
}

}  // namespace cthip
