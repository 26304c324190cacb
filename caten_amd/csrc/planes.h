// GEMM operands in memory as bf16 terms (gemm_planes.hip): layout and the epilogue shared by its instantiations.
#pragma once
#include "common.h"

namespace cthip {

enum { PL_PLANES = 0, PL_INT = 1 };

struct PlaneGemmArgs {
  float *C;
  const unsigned char *A, *B;
  const unsigned short *bd;  // scales of quants
  int apitch, bpitch;        // bytes between rows
  int dpitch;                // scales between rows
  int M, N, nkb;             // nkb: blocks of 32 k
  const float *bias, *residual;
  int act;
  int tm, tn, band, chunk;   // tile -> workgroup mapping
  int pairs;                 // columns (2j, 2j + 1) are (gate, up): C (M, N / 2) gets silu(gate) * up
  int routed;
  GemmRoute route;
  unsigned short *planes;    // non-null: the result goes out as planes of two terms instead of C
  int pkb;                   // blocks of 32 columns per row of `planes` (k_gemm_digits: or `digits`)
};

#if defined(__HIPCC__)
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf_pl __attribute__((ext_vector_type(2)));
typedef float v2f_pl __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned pack_bf16_pl(float x0, float x1) {  // one v_cvt_pk_bf16_f32, round to nearest even
  const v2f_pl v = {x0, x1};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, v2bf_pl));
}
template <int NP>
__device__ __forceinline__ void split4_planes(float r0, float r1, float r2, float r3, uint2 *pl) {
#pragma unroll
  for (int p = 0; p < NP; p++) {
    pl[p].x = pack_bf16_pl(r0, r1);
    pl[p].y = pack_bf16_pl(r2, r3);
    if (p + 1 < NP) {  // exact: the difference of a float and its own leading bits
      r0 -= __uint_as_float(pl[p].x << 16);
      r1 -= __uint_as_float(pl[p].x & 0xffff0000u);
      r2 -= __uint_as_float(pl[p].y << 16);
      r3 -= __uint_as_float(pl[p].y & 0xffff0000u);
    }
  }
}
template <int NP>
__device__ __forceinline__ void split8_planes(const float *v, uint4 *pl) {
  uint2 a[NP], b[NP];
  split4_planes<NP>(v[0], v[1], v[2], v[3], a);
  split4_planes<NP>(v[4], v[5], v[6], v[7], b);
#pragma unroll
  for (int p = 0; p < NP; p++) pl[p] = make_uint4(a[p].x, a[p].y, b[p].x, b[p].y);
}
// four consecutive columns col .. col + 3 (col a multiple of 4) of a row as two-term planes
__device__ __forceinline__ void store_planes4(unsigned short *planes, int64_t row, int pkb, int col, const float *v) {
  uint2 pl[2];
  split4_planes<2>(v[0], v[1], v[2], v[3], pl);
  unsigned short *p = planes + (row * pkb + (col >> 5)) * 64 + (col & 31);
  *(uint2 *)p = pl[0];
  *(uint2 *)(p + 32) = pl[1];
}

// The same for a handful of rows (linear_few.hip), as operands of v_mfma_f32_16x16x32_bf16 lie in a wavefront: [block of 32 k][term][16 rows][lane][8 k],
// lane = 16 (k / 8 of the block) + row % 16, row_blocks = blocks of 16 rows
__device__ __forceinline__ void store_operands4(unsigned short *planes, int row, int row_blocks, int col, const float *v) {
  uint2 pl[2];
  split4_planes<2>(v[0], v[1], v[2], v[3], pl);
  const int lane = 16 * ((col >> 3) & 3) + (row & 15);
  unsigned short *p = planes + (((int64_t)(col >> 5) * 2 * row_blocks + (row >> 4)) * 64 + lane) * 8 + (col & 7);
  *(uint2 *)p = pl[0];
  *(uint2 *)(p + row_blocks * 512) = pl[1];
}

typedef float v16f __attribute__((ext_vector_type(16)));

// 16 bytes per lane from sbase + voff straight into LDS at lds + 16 * lane.  Written out because the compiler, which
// cannot tell the buffers of a ring apart, waits for ALL such loads before every LDS read; the kernel below counts
// them itself (the reads it protects lie behind the same asm's "memory" clobber).
__device__ __forceinline__ void dma16(const void *sbase, unsigned voff, unsigned lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds) : "memory");
}
// 2 bytes per lane, zero-extended to the dword at lds + 4 * lane
__device__ __forceinline__ void dma2(const void *sbase, unsigned voff, unsigned lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_ushort %0, %1" ::"v"(voff), "s"(sbase), "s"(lds) : "memory");
}
// 4 bytes per lane
__device__ __forceinline__ void dma4(const void *sbase, unsigned voff, unsigned lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(sbase), "s"(lds) : "memory");
}
// a value that is the same in every lane, in scalar registers
__device__ __forceinline__ const unsigned char *uniform(const unsigned char *p) {
  const uint64_t v = (uint64_t)p;
  return (const unsigned char *)(((uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) | (unsigned)__builtin_amdgcn_readfirstlane((int)v));
}
// all but the youngest N of this wavefront's loads have landed
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// this wavefront's LDS reads are done
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
// all but the youngest N of this wavefront's loads have landed, its LDS reads are done, and so are everybody else's
template <int N>
__device__ __forceinline__ void wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

__device__ __forceinline__ unsigned pack_int_bf16(float x0, float x1) {
  return __builtin_amdgcn_perm(__float_as_uint(x1), __float_as_uint(x0), 0x07060302u);  // high halves of both
}
// 8 int8 -> 8 bf16, exact
__device__ __forceinline__ v8bf bf_of_q8(unsigned a, unsigned b) {
  return __builtin_bit_cast(v8bf, make_uint4(pack_int_bf16(sbyte0_f32(a), sbyte1_f32(a)), pack_int_bf16(sbyte2_f32(a), sbyte3_f32(a)),
                                             pack_int_bf16(sbyte0_f32(b), sbyte1_f32(b)), pack_int_bf16(sbyte2_f32(b), sbyte3_f32(b))));
}
// What the end of a kernel needs of its arguments, loaded where this is made
struct PlaneStore {
  float *C;
  const float *bias, *residual;
  unsigned short *planes;
  int M, N, act, pairs, routed, pkb;
  const GemmRoute &route;
  __device__ __forceinline__ PlaneStore(const PlaneGemmArgs &a)
      : C(early(a.C)), bias(early(a.bias)), residual(early(a.residual)), planes(early(a.planes)), M(early(a.M)), N(early(a.N)), act(early(a.act)), pairs(early(a.pairs)),
        routed(early(a.routed)), pkb(early(a.pkb)), route(a.route) {}
  // left to the compiler, right in front of their use: kernels whose first loads are what a launch waits for
  struct Late {};
  __device__ __forceinline__ PlaneStore(const PlaneGemmArgs &a, Late)
      : C(a.C), bias(a.bias), residual(a.residual), planes(a.planes), M(a.M), N(a.N), act(a.act), pairs(a.pairs), routed(a.routed), pkb(a.pkb), route(a.route) {}
};
// columns col .. col + 3, all of them inside, of one row of a finished tile: bias bb (where a.bias), activation, residual rr (where a.residual), and where they go
__device__ __forceinline__ void plane_gemm_finish(const PlaneStore &a, int N, int row, int col, float4 v4, float4 bb, float4 rr) {
  float v[4] = {v4.x, v4.y, v4.z, v4.w};
  if (a.bias) v[0] += bb.x, v[1] += bb.y, v[2] += bb.z, v[3] += bb.w;
  if (a.pairs) {
    v[0] = apply_act(CTHIP_ACT_SILU, v[0]) * v[1], v[1] = apply_act(CTHIP_ACT_SILU, v[2]) * v[3];
    if (a.planes) {  // two columns of the result: neighbours in both terms
      const unsigned h = pack_bf16_pl(v[0], v[1]);
      const unsigned l = pack_bf16_pl(v[0] - __uint_as_float(h << 16), v[1] - __uint_as_float(h & 0xffff0000u));
      unsigned short *p = a.planes + ((int64_t)row * a.pkb + (col >> 6)) * 64 + ((col >> 1) & 31);
      *(unsigned *)p = h;
      *(unsigned *)(p + 32) = l;
    } else {
      *(float2 *)(a.C + (int64_t)row * (N >> 1) + (col >> 1)) = make_float2(v[0], v[1]);
    }
    return;
  }
  if (a.act != CTHIP_ACT_NONE)
#pragma unroll
    for (int t = 0; t < 4; t++) v[t] = apply_act(a.act, v[t]);
  if (a.residual) v[0] += rr.x, v[1] += rr.y, v[2] += rr.z, v[3] += rr.w;
  if (a.planes) {
    store_planes4(a.planes, row, a.pkb, col, v);
    return;
  }
  float *dst = a.C;
  int ldd = N, cbase = 0;
  if (a.routed) {
    // (selected, not indexed: an index would put the arguments into scratch memory)
    const bool p2 = col >= a.route.c0[2], p1 = col >= a.route.c0[1];
    dst = p2 ? a.route.dst[2] : p1 ? a.route.dst[1] : a.route.dst[0];
    ldd = p2 ? a.route.ld[2] : p1 ? a.route.ld[1] : a.route.ld[0];
    cbase = p2 ? a.route.c0[2] : p1 ? a.route.c0[1] : 0;
  }
  *(f4_any *)(dst + (int64_t)row * ldd + (col - cbase)) = f4_any{v[0], v[1], v[2], v[3]};
}
// the same where a row ends within them
__device__ __forceinline__ void plane_gemm_finish_any(const PlaneStore &a, int row, int col, float4 v4) {
  const float v[4] = {v4.x, v4.y, v4.z, v4.w};
  for (int t = 0; t < 4 && col + t < a.N; t++) {
    float x = apply_act(a.act, v[t] + (a.bias ? a.bias[col + t] : 0.0f));
    if (a.residual) x += a.residual[(int64_t)row * a.N + col + t];
    a.C[(int64_t)row * a.N + col + t] = x;
  }
}
// columns col .. col + 3 of one row: the same where bias and residual are asked for as a thread goes (linear_rows.hip)
__device__ __forceinline__ void plane_gemm_store(const PlaneGemmArgs &args, int row, int col, float4 v4) {
  const PlaneStore a(args, PlaneStore::Late());
  if (row >= a.M || col >= a.N) return;
  if (a.N & 3) {
    plane_gemm_finish_any(a, row, col, v4);
    return;
  }
  float4 bb = make_float4(0.0f, 0.0f, 0.0f, 0.0f), rr = bb;
  if (a.bias) bb = *(const float4 *)(a.bias + col);
  if (a.residual && !a.pairs) rr = *(const float4 *)(a.residual + (int64_t)row * a.N + col);
  plane_gemm_finish(a, a.N, row, col, v4, bb, rr);
}
// A wavefront's 32 rows of 32 NB columns, which lie in LDS (pitch 32 NB + 4), to where they go.  A lane stores the same four columns of every 64 / C4-th row, so that their bias is
// read once, by plane_gemm_bias, long before; the residual of plain rows is asked for several rows at a time.  Short code: with every row's
// cases copied out a kernel was 14 - 50 KB, now 8 - 33, and a launch of a few steps waited for its instructions (4500 x 4500 x 600 at one term 59.7 -> 53.6 us with
// the shorter step, Q8_0 3072 x 1024 over 900 rows 31.1 -> 27.7).
template <int NB>
__device__ __forceinline__ float4 plane_gemm_bias(const PlaneStore &a, int col0, int lane) {
  if (!a.bias) return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const f4_any t = *(const f4_any *)(a.bias + min(col0 + 4 * (lane % (8 * NB)), a.N - 4));
  return make_float4(t[0], t[1], t[2], t[3]);
}
template <int NB, int AHEAD = 4>
__device__ __forceinline__ void plane_gemm_store_rows(const PlaneStore &a, const float *Cs, int row0, int col0, int lane, float4 bias) {
  constexpr int LDC = 32 * NB + 4, C4 = 8 * NB, RPI = 64 / C4, NU = 32 / RPI;  // rows per instruction
  const int lr = lane / C4, c4 = lane % C4, at = col0 + 4 * c4;
  const bool mine = lr < RPI && at + 4 <= a.N;  // (16-byte accesses at any alignment: rows of N floats)
  const float *p = Cs + lr * LDC + 4 * c4;
  if (a.act == CTHIP_ACT_NONE && !a.pairs && !a.planes && !a.routed) {
#pragma unroll
    for (int u0 = 0; u0 < NU; u0 += AHEAD) {
      f4_any rr[AHEAD];
      if (a.residual)
#pragma unroll
        for (int u = 0; u < AHEAD; u++) rr[u] = *(const f4_any *)(a.residual + (int64_t)min(row0 + lr + (u0 + u) * RPI, a.M - 1) * a.N + min(at, a.N - 4));
#pragma unroll
      for (int u = 0; u < AHEAD; u++) {
        const int row = row0 + lr + (u0 + u) * RPI;
        float4 v = *(const float4 *)(p + (u0 + u) * RPI * LDC);
        if (a.bias) v.x += bias.x, v.y += bias.y, v.z += bias.z, v.w += bias.w;
        if (a.residual) v.x += rr[u][0], v.y += rr[u][1], v.z += rr[u][2], v.w += rr[u][3];
        if (mine && row < a.M) *(f4_any *)(a.C + (int64_t)row * a.N + at) = f4_any{v.x, v.y, v.z, v.w};
      }
    }
  } else {
#pragma unroll 1
    for (int u = 0; u < NU; u++) {
      const int row = row0 + lr + u * RPI;
      const float4 v = *(const float4 *)(p + u * RPI * LDC);
      if (!mine || row >= a.M) continue;
      float4 rr = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (a.residual && !a.pairs) {
        const f4_any t = *(const f4_any *)(a.residual + (int64_t)row * a.N + at);
        rr = make_float4(t[0], t[1], t[2], t[3]);
      }
      plane_gemm_finish(a, a.N, row, at, v, bias, rr);
    }
  }
  if (a.N % 4 && lr < RPI && at < a.N && at + 4 > a.N)
#pragma unroll 1
    for (int r = lr; r < min(32, a.M - row0); r += RPI) plane_gemm_finish_any(a, row0 + r, at, *(const float4 *)(Cs + r * LDC + 4 * c4));
}
#endif

}  // namespace cthip
