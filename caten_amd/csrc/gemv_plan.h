// How a single-row Linear launch is laid out: which kernel variant, how many workgroups of how many threads, how
// much LDS, which of the kernel's modes.  Pure host arithmetic (no HIP): launch_gemv (linear.hip) executes the plan,
// and the bounds harness under tests/ walks the same plan thread by thread on the CPU.
#pragma once
#include <stddef.h>

#include <vector>

#include "../../include/caten_hip.h"

namespace cthip {

// the (lanes per row, 16-byte chunks per lane) shapes instantiated per weight type (gemv_*.hip)
#define GEMV_SHAPES_Q8(V) V(CTHIP_Q8_0, 16, 1) V(CTHIP_Q8_0, 16, 2) V(CTHIP_Q8_0, 16, 3) V(CTHIP_Q8_0, 16, 4) V(CTHIP_Q8_0, 32, 3) \
  V(CTHIP_Q8_0, 32, 4) V(CTHIP_Q8_0, 64, 3) V(CTHIP_Q8_0, 64, 4) V(CTHIP_Q8_0, 64, 6) V(CTHIP_Q8_0, 64, 8)
#define GEMV_SHAPES_Q4(V) V(CTHIP_Q4_0, 16, 1) V(CTHIP_Q4_0, 16, 2) V(CTHIP_Q4_0, 32, 2) V(CTHIP_Q4_0, 64, 1) V(CTHIP_Q4_0, 64, 2) \
  V(CTHIP_Q4_0, 64, 3) V(CTHIP_Q4_0, 64, 4)
#define GEMV_SHAPES_F32(V) V(CTHIP_F32, 16, 4) V(CTHIP_F32, 64, 1) V(CTHIP_F32, 64, 2) V(CTHIP_F32, 64, 3) V(CTHIP_F32, 64, 4) \
  V(CTHIP_F32, 64, 6) V(CTHIP_F32, 64, 8) V(CTHIP_F32, 64, 12) V(CTHIP_F32, 64, 16) V(CTHIP_F32, 64, 24)
#define GEMV_SHAPES_F16(V) V(CTHIP_F16, 16, 2) V(CTHIP_F16, 64, 1) V(CTHIP_F16, 64, 2) V(CTHIP_F16, 64, 3) V(CTHIP_F16, 64, 4) \
  V(CTHIP_F16, 64, 6) V(CTHIP_F16, 64, 8) V(CTHIP_F16, 64, 12)

// looping launches keep about 12 sixteen-byte loads per lane in flight; the widest 4-bit variants (96+ input floats per
// lane in registers) keep two tiles, which leaves room for a second wavefront per SIMD
#define PD_OF_T(T, KC) (KC >= 12 ? 1 : (KC >= 6 || ((T) == CTHIP_Q4_0 && KC >= 3)) ? 2 : 4)

// tiles a wavefront of the looping kernel keeps in flight
inline int gemv_ring_depth(int type, int KC) { return PD_OF_T(type, KC); }
struct GemvShape {
  int type, G, KC;
};
inline const std::vector<GemvShape> &gemv_shapes() {
  static const std::vector<GemvShape> all = {
#define GEMV_SHAPE_ENTRY(T, G, KC) {T, G, KC},
      GEMV_SHAPES_Q8(GEMV_SHAPE_ENTRY) GEMV_SHAPES_Q4(GEMV_SHAPE_ENTRY) GEMV_SHAPES_F32(GEMV_SHAPE_ENTRY) GEMV_SHAPES_F16(GEMV_SHAPE_ENTRY)
#undef GEMV_SHAPE_ENTRY
  };
  return all;
}

inline int gemv_xpc(int type) {  // input elements one 16-byte chunk multiplies
  switch (type) {
    case CTHIP_Q8_0: return 16;
    case CTHIP_Q4_0: return 32;
    case CTHIP_F16: return 8;
    default: return 4;
  }
}

// index into gemv_shapes() of the variant that covers `cols` with the least idle lanes, or -1
inline int gemv_pick_shape(int type, int cols) {
  const int xpc = gemv_xpc(type);
  if (cols % xpc) return -1;
  const int nchunks = cols / xpc;
  int best = -1, best_waste = 1 << 30;
  const std::vector<GemvShape> &all = gemv_shapes();
  for (int i = 0; i < (int)all.size(); i++) {
    const GemvShape &v = all[i];
    if (v.type != type || v.G * v.KC < nchunks) continue;
    const int waste = v.G * v.KC - nchunks;
    if (waste < best_waste || (waste == best_waste && best >= 0 && v.G < all[best].G)) {
      best = i;
      best_waste = waste;
    }
  }
  return best;
}

// Rows wider than any register-resident variant (FFN down-projections of 7B-class models and up) are multiplied as
// column slices of equal width, one launch each: slice 0 carries the epilogue, every later one adds its products to
// what is there.  Returns the number of slices (0 = the width needs none, or cannot be cut on block boundaries into
// widths that variants cover) and their width (the last slice has what is left).
inline int gemv_slices(int type, long long cols, int *width) {
  const int xpc = gemv_xpc(type);
  const int unit = (type == CTHIP_Q8_0 || type == CTHIP_Q4_0) ? 32 : xpc;  // a slice starts on a block scale
  if (cols <= 0 || cols > 0x7fffffff || cols % unit) return 0;
  int maxc = 0;
  for (const GemvShape &sh : gemv_shapes())
    if (sh.type == type && sh.G * sh.KC * xpc > maxc) maxc = sh.G * sh.KC * xpc;
  if (!maxc || cols <= maxc) return 0;
  for (int n = (int)((cols + maxc - 1) / maxc); n <= 64; n++) {
    const int wdt = (int)(((cols + n - 1) / n + unit - 1) / unit * unit);
    const long long last = cols - (long long)wdt * (n - 1);
    if (wdt <= maxc && last > 0 && gemv_pick_shape(type, wdt) >= 0 && gemv_pick_shape(type, (int)last) >= 0) {
      *width = wdt;
      return n;
    }
  }
  return 0;
}

struct GemvPlanIn {
  int type, rows, cols, m;
  int pro;            // CTHIP_PRO_*
  bool fold;          // a LayerNorm folded through the product (fold_s given)
  bool bias, bias0, residual, argmax;
  int compute_units;
  int occupancy;      // resident 256-thread workgroups of the looping kernel per compute unit (from the runtime)
};

enum GemvKernelKind { GEMV_K_SMALL, GEMV_K_LOOP, GEMV_K_LOOP_EPI, GEMV_K_LOOP_DIRECT };

struct GemvPlan {
  int shape = -1;      // index into gemv_shapes(); -1 = no register-resident variant (generic fallback)
  unsigned grid_x = 0, grid_y = 0, block = 0;
  size_t lds = 0;
  bool stage = false;  // the workgroup stages the input vector in LDS once
  bool unfold = false; // the launch drops the fold terms and normalises the staged vector itself
  GemvKernelKind kernel = GEMV_K_SMALL;
  int nwaves = 0;
  const char *error = nullptr;
};

inline GemvPlan gemv_plan(const GemvPlanIn &in) {
  GemvPlan p;
  p.shape = gemv_pick_shape(in.type, in.cols);
  p.grid_y = (unsigned)in.m;
  if (p.shape < 0) return p;
  const GemvShape &v = gemv_shapes()[p.shape];
  const int rpw = 64 / v.G;
  const int nrq = (in.rows + rpw - 1) / rpw;
  bool fold = in.fold, bias = in.bias, residual = in.residual;
  const bool folded = (in.pro == CTHIP_PRO_RMSNORM) || (in.pro == CTHIP_PRO_LAYERNORM && fold);
  const bool quantised = in.type == CTHIP_Q8_0 || in.type == CTHIP_Q4_0;
  // The input vector goes through LDS once per workgroup when it must be normalised or gated first, or when it is
  // large next to a weight tile (a 4-bit tile multiplies 8 input bytes per weight byte): then four wavefronts share
  // one copy and every wavefront takes several tiles.  Quantised launches with a folded norm stage at every size.
  p.stage = (in.pro != CTHIP_PRO_NONE && !folded) || (in.type == CTHIP_Q4_0 && in.cols >= 1024) || (folded && (in.cols >= 2048 || quantised));
  p.lds = p.stage ? sizeof(float) * (size_t)in.cols : 0;
  if (p.lds > 64 * 1024) {
    p.error = "input features exceed the LDS staging buffer";
    return p;
  }
  bool small, direct = false;
  if (!p.stage && nrq <= 2048) {
    // small matrices are pure latency: one tile per wavefront, one wavefront per workgroup, spread over as many
    // compute units as there are tiles
    small = true;
    p.block = 64;
    p.grid_x = (unsigned)nrq;
  } else if (p.stage && nrq <= in.compute_units * 3) {
    // one tile per wavefront, as many wavefronts per workgroup (at most three) as leave about one workgroup per
    // compute unit: fewer workgroups repeat the staging less, but idle units stream nothing
    small = true;
    int wpb = (nrq + in.compute_units - 1) / in.compute_units;
    wpb = wpb < 1 ? 1 : wpb > 3 ? 3 : wpb;
    p.block = 64u * (unsigned)wpb;
    p.grid_x = (unsigned)((nrq + wpb - 1) / wpb);
  } else {
    // larger matrices: at least one wavefront per SIMD, more (up to what the register budget keeps resident) once
    // every wavefront has four tiles
    small = false;
    const int occ = in.occupancy > 0 ? in.occupancy : 1;
    p.block = 256;
    const int base = in.compute_units * 4;
    // unstaged: a wavefront per tile up to three resident wavefronts per SIMD
    int wanted = p.stage ? (nrq + 3) / 4 : nrq;
    if (wanted < base) wanted = base;
    const int cap = base * (p.stage || occ < 3 ? occ : 3);
    if (wanted > cap) wanted = cap;
    // staged launches pay the input staging once per workgroup: whole workgroups per compute unit, two when there
    // is work for more than one
    if (p.stage && wanted > base && occ >= 2) wanted = 2 * base;
    const int iters = (nrq + wanted - 1) / wanted;
    // every resident wavefront slot is used even if some wavefronts then loop once more than others
    const int waves = wanted < nrq ? wanted : nrq;
    p.grid_x = (unsigned)((waves + 3) / 4);
    // the ring requests all its slots unconditionally: a wavefront with a single tile takes the kernel without one
    if (iters == 1) small = true;
    // a looping launch normalises the staged vector itself rather than carrying the fold terms: two more operands
    // per row in the weight ring hold the stream up more than the second barrier of the staging costs
    if (!small && p.stage && in.pro == CTHIP_PRO_LAYERNORM && fold && !in.bias0 && !residual && in.cols <= 4096) {
      p.unfold = true;
      fold = false;
      bias = false;
    }
    direct = !small && p.stage && in.pro == CTHIP_PRO_LAYERNORM && !fold && !bias && !residual && in.cols <= 4096;
  }
  p.nwaves = (int)(p.grid_x * (p.block / 64));
  const bool epi = bias || residual || fold;
  p.kernel = small ? GEMV_K_SMALL : epi ? GEMV_K_LOOP_EPI : direct ? GEMV_K_LOOP_DIRECT : GEMV_K_LOOP;
  // what the kernels assume of their launch
  if (p.kernel != GEMV_K_SMALL && p.block != 256) p.error = "a looping launch must have 256 threads per workgroup";
  if (p.block > 512) p.error = "more than eight wavefronts per workgroup";
  return p;
}

// The wide-row kernel (gemv_wide.hip): the input vector lives in LDS instead of in registers, so a row may be as
// wide as LDS holds and the registers a lane needs do not grow with the width.  A round = 64 chunks (one per lane);
// a tile = nc rounds of a pair of neighbouring rows, requested together; a row = tpr tiles.  lds counts floats: the staged vector, one
// sum per chunk for 4-bit weights, 16 for the reduction of a norm's statistics.
struct GemvWidePlan {
  bool ok = false;
  int nc = 0, tpr = 0, rw = 1;  // rw: rows a wavefront streams together (1 or 2)
  unsigned grid = 0, block = 512;
  size_t lds_floats = 0;
};
constexpr size_t kGemvWideMaxLdsBytes = 150 * 1024;
inline GemvWidePlan gemv_wide_plan(int type, long long rows, long long cols, int compute_units) {
  GemvWidePlan p;
  if (type != CTHIP_Q8_0 && type != CTHIP_Q4_0 && type != CTHIP_F16 && type != CTHIP_F32) return p;
  const int xpc = gemv_xpc(type);
  const bool quant = type == CTHIP_Q8_0 || type == CTHIP_Q4_0;
  if (rows <= 0 || rows > 0x7fffffff || cols < 64 || cols % (quant ? 32 : xpc) || cols > 0x7fffffff) return p;
  const int nchunks = (int)(cols / xpc);
  p.lds_floats = (size_t)cols + (type == CTHIP_Q4_0 ? (size_t)nchunks : 0) + 16;
  if (p.lds_floats * 4 > kGemvWideMaxLdsBytes) return p;
  const int rounds = (nchunks + 63) / 64;
  // (six 16-byte requests of weights per lane and tile: 3, 2 or 1 rounds of two rows)
  // (4-bit chunks are 32 inputs wide: with more than one round's inputs between LDS and the arithmetic the kernel
  // does not fit the 128 registers that let four wavefronts share a SIMD)
  p.nc = type == CTHIP_Q4_0 ? 1 : rounds % 3 == 0 ? 3 : rounds % 2 == 0 ? 2 : 1;
  p.tpr = rounds / p.nc;
  // two workgroups per compute unit where LDS holds two copies of the vector; never more wavefronts than rows
  const long long per_cu = p.lds_floats * 4 * 2 <= kGemvWideMaxLdsBytes ? 2 : 1;
  long long grid = (long long)compute_units * per_cu;
  // rows go in pairs where the pairs still fill every wavefront slot of the launch
  p.rw = (rows + 1) / 2 >= grid * 8 ? 2 : 1;
  const long long need = ((rows + p.rw - 1) / p.rw + 7) / 8;
  if (grid > need) grid = need;
  p.grid = (unsigned)(grid < 1 ? 1 : grid);
  p.ok = true;
  return p;
}

// The integer kernel (gemv_int.hip): ks wavefronts share a group of 16 rows, each takes upw units (128 bytes) of every row; a
// workgroup has rgp such sets and goes over its groups of 16 rgp rows grid apart.  lds: bytes (256 of zeros, digits and scales of the vector,
// 32 words of reductions, the partial sums of every wavefront and group).
// Eight wavefronts and two workgroups to a compute unit where there are groups enough for that and a row is not too long for them, else
// sixteen (us, 16 / 8: 12288 x 4096 9.9 / 8.6, 22016 x 4096 14.6 / 13.3, 4096 x 4096 6.1 / 6.2, 4096 x 11008 10.0 / 10.9).
struct GemvIntPlan {
  bool ok = false;
  int upw = 0, ks = 0, rgp = 0, iters = 0;
  unsigned grid = 0;
  size_t lds = 0;
};
constexpr size_t kGemvIntMaxLdsBytes = 156 * 1024;
inline GemvIntPlan gemv_int_plan(int type, long long rows, long long cols, int compute_units) {
  GemvIntPlan p;
  // (pairs of scales are fetched as one dword)
  if (type != CTHIP_Q4_0 || rows <= 0 || rows > 0x7fffffff - 1024 || cols < 64 || cols % 64 || cols > (1 << 20)) return p;
  const long long groups = (rows + 15) / 16;
  const int units = (int)((cols / 2 + 127) / 128), cap = units <= 16 && groups >= 2ll * compute_units ? 8 : 16;
  p.upw = (units + cap - 1) / cap;
  p.ks = (units + p.upw - 1) / p.upw;
  if (p.ks < 4) return p;  // rows of less than 512 bytes
  p.rgp = cap / p.ks;
  while (p.rgp > 1 && groups / p.rgp < compute_units) p.rgp--;
  const long long nsg = (groups + p.rgp - 1) / p.rgp, slots = (long long)compute_units * (16 / (p.ks * p.rgp));
  p.grid = (unsigned)(nsg < slots ? nsg : slots);
  const long long iters = (nsg + p.grid - 1) / p.grid;
  if (iters * 16 > 64 * p.ks) return p;  // a thread per row of a workgroup
  p.iters = (int)iters;
  const size_t cpad = (size_t)p.ks * p.upw * 8;
  p.lds = 256 + cpad * 132 + 32 * 4 + (size_t)iters * p.ks * p.rgp * 64;
  p.ok = p.lds <= kGemvIntMaxLdsBytes;
  return p;
}
// Where that kernel is the faster one.  It goes over groups of 16 rows in rounds of one (long rows) or two to a compute unit; the vector kernels spread any number of
// rows over their wavefronts, and multiply rows that fill their lanes at the rate that the weights arrive.  us, vector / integer, matrices out of memory:
//   most sizes                          12288 x 4096 9.9 / 8.5, 22016 x 4096 13.9 / 12.6, 4096 x 11008 12.5 / 10.5, 50257 x 1280 13.8 / 9.3, 32000 x 8192 39.4 / 35.0
//   rows under 5/8 of a round           2048 x 2048 4.3 / 4.3, 2048 x 4096 5.1 / 5.4, 1536 x 6144 6.4 / 6.4 (2304 x 4096 5.7 / 5.5: what lies between is not looked at)
//   a quarter of a second round         4608 x 4096 6.5 / 7.3, 4352 x 2560 5.8 / 6.1, 4864 x 5120 7.6 / 8.0, 4608 x 8192 11.9 / 12.4 (no less at 4608 x 6656 11.0 / 9.6)
//   3072 .. 4096 columns, while the vector kernels' rows fit one more of their rounds
//                                       7168 x 3584 6.9 / 7.2, 9216 x 4096 8.2 / 8.6; past that 7936 x 3584 7.4 / 7.4, 9728 x 4096 9.2 / 8.8
//   4608 .. 6144 columns (10 .. 12 wavefronts, the others' places empty), from 3584 on rows that are no whole units: a last round that is less than half full
//                                       13312 x 5760 13.2 / 14.0, 9216 x 6144 11.3 / 12.4, 50257 x 5632 33.2 / 35.2, 9216 x 3968 8.1 / 9.1;
//                                       full ones 12288 x 6144 13.1 / 12.3, 14336 x 5120 13.6 / 13.0
//   9728 .. 10240 columns               14 wavefronts of 42 units for 40 against five whole steps of gemv_wide.hip: 5120 x 10240 15.3 / 16.6, 9216 x 10240 21.5 / 22.4
inline bool gemv_int_pays(long long rows, long long cols, int compute_units) {
  const long long round = 16ll * compute_units, last = rows % round;
  if (8 * rows < 5 * round || cols > 16384) return false;
  if (rows <= round) return true;
  if (4 * rows <= 5 * round && ((cols > 2304 && cols <= 6144) || cols == 8192)) return false;
  if (cols > 3072 && cols <= 4096 && 16 * rows <= (cols > 3584 ? 37 : 29) * round) return false;
  if (cols > 3584 && cols <= 6144 && (cols > 4608 || cols % 256) && rows > 2 * round && last > 0 && 2 * last < round) return false;
  return !(cols > 9728 && cols <= 10240);
}

// How the split-K reduction + norm pass (rowops.hip) lays a row out: `wide` = four wavefronts per row instead of
// one; `vpl` = the float4-per-lane count of the kernel instantiation chosen (one of 1,2,3,4,6,8 narrow / 1,2,4,8
// wide); `nz` = the share bucket.  ok is false when no instantiation covers the row.
struct ReduceNormPlan {
  bool ok, wide;
  int vpl, nz;
};
inline ReduceNormPlan reduce_norm_plan(int n, int nparts, long long rows) {
  ReduceNormPlan p = {false, false, 0, 0};
  if (n < 4 || n % 4 || n > 8192 || nparts < 1 || nparts > 16) return p;
  p.nz = nparts <= 2 ? 2 : nparts <= 4 ? 4 : nparts <= 8 ? 8 : 16;
  const int v1 = (n / 4 + 63) / 64, v4 = (n / 4 + 255) / 256;
  // the shares of a row are all requested at once: VPL x NZ float4 per lane have to stay in registers
  const bool narrow_fits = v1 * p.nz <= 32 && v1 <= 8, wide_fits = v4 * p.nz <= 32 && v4 <= 8;
  if (!narrow_fits && !wide_fits) return p;
  // four wavefronts per row where one cannot hold the row's shares, and for a prompt's few rows of some width: the
  // pass is a single memory round trip, and four times the threads ask for it four times as wide
  p.wide = !narrow_fits || (wide_fits && rows <= 2048 && n >= 512);
  if (p.wide) p.vpl = v4 <= 1 ? 1 : v4 <= 2 ? 2 : v4 <= 4 ? 4 : 8;
  else p.vpl = v1 <= 4 ? v1 : v1 <= 6 ? 6 : 8;
  p.ok = true;
  return p;
}

}  // namespace cthip
