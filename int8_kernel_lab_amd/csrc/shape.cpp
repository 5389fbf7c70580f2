// Shape validation, tile planners and eligibility predicates (host only).
#include <limits.h>
#include <stdint.h>

#include <algorithm>
#include <string>

#include "i8conv_internal.hpp"

namespace i8conv {

// conv_shape.cuh:22-35.  out_h/out_w use the same C++ expression (integer
// division truncating toward zero) so that every shape the reference
// accepts derives to the same geometry.
int derive(const i8conv_shape &s, i8conv_geometry *g) {
  if (s.n < 1 || s.h < 1 || s.w < 1 || s.c < 1 || s.k < 1 || s.r < 1 ||
      s.s < 1 || s.pad_h < 0 || s.pad_w < 0 || s.stride_h < 1 ||
      s.stride_w < 1 || s.dilation_h < 1 || s.dilation_w < 1) {
    set_error("shape fields out of range (sizes, strides, dilations >= 1, pads >= 0)");
    return I8CONV_BAD_SHAPE;
  }
  if (s.c % 16 != 0) {
    set_error("input channels must be divisible by 16");
    return I8CONV_BAD_SHAPE;
  }
  const int64_t num_h = int64_t(s.h) + 2 * int64_t(s.pad_h) -
                        int64_t(s.dilation_h) * (s.r - 1) - 1;
  const int64_t num_w = int64_t(s.w) + 2 * int64_t(s.pad_w) -
                        int64_t(s.dilation_w) * (s.s - 1) - 1;
  const int64_t out_h = num_h / s.stride_h + 1;
  const int64_t out_w = num_w / s.stride_w + 1;
  if (out_h <= 0 || out_w <= 0) {
    set_error("output must be nonempty");
    return I8CONV_BAD_SHAPE;
  }
  const int64_t gemm_m = int64_t(s.n) * out_h * out_w;
  const int64_t gemm_k = int64_t(s.r) * s.s * s.c;
  const int64_t in_el = int64_t(s.n) * s.h * s.w * s.c;
  const int64_t f_el = int64_t(s.k) * gemm_k;
  const int64_t out_el = gemm_m * s.k;
  if (in_el > INT32_MAX || f_el > INT32_MAX || gemm_m > INT32_MAX ||
      gemm_k > INT32_MAX || out_el > (int64_t(1) << 40) || out_h > INT32_MAX ||
      out_w > INT32_MAX) {
    set_error("tensor too large (input/filter bytes and M must be < 2^31)");
    return I8CONV_BAD_SHAPE;
  }
  if (g) {
    g->out_h = int32_t(out_h);
    g->out_w = int32_t(out_w);
    g->gemm_m = gemm_m;
    g->gemm_n = s.k;
    g->gemm_k = int32_t(gemm_k);
    g->input_elements = in_el;
    g->filter_elements = f_el;
    g->output_elements = out_el;
  }
  return I8CONV_OK;
}

namespace {

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

}  // namespace

// Workgroup tiles instantiated in kernel_gemm.hip (BM pixels x BN channels).
bool gemm_tile_supported(int bm, int bn) {
  switch (bm * 1000 + bn) {
    case 64032: case 64064: case 64128: case 128032: case 128064:
    case 128128: case 256064: case 256128:
      return true;
    default:
      return false;
  }
}

// The LDS-DMA pipelined kernel (kernel_gemm_dma.hip) needs every 128-byte
// k-stage inside one filter tap: c % 128 == 0.
static bool dma_eligible(const i8conv_shape &s) { return s.c % kStageBytes == 0; }

// Generic tile choice.  Pipelined kernel: 128 output channels per tile
// (64 when N <= 64), and 256 pixels when that still gives the grid about
// three quarters of the 256 compute units, else 128.  Short reductions (at
// most 4 stages: 1x1 layers) take 128 pixels regardless: they are bound by
// HBM, and the smaller LDS ring lets three workgroups share a compute unit
// (measured on a 1x1 C = 256 -> 64 layer: 20.0 us vs 25.1 us with 256).  Register-staged
// kernel: the smallest supported width covering N (32/64/128 columns, 128
// for wider layers); the pixel tile shrinks from 256 until the grid has
// enough workgroups to cover the 256 compute units.
// Pipelined kernel, tile step: when ceil(M / bm) * tiles_n workgroups (more
// than one per compute unit) leave a last round that covers only part of
// the 256 compute units, the layer waits on a few workgroups that run alone
// (a 1x1 C = 256 -> 64 layer: 1568 tiles of 128 pixels take 19.2 us, 1536
// take 17.8 us).  A tile that stores fewer pixel rows (a multiple of 16; its
// last rows are zero-filled by out-of-range copies) evens the rounds out:
// the step minimises ceil(tiles / 256) * (bn + step), ties to the larger
// step (config 4a: 1792 tiles storing 112 rows, 19.2 -> 18.8 us).  The
// zero-filled rows still pass through the copy path, so a grid of one round
// keeps whole tiles (config 3 with 208-row steps: 15.15 vs 15.07 us).
int gemm_dma_step(int64_t gemm_m, int64_t tiles_n, int bm, int bn) {
  int best = bm;
  const int64_t tiles = ceil_div(gemm_m, bm) * tiles_n;
  if (tiles <= 256) return best;
  int64_t best_cost = ceil_div(tiles, 256) * (bn + bm);
  for (int step = bm - 16; step > bm / 2; step -= 16) {
    const int64_t cost = ceil_div(ceil_div(gemm_m, step) * tiles_n, 256) * (bn + step);
    if (cost < best_cost) {
      best = step;
      best_cost = cost;
    }
  }
  return best;
}

// Pointwise streaming form: instances for C in {64, 128, 256, 512} and N in
// {32, 64, 128, 256}.  A wave holds a slice of the filter as MFMA A
// operands, at most 16384 bytes (64 VGPRs per lane): slices of
// min(N, 16384 / C) output channels, 2 to 8 of them where N * C > 16384.
bool pointwise_supported(int c, int n) {
  const bool cs = c == 64 || c == 128 || c == 256 || c == 512;
  const bool ns = n == 32 || n == 64 || n == 128 || n == 256;
  return cs && ns;
}

int pointwise_slices(int c, int n) {
  const int per = std::min(n, 16384 / c);
  return n / per;
}

bool pointwise_requant_supported(int c, int n) {
  if (!pointwise_supported(c, n)) return false;
  const int per = n / pointwise_slices(c, n);
  return per == 64 || per == 128;
}

// Two-wave workgroups of one fragment stream each, or one workgroup of SL
// waves per stream; at most kPwMaxWaves waves (fewer streams than
// fragments otherwise).
int pointwise_waves(int64_t gemm_m, int slices) {
  const int group = pw_group_waves(slices), streams_per_group = group / slices;
  const int64_t streams = std::min<int64_t>(ceil_div(gemm_m, 16), kPwMaxWaves / slices);
  return int(ceil_div(streams, streams_per_group) * group);
}

static bool pointwise_eligible(const i8conv_shape &s, const i8conv_geometry &g) {
  // 32-bit buffer offsets: input and output below 2 GiB, so that the
  // out-of-range offset 2^31 lies past both
  return s.r == 1 && s.s == 1 && s.stride_h == 1 && s.stride_w == 1 && s.pad_h == 0 &&
         s.pad_w == 0 && pointwise_supported(s.c, g.gemm_n) &&
         g.gemm_m * s.c < (int64_t(1) << 31) && g.gemm_m * g.gemm_n * 4 < (int64_t(1) << 31);
}

static GemmPlan plan_staged(const i8conv_shape &s, const i8conv_geometry &g) {
  GemmPlan p;
  p.stages = int(ceil_div(g.gemm_k, kStageBytes));
  p.splits = 1;
  p.stages_per_split = p.stages;
  if (dma_eligible(s)) {
    p.dma = true;
    p.bn = g.gemm_n <= 64 ? 64 : 128;
    const int64_t tiles_n = ceil_div(g.gemm_n, p.bn);
    p.wide = g.gemm_n > kWideChannels;
    p.bm = !p.wide && p.stages > 4 && ceil_div(g.gemm_m, 256) * tiles_n >= 192 ? 256 : 128;
    p.m_step = gemm_dma_step(g.gemm_m, tiles_n, p.bm, p.bn);
    return p;
  }
  p.bn = g.gemm_n <= 32 ? 32 : (g.gemm_n <= 64 ? 64 : 128);
  const int64_t tiles_n = ceil_div(g.gemm_n, p.bn);
  p.bm = 64;
  for (int bm : {256, 128}) {
    if (!gemm_tile_supported(bm, p.bn)) continue;
    if (ceil_div(g.gemm_m, bm) * tiles_n >= 512) {
      p.bm = bm;
      break;
    }
  }
  if (!gemm_tile_supported(p.bm, p.bn)) p.bm = 128;
  return p;
}

int64_t staged_tiles(const i8conv_shape &s, const i8conv_geometry &g) {
  const GemmPlan p = plan_staged(s, g);
  return ceil_div(g.gemm_m, p.bm) * ceil_div(g.gemm_n, p.bn);
}

static void set_gemm32(const i8conv_geometry &g, GemmPlan &p, int bm, int bn) {
  const int64_t tiles = ceil_div(g.gemm_m, bm) * ceil_div(g.gemm_n, bn);
  p.m32 = true;
  p.bm = p.m_step = bm;
  p.bn = bn;
  if (bm == 64 && p.stages >= 6 && tiles <= (p.stages >= 8 ? 1152 : 512))
    p.kg = p.stages >= 24 && tiles <= 256 ? 4 : 2;
}

// The 32 x 32 x 32 MFMA kernel's tile for any channel count, or none (below).
static void gemm32_tile(const i8conv_geometry &g, GemmPlan &p) {
  auto tiles = [&](int bm, int bn) { return ceil_div(g.gemm_m, bm) * ceil_div(g.gemm_n, bn); };
  if (g.gemm_n > 64 && p.stages >= 8 && tiles(64, 64) <= 896)
    set_gemm32(g, p, 64, 64);
  else if (g.gemm_n > 64 && tiles(128, 128) >= 256)
    set_gemm32(g, p, 128, 128);
  else if (tiles(128, 64) >= (g.gemm_n <= 32 ? 256 : 512))
    set_gemm32(g, p, 128, g.gemm_n <= 32 ? 32 : 64);
  else if (g.gemm_n > 64 || p.stages >= 6 ||
           (tiles(64, 64) > 256 && (g.gemm_n > 32 || p.stages > 3)))
    set_gemm32(g, p, 64, 64);
}

// Which kernel runs a generic layer, and on which tile (microseconds per
// back-to-back launch on one MI355X, before -> after unless said otherwise).
// C % 128 != 0: the 32 x 32 x 32 MFMA kernel instead of the register-staged
// one, on the largest tile that keeps the compute units covered:
//   * 128 x 128, two workgroups per unit, for N > 64 with at least 256 tiles
//     (256x256, 64 -> 255 3x3: 43 -> 21; 7 x 196x196, 80 -> 209 1x3: 202 ->
//     48; 16 x 224x224, 32 -> 96 4x4 stride 4: 15.8 -> 8.6, 64 x 64: 10.0);
//     But at most 896 tiles of 64 x 64, 1.75 rounds, and eight or more stages:
//     those with two groups of waves, as they leave fewer dead columns (64 x 64,
//     128 x 128: 130x130, 224 -> 160 3x3, 795 tiles: 17.2, 17.9; 4 x 135x135,
//     400 -> 160 5x5 stride 2, 867, int8: 68.1, 70.8; 2 x 238x25, 400 -> 288
//     3x3, 930: 29.4, 28.3; 8 x 64x64, 160 -> 72 3x3, 1024, int8: 15.4, 12.2;
//     22 x 40x40, 400 -> 96 1x3, 1100: 15.8, 14.6, int8 16.8, 15.0);
//   * 128 x 64, three per unit, with at least 512 tiles (16 x 224x224, 32 ->
//     64 7x7 stride 2: 101 -> 35; 256x256, 64 -> 63: 16.4 -> 9.3), 128 x 32
//     for at most 32 channels (30 x 97x108, 32 -> 32 7x7 stride 2: 128 x 64
//     18.0 -> 15.6; 16 x 56x56, 96 -> 32: 8.0 -> 7.3), from 256 tiles on: half
//     of a 64 x 64 tile would be dead (register-staged, 64 x 64, 128 x 32:
//     248x248, 160 -> 32 3x3: 13.8, 14.4, 10.4; 223x223, 48 -> 32 3x3: 6.9,
//     7.4, 5.9; 184x184, 48 -> 32: 6.2, 6.4, 5.6);
//   * 64 x 64, four per unit, below that (416x416, 32 -> 64 3x3 stride 2: 7.3
//     -> 5.9, 128 x 64: 7.6).  With at most two tiles per unit a stage's
//     latency counts, not its throughput: then groups of waves share a tile's
//     stages (one group, two, four): two of them from six stages on (2 x
//     118x118, 96 -> 72 3x3 stride 2, 7 stages: 6.0, 5.6; 4 x 28x28, 192 -> 192
//     3x3, 14 stages: 8.2, 6.8, 7.6; 7 x 38x38, 288 -> 32, 21 stages: 10.6, 8.4,
//     8.9; 2 x 70x70, 288 -> 160, 462 tiles: 13.5, 12.4), four from 24 stages on
//     and at most one tile per unit (193x34, 432 -> 96, 31 stages: 14.2, 10.9,
//     10.8; 16 x 12x12, 400 -> 192 5x3 stride 2, 47 stages: 19.4, 13.7, 13.0);
//   * the register-staged kernel keeps layers of at most 64 channels, fewer
//     than six stages and one round of 64-pixel tiles (2 x 30x30, 48 -> 64
//     3x3: 5.5 against 6.0), and those of at most 32 channels and three stages
//     that are too small for 128 x 32 (130x130, 32 -> 32 1x1: 3.8, 4.1; 176x176,
//     32 -> 32 3x3: 5.1, 5.3; five stages, 352x352, 64 -> 32 3x3 stride 2: 6.9,
//     6.2).
// C % 128 == 0: the pipelined kernel, except
//   * at most one tile of 64 x 64 per unit and six stages or more: 64 x 64
//     (pipelined, 64 x 64: 52x52, 256 -> 512 3x3 stride 2: 10.0, 7.5; 2 x 40x40,
//     256 -> 192, 150 tiles: 10.1, 7.7; 36x36, 512 -> 256, 36 stages: 16.0,
//     11.2; 2 x 128x128, 384 -> 72 stride 2, 256 tiles, int8: 14.0, 11.6; beyond
//     that two rounds: 2 x 134x134, 256 -> 72 dilated, 282 tiles: 10.3, 11.1;
//     180x180, 128 -> 256 stride 2, 508 tiles: 7.6, 8.6);
//   * three or four stages and N no multiple of 128, up to 64 too: 128 x 64
//     from 512 tiles on (64 x 28x28, 384 -> 192 1x1: 19.0 -> 12.3; 53 x 62x62,
//     512 -> 288: 103 -> 94; 30 x 60x60, 384 -> 64: 14.6 -> 12.5; 20 x 60x60,
//     128 -> 64 1x3: 10.8 -> 8.1; two stages, 32 x 56x56, 256 -> 160: 24.7, 25.4);
//   * at least two rounds of 256 x 256 tiles: a third fewer copied bytes per
//     operation (16 x 256x256, 256 -> 256 3x3: 718 -> 614; 5x5 stride 2 with
//     int8 output: 411 -> 376).  Not where they compute more than 8/7 of the
//     channel columns that 128-wide tiles do (128-wide, 256-wide: 4 x 128x140
//     dilated, 256 -> 288: 71, 95, int8 67, 90; 8 x 128x128, 128 -> 260: 74,
//     85; 512x128, 256 -> 640: 104, 109; 256 -> 1152: 181, 177), nor, from 16
//     stages on, where more than an eighth of the rounds would be empty
//     (520x128, 512 -> 512, 520 tiles: 166, 186; 850x128, 256 -> 512, 850
//     tiles: 140, 145; with nine stages int8 gains what int32 loses: 1200x128,
//     128 -> 256, 600 tiles: 78.6, 69.5 and 67.7, 71.1).
static bool wide_tiles(const i8conv_geometry &g, int stages) {
  const int64_t tiles_n = ceil_div(g.gemm_n, 256), narrow_n = ceil_div(g.gemm_n, 128);
  const int64_t tiles = ceil_div(g.gemm_m, 256) * tiles_n, rounds = ceil_div(tiles, 256);
  return stages >= 8 && tiles >= 512 && 7 * 2 * tiles_n <= 8 * narrow_n &&
         (stages < 16 || 8 * tiles >= 7 * 256 * rounds);
}

GemmPlan plan_generic(const i8conv_shape &s, const i8conv_geometry &g) {
  GemmPlan p = plan_staged(s, g);
  if (pointwise_eligible(s, g)) {
    p.pw = true;
    p.pw_waves = pointwise_waves(g.gemm_m, pointwise_slices(s.c, int(g.gemm_n)));
    if (p.dma) return p;  // the fallback for unaligned pointers stays pipelined
  }
  if (!gemm32_eligible(s, g)) return p;
  auto tiles = [&](int bm, int bn) { return ceil_div(g.gemm_m, bm) * ceil_div(g.gemm_n, bn); };
  if (!p.dma)
    gemm32_tile(g, p);
  else if (wide_tiles(g, p.stages))
    set_gemm32(g, p, 256, 256);
  else if (p.stages >= 3 && p.stages <= 4 && g.gemm_n % 128 != 0 && tiles(128, 64) >= 512)
    set_gemm32(g, p, 128, 64);
  else if (p.stages >= 6 && tiles(64, 64) <= 256)
    set_gemm32(g, p, 64, 64);
  return p;
}

// The 32 x 32 x 32 MFMA kernel's plan for int8 output in byte stores, where
// the dispatched kernel cannot requantize (the pipelined kernel with N % 4 != 0
// or a misaligned output, the register-staged, halo and strip kernels).
GemmPlan plan_gemm32(const i8conv_shape &s, const i8conv_geometry &g) {
  GemmPlan p = plan_generic(s, g);
  if (p.m32 || !gemm32_eligible(s, g)) return p;
  p.pw = false;
  gemm32_tile(g, p);
  if (!p.m32) set_gemm32(g, p, 64, 64);
  return p;
}

// Split-K: a 128-pixel tile (64 for tiny M on the register-staged kernel),
// with the 128-byte k stages divided among enough splits to give about one
// workgroup per compute unit (pipelined kernel: its LDS ring allows one per
// unit) or two (register-staged).
GemmPlan plan_splitk(const i8conv_shape &s, const i8conv_geometry &g) {
  GemmPlan p;
  p.stages = int(ceil_div(g.gemm_k, kStageBytes));
  // 3x3 stride-1 layers whose output pixels all fit one workgroup's LDS
  // planes: the deep-channel kernel, one split per 128 input channels
  if (plan_deepk(s, g, &p.deep_plan)) {
    p.deep = true;
    p.dma = true;
    p.bm = int(g.gemm_m);
    p.bn = 32;
    p.splits = p.deep_plan.splits;
    p.stages_per_split = int(ceil_div(9 * 128, kStageBytes));
    return p;
  }
  p.dma = dma_eligible(s);
  if (p.dma) {
    p.wide = g.gemm_n > kWideChannels;
    p.bn = g.gemm_n <= 64 ? 64 : 128;
    p.bm = 128;
  } else {
    p.bn = g.gemm_n <= 32 ? 32 : (g.gemm_n <= 64 ? 64 : 128);
    p.bm = g.gemm_m <= 64 ? 64 : 128;
    if (!gemm_tile_supported(p.bm, p.bn)) p.bm = 128;
  }
  const int64_t tiles = ceil_div(g.gemm_m, p.bm) * ceil_div(g.gemm_n, p.bn);
  int64_t splits = ceil_div(p.dma ? 256 : 512, tiles);
  splits = std::max<int64_t>(2, std::min<int64_t>(splits, p.stages));
  p.stages_per_split = int(ceil_div(p.stages, splits));
  p.splits = int(ceil_div(p.stages, p.stages_per_split));
  return p;
}

size_t splitk_workspace_bytes(const i8conv_geometry &g, const GemmPlan &p) {
  return size_t(p.splits) * size_t(g.gemm_m) * size_t(g.gemm_n) * sizeof(int32_t);
}

namespace {

constexpr int kMaxTilePixels = 128;   // 8 MFMA column fragments
constexpr int kMaxStagePixels = 768;  // 12 staged 16-byte chunks per thread

enum class PatchMode { kStagedHalo, kStrip };

// Resident-halo plan (kernel_halo.hip).  The filter slice of a wave
// (16*fn channels x gemm_k bytes) must match an instantiated kernel, and
// every tap of every output pixel must land inside the zero-padded image
// (true unless out_h/out_w come from the truncating formula with a negative
// numerator).  Ranges: as few as fill the compute units once, more while
// the input rows of the longest range do not fit LDS.
bool plan_resident(const i8conv_shape &s, const i8conv_geometry &g, PatchPlan *p) {
  if (s.c % 64 != 0 || g.gemm_k % 64 != 0) return false;
  const int steps = g.gemm_k / 64;
  const int fn = (s.k > 64 && halo_instance_exists(2, steps)) ? 2 : 1;
  if (!halo_instance_exists(fn, steps)) return false;
  const int hp = s.h + 2 * s.pad_h;
  const int wp = s.w + 2 * s.pad_w;
  if (int64_t(g.out_h - 1) * s.stride_h + int64_t(s.r - 1) * s.dilation_h >= hp) return false;
  if (int64_t(g.out_w - 1) * s.stride_w + int64_t(s.s - 1) * s.dilation_w >= wp) return false;
  const int64_t total_frags = ceil_div(g.gemm_m, 16);
  const int tiles_n = int(ceil_div(s.k, 64 * fn));
  auto vrow = [&](int64_t m) {
    const int64_t b = m / (int64_t(g.out_h) * g.out_w);
    const int64_t oy = (m % (int64_t(g.out_h) * g.out_w)) / g.out_w;
    return b * hp + oy * s.stride_h;
  };
  const HaloRowLayout row = halo_row_layout(wp, s.c, kHaloPadUnits);
  if (row.row_bytes > kLdsBudget) return false;
  const int64_t first = std::max<int64_t>(1, std::min(total_frags, ceil_div(256, tiles_n)));
  const int64_t chunks = ceil_div(g.gemm_k, 128);
  for (int64_t ranges = first; ranges <= total_frags;
       ranges = std::min(total_frags, ranges * 5 / 4 + 1)) {
    // each workgroup re-reads the whole filter slice: beyond the first grid
    // that fills the compute units, keep at least four fragments per range
    if (ranges > first && total_frags / ranges < 4) break;
    int64_t max_rows = 0;
    for (int64_t r = 0; r < ranges; ++r) {
      const int64_t f0 = r * total_frags / ranges, f1 = (r + 1) * total_frags / ranges;
      if (f1 <= f0) continue;
      const int64_t m0 = f0 * 16, m1 = std::min<int64_t>(f1 * 16, g.gemm_m) - 1;
      const int64_t rows = vrow(m1) - vrow(m0) + int64_t(s.r - 1) * s.dilation_h + 1;
      max_rows = std::max(max_rows, rows);
    }
    const int64_t input_lds = kHaloBiasLds + max_rows * row.row_bytes;
    const int64_t slot = int64_t(halo_ring_slot_bytes(fn));
    const int64_t ring = input_lds >= kLdsBudget ? 0 :
        std::min<int64_t>({kHaloRing, chunks, (kLdsBudget - input_lds) / slot});
    if (ring >= 1 && ranges * tiles_n <= INT32_MAX) {
      p->ring = int(ring);
      p->resident = true;
      p->strip = false;
      p->bn = 64 * fn;
      p->tiles_n = tiles_n;
      p->ranges = int(ranges);
      p->rows = int(max_rows);
      p->frags_m = int(ceil_div(total_frags, ranges));
      p->th = p->tw = p->ph = p->pw = 0;
      p->tiles_y = p->tiles_x = 1;
      p->stage_pixels = int(max_rows * wp);
      return true;
    }
    if (ranges == total_frags) break;
  }
  return false;
}

// Row-streaming plan (kernel_row.hip): 3x3, stride 1, dilation 1, c % 64.
// Output rows of each image are cut into `blocks` near-equal blocks so the
// grid (n * blocks * tiles_n workgroups) covers the 256 compute units; a
// block's padded input rows (its rows plus two) must fit in LDS beside the
// filter ring.
bool plan_row(const i8conv_shape &s, const i8conv_geometry &g, PatchPlan *p) {
  if (!(s.r == 3 && s.s == 3 && s.stride_h == 1 && s.stride_w == 1 && s.dilation_h == 1 &&
        s.dilation_w == 1 && s.c % 64 == 0))
    return false;
  // the row kernels' geometry travels in packed preloaded argument words and
  // their grid is (channel tiles, row blocks, images)
  if (s.n >= 65536 || s.h >= 65536 || s.w >= 65536 || s.pad_h >= 256 || s.pad_w >= 256)
    return false;
  const int cg = s.c / 64;
  const int nfr = int(ceil_div(g.out_w, 16));
  const HaloRowLayout row = halo_row_layout(int64_t(s.w) + 2 * s.pad_w, s.c, kRowPadUnits);
  const int64_t chunks = ceil_div(g.gemm_k, 128);
  // For each channel slice width (16*fn channels per wave), the smallest
  // number of row blocks per image that gives every compute unit a
  // workgroup and fits in LDS.  Among the widths with a plan, keep the one
  // whose workgroup copies the fewest bytes (input rows + filter slice):
  // that copy is what the workgroup waits for before its MFMAs can run.
  bool found = false;
  int64_t best_bytes = 0;
  for (int fn : {2, 1}) {
    if (fn == 2 && s.k <= 64) continue;
    if (!row_instance_exists(fn, cg, nfr)) continue;
    const int tiles_n = int(ceil_div(s.k, 64 * fn));
    const int64_t slot = int64_t(halo_ring_slot_bytes(fn));
    int64_t blocks = std::min<int64_t>(g.out_h, std::max<int64_t>(1, ceil_div(256, int64_t(s.n) * tiles_n)));
    for (; blocks <= g.out_h; ++blocks) {
      const int64_t rows = ceil_div(g.out_h, blocks) + 2;
      const int64_t input_lds = kHaloBiasLds + rows * row.row_bytes;
      if (input_lds >= kLdsBudget) continue;
      const int64_t ring = std::min<int64_t>({kHaloRing, chunks, (kLdsBudget - input_lds) / slot});
      if (ring < 1) continue;
      if (int64_t(s.n) * blocks * tiles_n > INT32_MAX) break;
      const int64_t bytes = rows * row.row_bytes + int64_t(64) * fn * g.gemm_k;
      if (!found || bytes < best_bytes) {
        found = true;
        best_bytes = bytes;
        *p = PatchPlan{};
        p->row = true;
        p->bn = 64 * fn;
        p->tiles_n = tiles_n;
        p->ranges = int(blocks);
        p->rows = int(rows);
        p->ring = int(ring);
        p->frags_m = nfr;
        p->tiles_y = p->tiles_x = 1;
        p->stage_pixels = int(rows * (s.w + 2 * s.pad_w));
      }
      break;
    }
  }
  if (!found) return false;
  // 128 channels in 64-channel slices: the form with copy waves when it fits
  p->streamed = s.c == 128 && p->bn == 64 && rowpass_nfr(g.out_w) != 0 &&
                p->rows - 2 <= rowpass_max_rows(rowpass_nfr(g.out_w)) &&
                rowpass_lds_bytes(s.w + 2 * s.pad_w, p->rows - 2) <= size_t(kLdsBudget) &&
                g.output_elements * 4 <= INT32_MAX;
  // A grid of one round and a bit (273 workgroups) takes fewer blocks per
  // image, so that it is one round, where a block's input rows then grow by at
  // most a quarter, or by half where two blocks do not fit a unit's LDS (us per
  // launch before -> after): 21 x 36x36, 64 -> 64: 8.6 -> 5.3 (same rows); 37 x
  // 20x20, 256 -> 64: 15.5 -> 9.7 (5 -> 6); 9 x 50x50, 64 -> 192: 14.3 -> 8.3
  // (7 -> 8); 13 x 30x30, 128 -> 416, 125 KB of LDS: 20.3 -> 13.3 (12 -> 17); 25
  // x 24x24, 64 -> 256, 72 KB, would take 14 rows instead of 10: 8.4 -> 8.9,
  // int8 9.7 -> 13.4.
  const int64_t per_block = int64_t(s.n) * p->tiles_n;
  const int64_t fewer = 256 / per_block;
  if (!p->streamed && per_block * p->ranges > 256 && fewer >= 1 && fewer < p->ranges) {
    const int64_t slot = int64_t(halo_ring_slot_bytes(p->bn / 64));
    const int64_t rows = ceil_div(g.out_h, fewer) + 2;
    const int64_t input_lds = kHaloBiasLds + rows * row.row_bytes;
    const int64_t ring = std::min<int64_t>({kHaloRing, chunks, (kLdsBudget - input_lds) / slot});
    const int64_t now = kHaloBiasLds + p->rows * row.row_bytes + p->ring * slot;
    if (input_lds < kLdsBudget && ring >= 1 &&
        4 * rows <= (2 * now > kLdsBudget ? 6 : 5) * int64_t(p->rows)) {
      p->ranges = int(fewer);
      p->rows = int(rows);
      p->ring = int(ring);
      p->stage_pixels = int(rows * (s.w + 2 * s.pad_w));
    }
  }
  return true;
}

bool finish_patch_plan(const i8conv_shape &s, const i8conv_geometry &g,
                       PatchMode mode, PatchPlan *p) {
  (void)mode;
  p->stage_pixels = p->ph * p->pw;
  if (p->stage_pixels > kMaxStagePixels) return false;
  if (size_t(2) * p->stage_pixels * 64 > size_t(kLdsBudget)) return false;
  p->tiles_y = int(ceil_div(g.out_h, p->th));
  p->tiles_x = int(ceil_div(g.out_w, p->tw));
  p->tiles_n = int(ceil_div(s.k, p->bn));
  p->frags_m = int(ceil_div(int64_t(p->th) * p->tw, 16));
  p->loads_per_thread = int(ceil_div(int64_t(p->stage_pixels) * 4, kThreads));
  const int64_t blocks = int64_t(s.n) * p->tiles_y * p->tiles_x * p->tiles_n;
  return blocks <= INT32_MAX;
}

// Tile search shared by halo and strip: the widest tile (whole output rows
// when out_w <= 128) whose staged region fits, preferring pixel counts that
// fill whole 16-column MFMA fragments.
bool search_patch_plan(const i8conv_shape &s, const i8conv_geometry &g,
                       PatchMode mode, int bn, PatchPlan *out) {
  PatchPlan best;
  bool found = false;
  double best_score = -1.0;
  for (int tw = std::min(g.out_w, kMaxTilePixels); tw >= 1; --tw) {
    // only full-width tiles, or widths that split the row evenly
    if (tw != g.out_w && g.out_w % tw != 0) continue;
    const int th_max = std::min(g.out_h, kMaxTilePixels / tw);
    for (int th = th_max; th >= 1; --th) {
      PatchPlan p;
      p.strip = mode == PatchMode::kStrip;
      p.th = th;
      p.tw = tw;
      p.bn = bn;
      if (p.strip) {
        p.ph = th;
        p.pw = tw + s.s - 1;
      } else {
        p.ph = (th - 1) * s.stride_h + (s.r - 1) * s.dilation_h + 1;
        p.pw = (tw - 1) * s.stride_w + (s.s - 1) * s.dilation_w + 1;
      }
      if (!finish_patch_plan(s, g, mode, &p)) continue;
      const int px = th * tw;
      // useful fraction of the MFMA columns the whole grid computes (edge
      // tiles included), times a mild preference for big tiles (less halo
      // re-read, fewer passes over the filter)
      const double fill = double(g.out_h) * g.out_w /
                          (double(p.tiles_y) * p.tiles_x * p.frags_m * 16);
      const double score = fill * (0.75 + 0.25 * double(px) / kMaxTilePixels);
      if (score > best_score + 1e-9) {
        best_score = score;
        best = p;
        found = true;
      }
      break;  // larger th is better for a given tw; stop at first fit
    }
  }
  if (found) *out = best;
  return found;
}

}  // namespace

// Halo-tiled predicate: 64-channel groups and a tile whose receptive field
// fits LDS.  Any filter size, stride and dilation.  3x3 layers whose halo of
// all channel groups fits LDS use the resident-halo kernel (input read once
// per tile, filter streamed); the others stage one channel group at a time.
bool plan_halo(const i8conv_shape &s, const i8conv_geometry &g, PatchPlan *p) {
  if (s.c % 64 != 0) return false;
  const int bn = s.k > 64 ? 128 : 64;
  if (plan_row(s, g, p) || plan_resident(s, g, p))
    return true;
  return search_patch_plan(s, g, PatchMode::kStagedHalo, bn, p);
}

// Spatial-strip predicate, re-derived from spatial_strip.cuh:11-15 for the
// gfx950 tile: 3x3 filter, horizontal stride and dilation 1 (the strip is
// reused across the three filter columns), C % 64 == 0 (one 64-channel MFMA
// k-block per stage).  The reference's K % 64 and out_w % 128 conditions are
// gone: the tile covers whole output rows (or an even split of a row) and
// the epilogue guards the channel tail.  Vertical stride/dilation and padding
// are free, as in the reference.
bool plan_strip(const i8conv_shape &s, const i8conv_geometry &g, PatchPlan *p) {
  if (!(s.r == 3 && s.s == 3 && s.stride_w == 1 && s.dilation_w == 1 &&
        s.c % 64 == 0))
    return false;
  return search_patch_plan(s, g, PatchMode::kStrip, s.k > 64 ? 128 : 64, p);
}

ConvArgs make_args(const i8conv_shape &s, const i8conv_geometry &g,
                   const int8_t *x, const int8_t *w, const int32_t *bias,
                   int32_t *y) {
  ConvArgs a{};
  a.x = x;
  a.w = w;
  a.bias = bias;
  a.y = y;
  a.partial = nullptr;
  a.n = s.n;
  a.h = s.h;
  a.wd = s.w;
  a.c = s.c;
  a.k = s.k;
  a.r = s.r;
  a.s = s.s;
  a.pad_h = s.pad_h;
  a.pad_w = s.pad_w;
  a.stride_h = s.stride_h;
  a.stride_w = s.stride_w;
  a.dil_h = s.dilation_h;
  a.dil_w = s.dilation_w;
  a.out_h = g.out_h;
  a.out_w = g.out_w;
  a.gemm_m = int(g.gemm_m);
  a.gemm_n = g.gemm_n;
  a.gemm_k = g.gemm_k;
  a.x_bytes = uint32_t(g.input_elements);
  a.w_bytes = uint32_t(g.filter_elements);
  a.div_c = make_fastdiv(uint32_t(s.c));
  a.div_s = make_fastdiv(uint32_t(s.s));
  a.div_ow = make_fastdiv(uint32_t(g.out_w));
  a.div_ohw = make_fastdiv(uint32_t(int64_t(g.out_h) * g.out_w));
  a.stages_per_split = 0;
  a.splits = 1;
  a.m_step = 0;
  return a;
}

}  // namespace i8conv
