// Dispatch policy, kept outside the kernels (the reference's workflow,
// README.md:92-99: sweep, then encode the policy outside the kernels while
// eligibility stays an explicit predicate next to each kernel).
//
// The policy only ever returns an eligible kernel.  Its rules, in order,
// read off a sweep of the reference's 41-layer table on one MI355X:
//   1. the row-streaming 3x3 stride-1 kernel (a halo plan) whenever it has a
//      plan: it won every layer it covers (ResNet/Darknet 3x3 stages,
//      batched 56x56 and 28x28 layers, 14x14 C = 256);
//   2. split-K when the generic grid is tiny (at most 16 tiles) and the
//      reduction long: at least 16 stages of 128 k-bytes, or 8 for a 1x1
//      filter (deep 7x7 / 13x13 / 14x14 layers and stride-2 downsamplers at
//      batch 1: it won all of them; at 24 tiles and 18 stages the generic
//      GEMM won, 15.0 vs 15.7 us, and on a 32x32 3x3 layer of 9 stages the
//      halo kernel, 9.3 vs 11.0 us);
//   3. the resident-rows form of the halo kernel where each of its workgroups
//      has one fragment of 16 pixels, a filter slice of at most 72 KB and at
//      most 28 KB of input rows: the generic kernel's smallest grids are slower
//      there, by less the more input a workgroup copies first (3 x 9x9, 192 ->
//      96 1x3, 9 KB: 4.5 against 5.0 us; 2 x 24x24, 192 -> 160 1x3, 13 KB: 4.7,
//      5.1; 1 x 15x15, 128 -> 64 dilated 2, 19 KB: 5.4, 5.6; level at 25 to 30 KB;
//      1 x 38x38, 192 -> 128 3x1, 32 KB: 5.3, 5.1);
//   4. the generic GEMM wherever it runs its pipelined form (C % 128 == 0) or
//      the 32 x 32 x 32 MFMA one: they beat every other halo and strip plan
//      without row streaming (C % 128 == 0: 3 x 44x44, 512 -> 160 3x1: 25.6 ->
//      8.3; 36x36, 512 -> 256 3x3: 45.9 -> 16.1; 2 x 40x40 dilated 256 -> 192: 27.7
//      -> 10.0; 4 x 60x30, 128 -> 64 1x3: 7.9 -> 4.5; others: 1x3, 64 -> 128:
//      22.3 -> 14.2; 256x256, 64 -> 63, 69, 255: 16.4, 19.2, 43 -> 9.3, 11.1,
//      21; dilated 64 -> 128: 6.3 -> 5.3);
//   5. otherwise an input-reuse kernel for a stride-1 spatial filter
//      (r*s > 1): halo when eligible, else strip (small dilated layers,
//      asymmetric 1x3/3x1, C = 64 layers wider than the row kernel's four
//      fragments); at stride 2 the generic GEMM beat the halo kernel on
//      every such layer (15.0 vs 18.0 us at 52x52, C = 256);
//   6. otherwise the generic implicit GEMM (1x1 layers, strided layers,
//      C % 64 != 0).
#include <cstring>
#include <mutex>

#include "i8conv_internal.hpp"

namespace i8conv {

namespace {
struct Choice {
  int id;
  bool patch;  // dispatch_patch_layer
};
Choice dispatch_uncached(const i8conv_shape &s);

// The policy is a pure function of the shape, and its planners search
// (the resident-rows plan of a 64x64 dilated layer takes ~50 us of host
// time), so results are kept in a small direct-mapped cache: launches that
// go through the policy every call (the requantized launch, conv2d) then
// cost a lookup.
struct DispatchEntry {
  i8conv_shape shape;
  Choice choice;
  bool used;
};
constexpr size_t kDispatchCache = 64;
std::mutex g_dispatch_mutex;
DispatchEntry g_dispatch_cache[kDispatchCache];

size_t shape_slot(const i8conv_shape &s) {
  const int *f = reinterpret_cast<const int *>(&s);
  uint32_t h = 2166136261u;  // FNV-1a over the 13 int fields
  for (size_t i = 0; i < sizeof(s) / sizeof(int); ++i) h = (h ^ uint32_t(f[i])) * 16777619u;
  return h % kDispatchCache;
}

Choice lookup(const i8conv_shape &s) {
  static_assert(sizeof(i8conv_shape) == 13 * sizeof(int), "shape fields are 13 ints");
  const size_t slot = shape_slot(s);
  {
    std::lock_guard<std::mutex> lock(g_dispatch_mutex);
    const DispatchEntry &e = g_dispatch_cache[slot];
    if (e.used && std::memcmp(&e.shape, &s, sizeof(s)) == 0) return e.choice;
  }
  const Choice choice = dispatch_uncached(s);
  std::lock_guard<std::mutex> lock(g_dispatch_mutex);
  g_dispatch_cache[slot] = DispatchEntry{s, choice, true};
  return choice;
}
}  // namespace

int dispatch(const i8conv_shape &s) { return lookup(s).id; }

bool dispatch_patch_layer(const i8conv_shape &s) { return lookup(s).patch; }

namespace {
Choice dispatch_uncached(const i8conv_shape &s) {
  i8conv_geometry g;
  if (derive(s, &g) != I8CONV_OK) return {-1, false};
  PatchPlan pp;
  const bool halo = plan_halo(s, g, &pp);
  if (halo && pp.row) return {I8CONV_KERNEL_HALO, false};
  const GemmPlan gp = plan_generic(s, g);
  const int64_t tiles = staged_tiles(s, g);
  const bool spatial = int64_t(s.r) * s.s > 1;
  if (tiles <= 16 && (gp.stages >= 16 || (!spatial && gp.stages >= 8)))
    return {I8CONV_KERNEL_SPLITK, false};
  const bool reuse = spatial && s.stride_h == 1 && s.stride_w == 1;
  if (halo && reuse && pp.resident && pp.frags_m == 1 &&
      int64_t(pp.bn) * g.gemm_k <= 72 * 1024 &&
      pp.rows * halo_row_layout(int64_t(s.w) + 2 * s.pad_w, s.c, kHaloPadUnits).row_bytes <=
          28 * 1024)
    return {I8CONV_KERNEL_HALO, false};
  const bool patch = reuse && gp.dma && tiles < 128 && (halo || plan_strip(s, g, &pp));
  if (gp.m32 || gp.dma) return {I8CONV_KERNEL_GENERIC, patch};
  if (reuse) {
    if (halo) return {I8CONV_KERNEL_HALO, false};
    if (plan_strip(s, g, &pp)) return {I8CONV_KERNEL_STRIP, false};
  }
  return {I8CONV_KERNEL_GENERIC, false};
}
}  // namespace

}  // namespace i8conv
