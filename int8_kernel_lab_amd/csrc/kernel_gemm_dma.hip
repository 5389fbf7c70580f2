// Pipelined generic implicit GEMM on gfx950 INT8 MFMA, for layers whose
// input channels are a multiple of 128 (every 128-byte k-stage then lies in
// one filter tap), and its split-K form.
//
// Same GEMM view and semantics as kernel_gemm.hip (generic_implicit_gemm.cuh
// :90-153 of the reference: M = n*out_h*out_w pixels, N = k output
// channels, K = r*s*c with k = (fy*s + fx)*c + ci); what changes is how the
// operands reach the MFMAs:
//   * each 128-byte k-stage of the BN filter rows and the BM im2col rows is
//     copied straight from global memory into LDS by the buffer unit
//     (buffer_load ... lds, 1 KB per wave instruction), no VGPR round trip;
//   * a ring of three stage buffers: stage s + 2 is in flight while stage s
//     feeds the MFMAs, one barrier per stage; the copies of stage s + 2 are
//     issued between the MFMA groups of stage s, or by copy waves (below);
//   * v_mfma_i32_32x32x32 with pixels as rows and channels as columns, and its
//     conflict-free LDS row swizzle (mfma32_tile.hpp).  A copy writes lane i's
//     16 bytes to LDS slot i of its 1 KB block, so the swizzle is applied on
//     the source side: the lane of slot (row, physical chunk) fetches the
//     logical chunk that belongs there;
//   * because a stage lies inside one tap, the tap decomposition is uniform
//     per stage: each lane keeps its rows' pixel origin and adds one tap
//     offset per stage, with two compares for padding;
//   * on the 256 x 128 and 128 x 128 tiles with four or more k-stages per
//     workgroup, waves that only issue the copies: an MFMA wave that also
//     issues copies stalls whenever the buffer unit's queue is full, and its
//     MFMAs wait behind the stalled issue.  256 x 128: eight MFMA waves of 64
//     x 64 and eight copy waves, four waves per SIMD (stride-2 128 -> 256
//     layer, 32 x 56x56: 13.6 us with eight copy waves, 14.9 with four; four
//     MFMA waves of 128 x 64 are 3 % faster on long reductions with int32
//     output but 17 % slower with int8, whose requantization then runs on
//     half the waves).  128 x 128: four MFMA waves of 64 x 64 and four copy
//     waves (32 x 14x14, 512 -> 512: 20.5 us; eight MFMA waves of 64 x 32,
//     which read half as much again from LDS, 21.5), with int8 output eight,
//     which share the requantization (launch_gemm_dma);
//   * an MFMA wave reads the fragments of the next k-step between the MFMAs of
//     the current one, across the stage barrier too.  Against the 16 x 16 x
//     64 form that read a stage's fragments and then ran its MFMAs (us per
//     launch over three sets of tensors, same box): 32 x 56x56, 128 -> 256
//     stride 2: 14.8 -> 12.9, with int8 output 15.2 -> 13.5; 16 x 28x28 1x1
//     512 -> 384: 13.0 -> 10.4; 64 x 28x28 1x1 384 -> 192: 25.0 -> 19.0; 5 x
//     86x86, 384 -> 96: 31.8 -> 26.0; 32 x 14x14, 512 -> 512: 20.4 -> 18.7; 8
//     x 64x64 dilated 256 -> 256: 22.6 -> 21.9 over 60 ms, no difference
//     over seconds, where the power drawn sets the clock: its MFMAs alone
//     take 15.4 us with the launch (2.9 POP/s), its stores, which come at the
//     end of its one round of tiles, 5;
//   * accumulators stay in VGPRs (built with -amdgpu-mfma-vgpr-form);
//   * XCD-aware tile order (see below);
//   * fragments wholly past the last pixel row run no MFMAs.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "i8conv_internal.hpp"
#include "mfma32_tile.hpp"

namespace i8conv {
namespace {

constexpr int kRing = 3;  // stage buffers in LDS

// Calls run(std::integral_constant<int, F>) with F = min(live, FMAX).
template <int F, int FMAX, class Run>
__device__ __forceinline__ void with_live_frags(int live, Run &run) {
  if constexpr (F < FMAX) {
    if (live <= F) {
      run(std::integral_constant<int, F>{});
      return;
    }
    with_live_frags<F + 1, FMAX>(live, run);
  } else {
    run(std::integral_constant<int, FMAX>{});
  }
}

// NCW == 0: every wave both copies and runs MFMAs.  NCW > 0: WM*WN MFMA
// waves plus NCW copy waves (waves WM*WN and up) that only issue the stage
// copies, so an MFMA wave never stalls on a copy issue.  The two roles run
// separate loops with the same one barrier per stage, so neither role's
// registers are live in the other's loop.
//
// kWide: more than kWideChannels output channels, where a tile's output window
// can pass 2 GiB: element stores at 64-bit addresses.
template <int BM, int BN, int WM, int WN, bool kSplit, int NCW, bool kWide>
__global__ __launch_bounds__(64 * (WM * WN + NCW)) void gemm_dma_kernel(ConvArgs a) {
  constexpr int NMW = WM * WN;             // MFMA waves
  constexpr int NW = NCW > 0 ? NCW : NMW;  // copy waves
  constexpr int TMW = BM / WM;  // pixels per wave
  constexpr int TNW = BN / WN;  // output channels per wave
  constexpr int FM = TMW / 32;  // 32 x 32 blocks
  constexpr int FN = TNW / 32;
  constexpr int KS = kStageBytes / 32;  // k-steps per stage
  constexpr int kRows = BM + BN;             // LDS rows per stage: filter, then pixels
  constexpr int kTile = kRows * kStageBytes;  // bytes per stage buffer
  constexpr int kCopies = kRows / 8;          // 1 KB copies per stage
  constexpr int CPW = kCopies / NW;           // per wave
  constexpr int CPA = BN / 8 / NW;            // of which filter rows
  static_assert(kCopies % NW == 0 && (BN / 8) % NW == 0 && FM >= 1 && FN >= 1, "tile shape");
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool copier = NCW > 0 && wave_id >= NMW;  // a copy-only wave
  const int wave = copier ? wave_id - NMW : wave_id;  // index within its role
  const int wm = wave % WM;
  const int wn = wave / WM;

  // Workgroup i runs on XCD i % 8 (round-robin dispatch), and each XCD has
  // its own L2.  Tiles are handed out so that every XCD gets a contiguous
  // run of them (both channel tiles of a pixel tile, then the next pixel
  // tile): neighbouring pixel tiles share input rows, which then stay in
  // that XCD's L2 instead of being fetched into two.  A bijection on
  // [0, gridDim.x): the first 8 * (gridDim.x / 8) workgroups are permuted,
  // the rest keep their index.
  const int per_xcd = int(gridDim.x) / 8;
  int tile = int(blockIdx.x);
  if (tile < 8 * per_xcd) tile = (tile % 8) * per_xcd + tile / 8;
  const int tiles_n = (a.gemm_n + BN - 1) / BN;
  const int tile_m = (tile / tiles_n) * a.m_step;
  // pixel rows this tile stores; rows from m_end on read as zeros
  const int m_end = min(a.gemm_m, tile_m + a.m_step);
  const int tile_n = (tile % tiles_n) * BN;
  const int stages = a.gemm_k / kStageBytes;
  int s_begin = 0, s_end = stages;
  if (kSplit) {
    s_begin = int(blockIdx.y) * a.stages_per_split;
    s_end = min(stages, s_begin + a.stages_per_split);
  }

  const v4u xd = make_desc(a.x, a.x_bytes);
  const v4u wd = make_desc(a.w, a.w_bytes);
  const uint32_t lds0 = lds_addr(smem);

  // Copy j of this wave is block q = wave + NW*j of the stage: rows 8q..8q+7,
  // lane -> row 8q + lane/8, physical chunk lane%8.  Copies j < CPA are
  // filter rows (q < BN/8), the rest pixel rows.
  uint32_t abase[CPA];  // filter byte offset of this lane's chunk at stage 0
#pragma unroll
  for (int j = 0; j < CPA; ++j) {
    const int r = 8 * (wave + NW * j) + (lane >> 3);
    const int lc = (lane & 7) ^ swz32_f(r);
    const int oc = tile_n + r;
    abase[j] = oc < a.gemm_n ? uint32_t(oc) * uint32_t(a.gemm_k) + uint32_t(lc * 16)
                             : kOutOfRange;
  }
  constexpr int CPB = CPW - CPA;
  int pix[CPB], iy0[CPB], ix0[CPB];
#pragma unroll
  for (int j = 0; j < CPB; ++j) {
    const int r = 8 * (wave + NW * (CPA + j)) + (lane >> 3);  // >= BN
    const int lc = (lane & 7) ^ swz32_f(r);
    const int m = tile_m + r - BN;
    if (m < m_end) {
      const int b = int(fast_div(uint32_t(m), a.div_ohw));
      const int rem = m - b * a.out_h * a.out_w;
      const int oy = int(fast_div(uint32_t(rem), a.div_ow));
      const int ox = rem - oy * a.out_w;
      iy0[j] = oy * a.stride_h - a.pad_h;
      ix0[j] = ox * a.stride_w - a.pad_w;
      pix[j] = ((b * a.h + iy0[j]) * a.wd + ix0[j]) * a.c + lc * 16;
    } else {
      iy0[j] = -(1 << 29);  // every tap out of the image -> zeros
      ix0[j] = 0;
      pix[j] = 0;
    }
  }

  // Copies of one stage (stage buffers are numbered from the first stage of
  // this workgroup).  Copy j < CPA: filter rows; j >= CPA: pixel rows, at the
  // stage's tap offset, zero-filled where the tap falls in the padding.
  struct StageTap {
    uint32_t dst;
    int dy, dx, tap_off;
  };
  auto stage_tap = [&](int stage) {
    StageTap t;
    t.dst = lds0 + uint32_t(((stage - s_begin) % kRing) * kTile);
    // the stage's tap and channel offset (uniform)
    const int k0 = stage * kStageBytes;
    const int tap = int(fast_div(uint32_t(k0), a.div_c));
    const int ci0 = k0 - tap * a.c;
    const int fy = int(fast_div(uint32_t(tap), a.div_s));
    const int fx = tap - fy * a.s;
    t.dy = fy * a.dil_h;
    t.dx = fx * a.dil_w;
    t.tap_off = (t.dy * a.wd + t.dx) * a.c + ci0;
    return t;
  };
  auto copy = [&](const StageTap &t, int stage, int j) {
    if (j < CPA) {
      lds_copy16(wd, t.dst + uint32_t(wave + NW * j) * 1024u, abase[j] + uint32_t(stage * kStageBytes));
    } else {
      const int jb = j - CPA;
      const bool ok = unsigned(iy0[jb] + t.dy) < unsigned(a.h) && unsigned(ix0[jb] + t.dx) < unsigned(a.wd);
      lds_copy16(xd, t.dst + uint32_t(wave + NW * j) * 1024u,
                 ok ? uint32_t(pix[jb] + t.tap_off) : kOutOfRange);
    }
  };
  auto issue = [&](int stage) {
    const StageTap t = stage_tap(stage);
#pragma unroll
    for (int j = 0; j < CPW; ++j) copy(t, stage, j);
  };

  if (NCW > 0 && copier) {
    // copy wave: keep two stages in flight ahead of the MFMA waves
    issue(s_begin);
    if (s_begin + 1 < s_end) issue(s_begin + 1);
    for (int st = s_begin; st < s_end; ++st) {
      if (st + 1 < s_end)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(CPW) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      // stage st is visible to the MFMA waves, and they are done with stage
      // st - 1, whose buffer stage st + 2 overwrites
      __syncthreads();
      if (st + 2 < s_end) issue(st + 2);
    }
    return;
  }

  // Fragment read offsets inside a stage buffer, per k-step: row 32 i + lane
  // % 32 (32 rows are four whole periods of the swizzle), chunk 2 ks + lane
  // / 32.
  int koff[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
    koff[ks] = (lane & 31) * kStageBytes + 16 * ((2 * ks + (lane >> 5)) ^ swz32_f(lane & 31));
  const int abuf = wn * TNW * kStageBytes, bbuf = (BN + wm * TMW) * kStageBytes;

  v16i acc[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;

  if (NCW > 0) {
    // MFMA wave of a split workgroup: the copy waves fill the ring.  The
    // wave's blocks that lie wholly at or past m_end (the padding of a last
    // pixel tile: 120 of the 128 rows of the deep-K layer's fourth) get no
    // fragment reads and no MFMAs: the walk runs with the live block count
    // as a compile-time constant.
    const int row0 = tile_m + wm * TMW;
    const int live = m_end <= row0 ? 0 : min(FM, (m_end - row0 + 31) / 32);
    auto walk = [&](auto live_frags) {
      constexpr int F = decltype(live_frags)::value;
      // The fragments of one k-step in two register sets: the next k-step's
      // reads go out between the MFMAs of the current one.  The last k-step
      // of a stage reads the next stage's first, so the barrier that says
      // that stage has landed (and that every wave has read all of this one)
      // comes before it.
      v4i af[2][FN], bf[2][F > 0 ? F : 1];
      auto read = [&](auto set, const int8_t *buf, int h, int q) {
        if (q < FN)
          af[set.value][q] = *reinterpret_cast<const v4i *>(buf + abuf + koff[h] + 32 * kStageBytes * q);
        else
          bf[set.value][q - FN] =
              *reinterpret_cast<const v4i *>(buf + bbuf + koff[h] + 32 * kStageBytes * (q - FN));
      };
      constexpr int kReads = F > 0 ? FN + F : 0, kMfma = FN * F;
      __syncthreads();
#pragma unroll
      for (int q = 0; q < kReads; ++q) read(std::integral_constant<int, 0>{}, smem, 0, q);
      int ring = 0;
      for (int st = s_begin; st < s_end; ++st) {
        const int next = ring + 1 == kRing ? 0 : ring + 1;
        const int8_t *buf = smem + ring * kTile, *nbuf = smem + next * kTile;
        auto step = [&](auto set, auto h) {
          constexpr bool kLast = h.value == KS - 1;
          if (kLast && st + 1 < s_end) __syncthreads();
          if constexpr (kMfma > 0) {
#pragma unroll
            for (int n = 0; n < kMfma; ++n) {
#pragma unroll
              for (int q = n * kReads / kMfma; q < (n + 1) * kReads / kMfma; ++q)
                read(std::integral_constant<int, 1 - set.value>{}, kLast ? nbuf : buf,
                     kLast ? 0 : h.value + 1, q);
              acc[n / F][n % F] = mfma32(bf[set.value][n % F], af[set.value][n / F], acc[n / F][n % F]);
              __builtin_amdgcn_sched_barrier(0);
            }
          }
        };
        static_assert(KS == 4, "four k-steps per stage");
        step(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 0>{}, std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 1>{}, std::integral_constant<int, 3>{});
        ring = next;
      }
    };
    with_live_frags<0, FM>(live, walk);
  }
  if (NCW == 0) issue(s_begin);
  if (NCW == 0 && s_begin + 1 < s_end) issue(s_begin + 1);
  for (int st = s_begin; NCW == 0 && st < s_end; ++st) {
    // stage st has landed once only stage st + 1 (if any) is outstanding
    if (st + 1 < s_end)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(CPW) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // every wave's copies of stage st are visible, and every wave is done
    // with stage st - 1, whose buffer the next issue overwrites
    __syncthreads();
    const bool more = st + 2 < s_end;
    const StageTap next = stage_tap(more ? st + 2 : st);
    const int8_t *buf = smem + ((st - s_begin) % kRing) * kTile;
    v4i af[KS][FN], bf[KS][FM];
#pragma unroll
    for (int h = 0; h < KS; ++h) {
#pragma unroll
      for (int i = 0; i < FN; ++i)
        af[h][i] = *reinterpret_cast<const v4i *>(buf + abuf + koff[h] + 32 * kStageBytes * i);
#pragma unroll
      for (int j = 0; j < FM; ++j)
        bf[h][j] = *reinterpret_cast<const v4i *>(buf + bbuf + koff[h] + 32 * kStageBytes * j);
    }
    // MFMAs in KS * FN groups of FM, with the copies of stage st + 2 spread
    // between the groups: a copy whose issue stalls (the buffer unit takes a
    // few in flight per wave) then holds back only a few queued MFMAs.
    constexpr int kGroups = KS * FN;
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      const int h = g / FN, i = g % FN;
#pragma unroll
      for (int j = 0; j < FM; ++j) acc[i][j] = mfma32(bf[h][j], af[h][i], acc[i][j]);
      if (more) {
#pragma unroll
        for (int c = (g * CPW + kGroups - 1) / kGroups; c < ((g + 1) * CPW + kGroups - 1) / kGroups; ++c)
          copy(next, st + 2, c);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // Epilogue (mfma32_tile.hpp): whole 128-byte pieces of output rows per
  // store.
  const int rows = m_end - tile_m;
  const int px0 = wm * TMW, oc0 = tile_n + wn * TNW;
  if constexpr (kWide) {
    int32_t *const y =
        kSplit ? a.partial + size_t(blockIdx.y) * size_t(a.gemm_m) * size_t(a.gemm_n) : a.y;
#pragma unroll
    for (int i = 0; i < FN; ++i) {
      const int oc = oc0 + 32 * i + (lane & 31);
      if (oc >= a.gemm_n) continue;
      const uint32_t bias = kSplit ? 0u : uint32_t(a.bias[oc]);
#pragma unroll
      for (int j = 0; j < FM; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int px = px0 + 32 * j + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
          if (px >= rows) continue;
          const size_t at = size_t(tile_m + px) * size_t(a.gemm_n) + size_t(oc);
          const int32_t v = int32_t(uint32_t(acc[i][j][e]) + bias);
          if (!kSplit && a.q_y)
            a.q_y[at] = int8_t(requant1(v, a.q_mult[oc], a.q_shift[oc], a.q_zp));
          else
            y[at] = v;
        }
    }
    return;
  }
  if (!kSplit && a.q_y) {
    const auto yr = make_rsrc(a.q_y + size_t(tile_m) * size_t(a.gemm_n),
                              uint32_t(rows) * uint32_t(a.gemm_n));
    const auto br = make_rsrc(a.bias, uint32_t(a.gemm_n) * 4u);
    const auto mr = make_rsrc(a.q_mult, uint32_t(a.gemm_n) * 4u);
    const auto sr = make_rsrc(a.q_shift, uint32_t(a.gemm_n) * 4u);
#pragma unroll
    for (int i = 0; i < FN; ++i) {
      const uint32_t off = uint32_t(oc0 + 32 * i + (lane & 31)) * 4u;
      const uint32_t bias = __builtin_amdgcn_raw_buffer_load_b32(br, off, 0, 0);
      const Requant32 r =
          requant32_params(int32_t(__builtin_amdgcn_raw_buffer_load_b32(mr, off, 0, 0)),
                           int32_t(__builtin_amdgcn_raw_buffer_load_b32(sr, off, 0, 0)), a.q_zp);
      const uint32_t base = quad_int8_base<false>(oc0 + 32 * i, a.gemm_n, lane);
#pragma unroll
      for (int j = 0; j < FM; ++j) {
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = int(uint32_t(acc[i][j][e]) + bias);
        requant_block32<false>(acc[i][j], r, a.q_zp, yr, base, px0 + 32 * j, a.gemm_n, lane);
      }
    }
    return;
  }
  int32_t *out = a.y;
  if (kSplit) {
    out = a.partial + size_t(blockIdx.y) * size_t(a.gemm_m) * size_t(a.gemm_n);
  } else {
    const auto br = make_rsrc(a.bias, uint32_t(a.gemm_n) * 4u);
#pragma unroll
    for (int i = 0; i < FN; ++i) {
      const uint32_t bias = __builtin_amdgcn_raw_buffer_load_b32(
          br, uint32_t(oc0 + 32 * i + (lane & 31)) * 4u, 0, 0);
#pragma unroll
      for (int j = 0; j < FM; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = int(uint32_t(acc[i][j][e]) + bias);
    }
  }
  const auto yr = make_rsrc(out + size_t(tile_m) * size_t(a.gemm_n),
                            uint32_t(rows) * uint32_t(a.gemm_n) * 4u);
  // Partial sums of the 64-channel tiles: short walks, where a quarter of the
  // stores counts for more than the code of the transposes (3 x 19x19, 256 ->
  // 48 dilated: 7.9 us in 4-byte stores, 7.7 so; two 128-channel tiles: no
  // difference on average, 3 x 27x27, 1024 -> 128 1x1: 6.9, 7.3).
  if constexpr (kSplit && BN == 64) {
    if ((a.gemm_n & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0) {
      if (sector_pitch(a.gemm_n))
        store_tile32_x4<kStoreThrough>(acc, yr, rows, px0, oc0, a.gemm_n, lane);
      else
        store_tile32_x4<0>(acc, yr, rows, px0, oc0, a.gemm_n, lane);
      return;
    }
  }
  // Outputs beyond 128 MiB: evict-first.  Written through, such outputs ran
  // up to 1.75x slower (16x256x256x256 1x1: 220 -> 388 us; 268 MB and up all
  // lost), while every output of the baseline layers (0.8-51 MB) gains from
  // it.
  if (!kSplit && int64_t(a.gemm_m) * a.gemm_n * 4 > kStreamOutputBytes)
    store_tile32<kStoreStream>(acc, yr, rows, px0, oc0, a.gemm_n, lane);
  else if (sector_pitch(a.gemm_n))
    store_tile32<kStoreThrough>(acc, yr, rows, px0, oc0, a.gemm_n, lane);
  else
    store_tile32<0>(acc, yr, rows, px0, oc0, a.gemm_n, lane);
}

template <int BM, int BN, int WM, int WN, int NCW = 0, bool kSplits = true, bool kWide = false>
int launch_tile(const ConvArgs &a, int splits, hipStream_t stream) {
  const int tiles = int(((int64_t(a.gemm_m) + a.m_step - 1) / a.m_step) * ((a.gemm_n + BN - 1) / BN));
  const int stages = a.gemm_k / kStageBytes;
  const int ring = std::min(kRing, splits > 1 ? a.stages_per_split : stages);
  const size_t lds = size_t(ring) * size_t(BM + BN) * kStageBytes;
  auto kern = gemm_dma_kernel<BM, BN, WM, WN, false, NCW, kWide>;
  if constexpr (kSplits) {
    if (splits > 1) kern = gemm_dma_kernel<BM, BN, WM, WN, true, NCW, kWide>;
  }
  static LdsLimit limits[2];
  if (const int rc = limits[splits > 1].raise(kern, lds); rc != I8CONV_OK) return rc;
  I8_LAUNCH(kern, dim3(unsigned(tiles), unsigned(splits)), dim3(64 * (WM * WN + NCW)),
                     lds, stream, a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error(std::string("pipelined gemm kernel launch: ") + hipGetErrorString(e));
    return I8CONV_HIP_ERROR;
  }
  return I8CONV_OK;
}

}  // namespace

bool gemm_dma_tile_supported(int bm, int bn) {
  switch (bm * 1000 + bn) {
    case 128064: case 128128: case 256064: case 256128:
      return true;
    default:
      return false;
  }
}

int gemm_dma_copy_waves(const GemmPlan &p) {
  // Copy waves pay off once a workgroup has a steady state to overlap: with
  // two or three k-stages the MFMA waves mostly wait on the first copies
  // anyway, and the split roles only add a barrier hop per stage.
  // The planner picks 256 x 128 only for more than four k-stages.
  const int per_workgroup = p.splits > 1 ? p.stages_per_split : p.stages;
  if (p.wide) return 0;
  if (p.bm == 256 && p.bn == 128) return 8;
  return p.bm == 128 && p.bn == 128 && per_workgroup >= 4 ? 4 : 0;
}

int launch_gemm_dma(const ConvArgs &args, const GemmPlan &p, int splits, void *stream) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  ConvArgs a = args;
  a.m_step = p.m_step > 0 ? p.m_step : p.bm;
  // the kernel's assumptions, checked on the host: whole 128-byte stages in
  // one tap, a stage range per split, a tile it was built for, and LDS rows
  // the ring can hold
  const int stages = a.gemm_k / kStageBytes;
  if (a.c % kStageBytes != 0 || (a.gemm_n > kWideChannels) != p.wide || a.gemm_k % kStageBytes != 0 || stages < 1 ||
      (splits > 1 && (a.stages_per_split < 1 || int64_t(splits - 1) * a.stages_per_split >= stages)) ||
      !gemm_dma_tile_supported(p.bm, p.bn) || a.m_step % 16 != 0 || a.m_step > p.bm ||
      a.m_step < 16 ||
      size_t(kRing) * size_t(p.bm + p.bn) * kStageBytes > size_t(kLdsBudget)) {
    set_error("pipelined gemm plan out of range");
    return I8CONV_BAD_ARGUMENT;
  }
  if (p.wide) {
    if (p.bm == 128 && p.bn == 128)
      return launch_tile<128, 128, 2, 4, 0, true, true>(a, splits, s);
    set_error("unsupported pipelined gemm tile");
    return I8CONV_BAD_ARGUMENT;
  }
  // copy waves on the wide tiles when the workgroup has k-stages enough
  const bool spec = gemm_dma_copy_waves(p) > 0;
  switch (p.bm * 1000 + p.bn) {
    case 128064: return launch_tile<128, 64, 2, 2>(a, splits, s);
    case 128128:
      if (!spec) return launch_tile<128, 128, 2, 4>(a, splits, s);
      // int8: eight MFMA waves of 64 x 32, which share the requantization (7 x
      // 11x14, 512 -> 128 1x1: 6.5 us with four, 6.1 with eight; 4 x 79x79, 256
      // -> 80 1x3, exact multipliers: 8.3 and 7.9)
      if (a.q_y) return launch_tile<128, 128, 2, 4, 4, false>(a, splits, s);
      return launch_tile<128, 128, 2, 2, 4>(a, splits, s);
    case 256064: return launch_tile<256, 64, 4, 2>(a, splits, s);
    case 256128: return launch_tile<256, 128, 4, 2, 8>(a, splits, s);
  }
  set_error("unsupported pipelined gemm tile");
  return I8CONV_BAD_ARGUMENT;
}

}  // namespace i8conv
