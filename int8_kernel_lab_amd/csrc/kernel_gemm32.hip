// Generic implicit GEMM on the 32 x 32 x 32 INT8 MFMA, for any input channel
// count (C % 16 == 0): the generic kernel's form for layers whose channels
// are no multiple of 128, for small grids of strided and 1x1 layers, and for
// the largest ones (plan_generic in shape.cpp has the rule and both sides'
// figures).  Same GEMM view as kernel_gemm_dma.hip (M = n*out_h*out_w pixels,
// N output channels, k = (fy*s + fx)*c + ci); what it does differently:
//   * pixels are the MFMA's rows and output channels its columns, so a lane
//     holds one channel of sixteen pixels and every 4-byte store of a wave
//     writes two whole 128-byte pieces of output rows, whatever N is.  With
//     the roles the other way round a 16-byte store scatters 32-byte pieces
//     over 32 pixels: 128 x 128 x 8 images, 64 -> 128 channels, 1x3: 28.1
//     against 15.1 us; 256 x 256, 64 -> 255 channels, 3x3: 43 us with the
//     element stores of the 16 x 16 forms, 23 us here;
//   * v_mfma_i32_32x32x32 does the operations of two 16 x 16 x 64 with half
//     the operand reads, and one wave per SIMD reaches with it what the power
//     allows: random operands, all SIMDs busy for 5 ms, 3.5 POP/s (4.95 with
//     constant ones, the full clock); 16 x 16 x 64 with 16 accumulators 2.9, 3.5
//     only with two waves per SIMD;
//   * k-stages of 128 bytes per row come by LDS-DMA (two stage buffers, one
//     barrier per stage).  A 128-byte row is a whole L2 line: the same copies
//     in 64-byte halves land at 70 instead of 130 GB/s per compute unit;
//   * with kLaneTap each lane decomposes its own 16-byte chunk's k into tap
//     and channel, so a stage may span taps (C % 128 != 0); otherwise a stage
//     lies inside one tap and the channel chunk is the outer loop, the taps
//     the inner one;
//   * workgroups are persistent: the next tile's first stages are copied
//     before the tile's stores go out.  Small tiles share a compute unit two
//     to four at a time, which hides their copy issue and LDS latency better
//     than more than two stage buffers did (4, 6 and 9 within 8 %);
//   * int8 output: each lane requantizes its channel (parameters read once
//     per tile), and the four lanes of a quad turn their bytes into one
//     pixel's four channels per lane; other channel counts and alignments
//     store single bytes, a pixel's 32 channels side by side (4 x 94x94, 256 ->
//     269 1x1: 16.1 us; int32 and a pass over it, 46.9).
#include <hip/hip_runtime.h>

#include <limits.h>

#include <algorithm>
#include <string>
#include <type_traits>

#include "i8conv_internal.hpp"
#include "mfma32_tile.hpp"

namespace i8conv {
namespace {

template <int N>
using Set = std::integral_constant<int, N>;

constexpr int kStageBuffers = 2;  // per group of waves

// What the epilogue writes: int32, or requantized int8 in 4-byte stores (N % 4
// == 0, output 4-byte aligned) or byte stores (any N).
enum OutKind { kOutInt32, kOutInt8, kOutInt8Bytes };

template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ void barrier_lds() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// BM pixels x BN channels over WM x WN waves; KG groups of such waves, each
// with stage buffers of its own, take the k-stages in turn (group g the
// stages g, g + KG, ...) and add their sums up through LDS at the end;
// fragments read GS k-steps of 32 bytes at a time; kOcc waves per SIMD.
template <int BM, int BN, int WM, int WN, int KG, int GS, bool kLaneTap, int kOut, int kPolicy,
          int kOcc>
__global__ __launch_bounds__(64 * WM * WN * KG, kOcc) void gemm32_kernel(ConvArgs a, int tiles) {
  constexpr int P = kStageBytes;             // bytes per LDS row: one k-stage
  constexpr int R = kStageBuffers;
  constexpr int KS = P / 32;                 // k-steps per stage
  constexpr int kWaves = WM * WN;
  constexpr int TM = BM / WM, TN = BN / WN;  // pixels and channels per wave
  constexpr int FM = TM / 32, FN = TN / 32;  // 32 x 32 blocks per wave
  constexpr int kTile = (BM + BN) * P;    // bytes per stage buffer
  constexpr int RPC = 1024 / P;           // rows per 1 KB copy
  constexpr int CPW = (BM + BN) / RPC / kWaves;  // copies per wave and stage
  constexpr int CPA = BN / RPC / kWaves;         // of which filter rows
  constexpr int CPB = CPW - CPA;
  constexpr bool kByte = kOut != kOutInt32;
  constexpr int kParams = kByte ? 3 : 1;  // bias, multipliers, shifts
  constexpr int kParamBytes = kParams * BN * 4;
  constexpr int ST = FM * FN * (kOut == kOutInt8 ? 4 : 16);  // stores per wave and tile
  static_assert(CPA >= 1 && CPB >= 1 && BN % (RPC * kWaves) == 0, "tile shape");
  static_assert(KG == 1 || (kLaneTap && FM == 1 && FN == 1 && 4 % KG == 0), "k groups");
  extern __shared__ __attribute__((aligned(16))) int8_t smem[];

  const int lane = threadIdx.x & 63;
  const int wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = wave_id / kWaves, wave = wave_id % kWaves;
  const int wm = wave % WM, wn = wave / WM;
  const v4u xd = make_desc(a.x, a.x_bytes);
  const v4u wd = make_desc(a.w, a.w_bytes);
  int8_t *const bufs = smem + group * R * kTile;  // this group's stage buffers
  const uint32_t lds0 = lds_addr(bufs);
  int8_t *const params = smem + KG * R * kTile;
  const uint32_t lds_params = lds_addr(params);
  // stages per group (the last ones may lie past the reduction: zeros)
  const int stages = (a.gemm_k + KG * P - 1) / (KG * P);
  const int tiles_n = (a.gemm_n + BN - 1) / BN;

  // this lane's chunk of every row it copies, and its row within a copy
  const int crow = lane / (P / 16);
  const int lk = 16 * ((lane % (P / 16)) ^ swz32_f(wave * RPC + crow));

  uint32_t abase[CPA];
  int pix[CPB], iy0[CPB], ix0[CPB];
  int tile_m = 0, tile_n = 0, m_end = 0;

  auto setup = [&](int t) {
    tile_m = (t / tiles_n) * a.m_step;
    tile_n = (t % tiles_n) * BN;
    m_end = min(a.gemm_m, tile_m + a.m_step);
#pragma unroll
    for (int j = 0; j < CPA; ++j) {
      const int oc = tile_n + (wave + kWaves * j) * RPC + crow;
      abase[j] = oc < a.gemm_n ? uint32_t(oc) * uint32_t(a.gemm_k) + uint32_t(lk) : kOutOfRange;
    }
#pragma unroll
    for (int j = 0; j < CPB; ++j) {
      const int m = tile_m + (wave + kWaves * j) * RPC + crow;
      if (m < m_end) {
        const int b = int(fast_div(uint32_t(m), a.div_ohw));
        const int rem = m - b * a.out_h * a.out_w;
        const int oy = int(fast_div(uint32_t(rem), a.div_ow));
        const int ox = rem - oy * a.out_w;
        iy0[j] = oy * a.stride_h - a.pad_h;
        ix0[j] = ox * a.stride_w - a.pad_w;
        pix[j] = ((b * a.h + iy0[j]) * a.wd + ix0[j]) * a.c + (kLaneTap ? 0 : lk);
      } else {
        iy0[j] = -(1 << 29);
        ix0[j] = 0;
        pix[j] = 0;
      }
    }
  };

  // The k-stages of a tile in order, one tap() per stage.  Where a stage
  // lies inside one tap (C % P == 0) the channel chunk is the outer loop and
  // the filter taps the inner ones.
  struct StageTap {
    int dy, dx, off, k0;
    bool live;
  };
  int next_fy = 0, next_fx = 0, next_ci = 0, next_k = 0;
  const int row_step = a.dil_h * a.wd * a.c, col_step = a.dil_w * a.c;
  // kLaneTap: this lane's chunk moves on by 128 KG bytes per stage, that is by
  // `d` taps and channels plus at most one carry of each, in full-rate adds
  // and selects (dividing by C and S anew each stage took a third of the
  // issue slots of the small tiles: 16 x 224x224, 32 -> 64 7x7 stride 2)
  const int d_tap = int(fast_div(uint32_t(KG * P), a.div_c)), d_ci = KG * P - d_tap * a.c;
  const int d_fy = int(fast_div(uint32_t(d_tap), a.div_s)), d_fx = d_tap - d_fy * a.s;
  const int d_off = d_fy * row_step + d_fx * col_step + d_ci;
  const int wrap_dx = a.s * a.dil_w, wrap_off = row_step - a.s * col_step;
  const int k0 = group * P + lk;
  const int tap0 = int(fast_div(uint32_t(k0), a.div_c)), ci0 = k0 - tap0 * a.c;
  const int fy0 = int(fast_div(uint32_t(tap0), a.div_s)), fx0 = tap0 - fy0 * a.s;
  int lane_ci = 0, lane_dx = 0, lane_dy = 0, lane_off = 0;
  auto restart = [&]() {
    next_fy = next_fx = next_ci = 0;
    next_k = group * P;
    if constexpr (kLaneTap) {
      lane_ci = ci0;
      lane_dx = fx0 * a.dil_w;
      lane_dy = fy0 * a.dil_h;
      lane_off = fy0 * row_step + fx0 * col_step + ci0;
    }
  };
  auto stage_tap = [&]() {
    StageTap t;
    if constexpr (kLaneTap) {
      t.k0 = next_k;
      t.live = lk < a.gemm_k - next_k;
      t.dy = t.live ? lane_dy : -(1 << 29);
      t.dx = lane_dx;
      t.off = lane_off;
      next_k += KG * P;
      lane_ci += d_ci;
      const bool carry = lane_ci >= a.c;
      lane_ci -= carry ? a.c : 0;
      lane_dx += d_fx * a.dil_w + (carry ? a.dil_w : 0);
      const bool wrap = lane_dx >= wrap_dx;
      lane_dx -= wrap ? wrap_dx : 0;
      lane_dy += d_fy * a.dil_h + (wrap ? a.dil_h : 0);
      lane_off += d_off + (carry ? col_step - a.c : 0) + (wrap ? wrap_off : 0);
    } else {
      t.live = true;
      t.k0 = (next_fy * a.s + next_fx) * a.c + next_ci;
      t.dy = next_fy * a.dil_h;
      t.dx = next_fx * a.dil_w;
      t.off = (t.dy * a.wd + t.dx) * a.c + next_ci;
      if (++next_fx == a.s) {
        next_fx = 0;
        if (++next_fy == a.r) {
          next_fy = 0;
          next_ci += P;
        }
      }
    }
    return t;
  };
  auto copy = [&](const StageTap &t, uint32_t buf, int j) {
    if (j < CPA) {
      const uint32_t off = abase[j] + uint32_t(t.k0);
      lds_copy16(wd, buf + uint32_t(wave + kWaves * j) * 1024u, t.live ? off : kOutOfRange);
    } else {
      const int b = j - CPA;
      const bool ok = unsigned(iy0[b] + t.dy) < unsigned(a.h) && unsigned(ix0[b] + t.dx) < unsigned(a.wd);
      lds_copy16(xd, buf + uint32_t(wave + kWaves * j) * 1024u,
                 ok ? uint32_t(pix[b] + t.off) : kOutOfRange);
    }
  };
  // per-channel parameters of the tile at tile_n into parameter slot `slot`
  auto copy_params = [&](int slot) {
    if (wave_id * 64 + lane < BN) {
      const uint32_t bytes = uint32_t(a.gemm_n) * 4u;
      const uint32_t off = uint32_t(tile_n + wave_id * 64 + lane) * 4u;
      const uint32_t dst = lds_params + uint32_t(slot * kParamBytes) + uint32_t(wave_id) * 256u;
      lds_copy4(make_desc(a.bias, bytes), dst, off);
      if constexpr (kByte) {
        lds_copy4(make_desc(a.q_mult, bytes), dst + BN * 4u, off);
        lds_copy4(make_desc(a.q_shift, bytes), dst + BN * 8u, off);
      }
    }
  };
  auto prologue = [&](int slot) {
    copy_params(slot);
    restart();
#pragma unroll
    for (int s = 0; s < R; ++s) {
      if (s >= stages) break;
      const StageTap t = stage_tap();
#pragma unroll
      for (int j = 0; j < CPW; ++j) copy(t, lds0 + uint32_t(s * kTile), j);
    }
  };

  const TileRun run = xcd_tile_run(tiles, int(gridDim.x), int(blockIdx.x));
  int t = run.first;
  if (t >= run.last) return;

  // fragment read offsets in a stage buffer: row 32 i + lane % 32 of the
  // wave's filter (or pixel) rows, chunk 2 ks + lane / 32
  const int frow = lane & 31;
  const int ff = swz32_f(frow);
  int koff[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) koff[ks] = frow * P + 16 * ((2 * ks + (lane >> 5)) ^ ff);
  const int abuf = wn * TN * P, bbuf = (BN + wm * TM) * P;

  setup(t);
  int slot = 0;
  bool pend = false;  // ST stores of the previous tile follow the prologue's copies
  prologue(slot);
  for (;;) {
    // the first stage has landed
    if (pend)
      wait_vm<(ST < 63 ? ST : 63)>();
    else if (stages > 1)
      wait_vm<CPW>();
    else
      wait_vm<0>();
    barrier_lds();

    v16i acc[FN][FM];
    const int8_t *const pr = params + slot * kParamBytes;
#pragma unroll
    for (int i = 0; i < FN; ++i) {
      const int v = group > 0 ? 0 : *reinterpret_cast<const int *>(
          pr + (wn * TN + 32 * i + (lane & 31)) * 4);
      v16i c;
#pragma unroll
      for (int e = 0; e < 16; ++e) c[e] = v;
#pragma unroll
      for (int j = 0; j < FM; ++j) acc[i][j] = c;
    }
    // Fragments of GS k-steps, two sets: one feeds the MFMAs while the other
    // is read.
    constexpr int NP = KS / GS;  // sets per stage
    v4i fa[2][GS][FN], fb[2][GS][FM];
    auto read = [&](auto set, const int8_t *buf, int part, int q) {
      const int ks = q / (FN + FM), n = q % (FN + FM);
      const int8_t *const p = buf + koff[part * GS + ks];
      if (n < FN)
        fa[set.value][ks][n] = *reinterpret_cast<const v4i *>(p + abuf + 32 * P * n);
      else
        fb[set.value][ks][n - FN] = *reinterpret_cast<const v4i *>(p + bbuf + 32 * P * (n - FN));
    };
    constexpr int kMfma = GS * FN * FM;
    constexpr int kReads = GS * (FN + FM);
#pragma unroll
    for (int q = 0; q < kReads; ++q) read(Set<0>{}, bufs, 0, q);

    int ring = 0;
    auto stage = [&](int s) {
      const int next = ring + 1 == R ? 0 : ring + 1;
      const int8_t *const buf = bufs + ring * kTile;
      const int8_t *const nbuf = bufs + next * kTile;
      const bool more = s + R < stages;
      StageTap tap{};
      if (more) tap = stage_tap();
      auto part = [&](auto set, auto last, int pt) {
        if (last.value) {
          // every wave has read all of stage s, and stage s + 1 has landed
          if (s + 1 < stages && !(pend && s + 1 < R)) wait_vm<0>();
          barrier_lds();
        }
#pragma unroll
        for (int n = 0; n < kMfma; ++n) {
#pragma unroll
          for (int q = n * kReads / kMfma; q < (n + 1) * kReads / kMfma; ++q)
            read(Set<1 - set.value>{}, last.value ? nbuf : buf, last.value ? 0 : pt + 1, q);
          if (last.value && more) {
#pragma unroll
            for (int q = n * CPW / kMfma; q < (n + 1) * CPW / kMfma; ++q)
              copy(tap, lds0 + uint32_t(ring * kTile), q);
          }
          const int ks = n / (FN * FM), i = n / FM % FN, j = n % FM;
          acc[i][j] = mfma32(fb[set.value][ks][j], fa[set.value][ks][i], acc[i][j]);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      static_assert(NP == 2 || NP == 4, "an even number of sets per stage");
      part(Set<0>{}, std::false_type{}, 0);
      if constexpr (NP == 4) {
        part(Set<1>{}, std::false_type{}, 1);
        part(Set<0>{}, std::false_type{}, 2);
      }
      part(Set<1>{}, std::true_type{}, NP - 1);
      ring = next;
    };
    for (int s = 0; s < stages; ++s) stage(s);

    const int out_m = tile_m, out_n = tile_n, out_end = m_end;
    t += run.step;
    const bool again = t < run.last;
    if constexpr (KG > 1) {
      // each wave's sums go to its 4 KB of the first stage buffers (every
      // wave has read its last stage), four elements per 1 KB; then group g
      // adds up and stores the elements of quads g, g + KG, ...
      const int rows = out_end - out_m;
      const int px0 = wm * TM + 4 * (lane >> 5), oc0 = out_n + wn * TN;
      auto part_of = [&](int grp, int q) {
        return reinterpret_cast<v4i *>(smem + grp * R * kTile + wave * 4096 + q * 1024 + lane * 16);
      };
      static_assert(kWaves * 4096 <= R * kTile, "sums fit the stage buffers");
      barrier_lds();
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *part_of(group, q) = v4i{acc[0][0][4 * q], acc[0][0][4 * q + 1], acc[0][0][4 * q + 2],
                                 acc[0][0][4 * q + 3]};
      barrier_lds();
      const int8_t *const pq = pr + (wn * TN + (lane & 31)) * 4;
      Requant32 r{};
      if constexpr (kByte)
        r = requant32_params(*reinterpret_cast<const int *>(pq + BN * 4),
                             *reinterpret_cast<const int *>(pq + BN * 8), a.q_zp);
      const uint32_t base = quad_int8_base<kOut == kOutInt8Bytes>(oc0, a.gemm_n, lane);
#pragma unroll
      for (int u = 0; u < 4 / KG; ++u) {
        const int q = group + KG * u;
        v4u sum = *reinterpret_cast<const v4u *>(part_of(0, q));
#pragma unroll
        for (int g = 1; g < KG; ++g) sum += *reinterpret_cast<const v4u *>(part_of(g, q));
        const v4i v = __builtin_bit_cast(v4i, sum);
        if constexpr (kByte) {
          const auto yr = make_rsrc(a.q_y + size_t(out_m) * size_t(a.gemm_n),
                                    uint32_t(rows) * uint32_t(a.gemm_n));
          if (__builtin_expect(r.odd, 1))
            store_quad_int8<kOut == kOutInt8Bytes, true>(v, r, a.q_zp, yr, base, wm * TM + 8 * q,
                                                         a.gemm_n, lane);
          else
            store_quad_int8<kOut == kOutInt8Bytes, false>(v, r, a.q_zp, yr, base, wm * TM + 8 * q,
                                                          a.gemm_n, lane);
        } else {
          const auto yr = make_rsrc(a.y + size_t(out_m) * size_t(a.gemm_n),
                                    uint32_t(rows) * uint32_t(a.gemm_n) * 4u);
          const int oc = oc0 + (lane & 31);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int px = px0 + 8 * q + e;
            __builtin_amdgcn_raw_buffer_store_b32(
                v[e], yr,
                px < rows && oc < a.gemm_n
                    ? (uint32_t(px) * uint32_t(a.gemm_n) + uint32_t(oc)) * 4u : kOutOfRange,
                0, kPolicy);
          }
        }
      }
      if (!again) return;
      barrier_lds();
      setup(t);
      slot ^= 1;
      prologue(slot);
      continue;
    }
    // the next tile's copies go out before this tile's stores
    if (again) {
      setup(t);
      prologue(slot ^ 1);
    }
    const int rows = out_end - out_m;
    const int px0 = wm * TM, oc0 = out_n + wn * TN;
    if constexpr (!kByte) {
      const auto yr = make_rsrc(a.y + size_t(out_m) * size_t(a.gemm_n),
                                uint32_t(rows) * uint32_t(a.gemm_n) * 4u);
      store_tile32<kPolicy>(acc, yr, rows, px0, oc0, a.gemm_n, lane);
    } else {
      const auto yr = make_rsrc(a.q_y + size_t(out_m) * size_t(a.gemm_n),
                                uint32_t(rows) * uint32_t(a.gemm_n));
#pragma unroll
      for (int i = 0; i < FN; ++i) {
        const int8_t *const pq = pr + (wn * TN + 32 * i + (lane & 31)) * 4;
        const Requant32 r = requant32_params(*reinterpret_cast<const int *>(pq + BN * 4),
                                             *reinterpret_cast<const int *>(pq + BN * 8), a.q_zp);
        const uint32_t base = quad_int8_base<kOut == kOutInt8Bytes>(oc0 + 32 * i, a.gemm_n, lane);
#pragma unroll
        for (int j = 0; j < FM; ++j)
          requant_block32<kOut == kOutInt8Bytes>(acc[i][j], r, a.q_zp, yr, base, px0 + 32 * j,
                                                 a.gemm_n, lane);
      }
    }
    if (!again) return;
    slot ^= 1;
    pend = true;
  }
}

template <int BM, int BN, int WM, int WN, int KG, int GS, bool kLaneTap, int kOcc, int kGroups,
          int kOut, int kPolicy>
int launch_tile(const ConvArgs &a, hipStream_t stream) {
  auto kern = gemm32_kernel<BM, BN, WM, WN, KG, GS, kLaneTap, kOut, kPolicy, kOcc>;
  const size_t lds =
      size_t(KG) * kStageBuffers * (BM + BN) * kStageBytes + 2 * (kOut == kOutInt32 ? 1 : 3) * BN * 4;
  const int tiles = int(((int64_t(a.gemm_m) + BM - 1) / BM) * ((a.gemm_n + BN - 1) / BN));
  static LdsLimit limit;
  if (const int rc = limit.raise(kern, lds); rc != I8CONV_OK) return rc;
  I8_LAUNCH(kern, dim3(unsigned(std::min(tiles, 256 * kGroups))), dim3(64 * WM * WN * KG),
            lds, stream, a, tiles);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error(std::string("gemm32 kernel launch: ") + hipGetErrorString(e));
    return I8CONV_HIP_ERROR;
  }
  return I8CONV_OK;
}

// The cache policies of kernel_gemm_dma.hip: int32 write-through where the
// pixel pitch keeps sectors whole and the output is at most 128 MiB,
// evict-first above, ordinary for other pitches and for int8.
template <int BM, int BN, int WM, int WN, int KG, int GS, bool kLaneTap, int kOcc, int kGroups>
int launch_out(const ConvArgs &a, hipStream_t s) {
  if (a.q_y && a.gemm_n % 4 == 0 && (reinterpret_cast<uintptr_t>(a.q_y) & 3) == 0)
    return launch_tile<BM, BN, WM, WN, KG, GS, kLaneTap, kOcc, kGroups, kOutInt8, 0>(a, s);
  if (a.q_y)
    return launch_tile<BM, BN, WM, WN, KG, GS, kLaneTap, kOcc, kGroups, kOutInt8Bytes, 0>(a, s);
  if (a.gemm_n % 8 != 0)
    return launch_tile<BM, BN, WM, WN, KG, GS, kLaneTap, kOcc, kGroups, kOutInt32, 0>(a, s);
  if (int64_t(a.gemm_m) * a.gemm_n * 4 > kStreamOutputBytes)
    return launch_tile<BM, BN, WM, WN, KG, GS, kLaneTap, kOcc, kGroups, kOutInt32, kStoreStream>(a, s);
  return launch_tile<BM, BN, WM, WN, KG, GS, kLaneTap, kOcc, kGroups, kOutInt32, kStoreThrough>(a, s);
}

}  // namespace

bool gemm32_eligible(const i8conv_shape &s, const i8conv_geometry &g) {
  // 32-bit tile, tap and k arithmetic, and a tile's output window below 2 GiB
  return int64_t(s.r) * s.dilation_h <= (1 << 28) && int64_t(s.s) * s.dilation_w <= (1 << 28) &&
         g.gemm_m <= (1 << 30) && g.gemm_k <= (1 << 30) && g.gemm_n <= kWideChannels &&
         ((g.gemm_m + 63) / 64) * ((int64_t(g.gemm_n) + 63) / 64) <= INT32_MAX;
}

int launch_gemm32(const ConvArgs &args, const GemmPlan &p, void *stream) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  ConvArgs a = args;
  a.m_step = p.bm;
  switch (p.bm * 1000 + p.bn) {
    case 64064:
      if (p.kg == 4) return launch_out<64, 64, 2, 2, 4, 2, true, 4, 1>(a, s);
      if (p.kg == 2) return launch_out<64, 64, 2, 2, 2, 2, true, 4, 2>(a, s);
      return launch_out<64, 64, 2, 2, 1, 2, true, 4, 4>(a, s);
    case 128032: return launch_out<128, 32, 4, 1, 1, 1, true, 3, 3>(a, s);
    case 128064: return launch_out<128, 64, 2, 2, 1, 1, true, 3, 3>(a, s);
    // four waves of 64 x 64: eight of 32 x 64 spill at four waves per SIMD (7 x
    // 196x196, 80 -> 209 1x3: 72 us, 48 with four; 256x256, 64 -> 255: 23.6, 21)
    case 128128: return launch_out<128, 128, 2, 2, 1, 1, true, 2, 2>(a, s);
    case 256256:
      // a stage lies inside one tap
      if (a.c % kStageBytes == 0) return launch_out<256, 256, 4, 2, 1, 1, false, 2, 1>(a, s);
      break;
  }
  set_error("gemm32: unsupported tile " + std::to_string(p.bm) + "x" + std::to_string(p.bn));
  return I8CONV_BAD_ARGUMENT;
}

}  // namespace i8conv
