// The 32 x 32 x 32 INT8 MFMA's building blocks, shared by the GEMM kernels:
// the LDS row swizzle of its fragments and the stores of its accumulators.
// Pixels are the MFMA's rows (A) and output channels its columns (B): lane
// (q, h) = (lane % 32, lane / 32) holds channel q of the 32 x 32 block's
// pixels 8 g + 4 h + e in element 4 g + e.
#pragma once

#include "i8conv_device.hpp"

namespace i8conv {

#if defined(__HIPCC__)

typedef int v16i __attribute__((ext_vector_type(16)));

__device__ __forceinline__ v16i mfma32(v4i a, v4i b, v16i c) {
  return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
}

// LDS rows of 128 bytes: logical 16-byte chunk j of row r sits at chunk j ^
// swz32_f(r).  A fragment read has lanes 0..31 on 32 consecutive rows of one
// chunk and lanes 32..63 on the next chunk: f takes each of its eight values
// once among the rows that share a position modulo 512 bytes, and four
// consecutive rows differ modulo 128 bytes (the ds_read_b128 rule in
// i8conv_device.hpp).
__device__ __forceinline__ int swz32_f(int row) { return ((row >> 2) + 2 * (row & 3)) & 7; }

// Byte transpose over the four lanes of a quad: lane k ends with byte k of
// lanes 0, 1, 2, 3 of its quad, in that order.
__device__ __forceinline__ uint32_t quad_transpose(uint32_t v, int lane) {
  // across lane bit 0: even lanes keep bytes 0, 2 and take the odd lane's;
  // odd lanes keep bytes 1, 3
  const uint32_t a =
      uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0xb1, 0xf, 0xf, false));  // 1 0 3 2
  v = __builtin_amdgcn_perm(a, v, lane & 1 ? 0x03070105u : 0x06020400u);
  // across lane bit 1, in halfwords
  const uint32_t b =
      uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x4e, 0xf, 0xf, false));  // 2 3 0 1
  return __builtin_amdgcn_perm(b, v, lane & 2 ? 0x03020706u : 0x05040100u);
}

// Stores a wave's FN x FM blocks as int32: rows [0, rows) of a window with
// `n` channels per pixel, px0 the wave's first pixel in it and oc0 its first
// channel.  Each store writes two whole 128-byte pieces of output rows,
// whatever n is.  The window is below 2 GiB.
template <int kPolicy, int FM, int FN>
__device__ __forceinline__ void store_tile32(const v16i (&acc)[FN][FM], __amdgpu_buffer_rsrc_t out,
                                             int rows, int px0, int oc0, int n, int lane) {
  const uint32_t pitch = uint32_t(n) * 4u;
  const int px = px0 + 4 * (lane >> 5), oc = oc0 + (lane & 31);
#pragma unroll
  for (int j = 0; j < FM; ++j)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int p = px + 32 * j + 8 * (e >> 2) + (e & 3);
      const uint32_t off = uint32_t(p) * pitch + uint32_t(oc) * 4u;
#pragma unroll
      for (int i = 0; i < FN; ++i)
        __builtin_amdgcn_raw_buffer_store_b32(
            acc[i][j][e], out, p < rows && oc + 32 * i < n ? off + 128u * i : kOutOfRange, 0,
            kPolicy);
    }
}

// 4 x 4 transpose of dwords over the four lanes of a quad: lane k of the quad
// ends with element k of lanes 0, 1, 2, 3.
__device__ __forceinline__ v4i quad_transpose4(v4i a, int lane) {
  const bool odd = lane & 1, high = lane & 2;
  v4i b, c;
#pragma unroll
  for (int e = 0; e < 4; e += 2) {  // across lane bit 0: quad_perm 1 0 3 2
    const int up = __builtin_amdgcn_update_dpp(0, a[e + 1], 0xb1, 0xf, 0xf, false);
    const int down = __builtin_amdgcn_update_dpp(0, a[e], 0xb1, 0xf, 0xf, false);
    b[e] = odd ? up : a[e];
    b[e + 1] = odd ? a[e + 1] : down;
  }
#pragma unroll
  for (int e = 0; e < 2; ++e) {  // across lane bit 1: quad_perm 2 3 0 1
    const int up = __builtin_amdgcn_update_dpp(0, b[e + 2], 0x4e, 0xf, 0xf, false);
    const int down = __builtin_amdgcn_update_dpp(0, b[e], 0x4e, 0xf, 0xf, false);
    c[e] = high ? up : b[e];
    c[e + 2] = high ? b[e + 2] : down;
  }
  return c;
}

// store_tile32 in 16-byte stores (n % 4 == 0, window 16-byte aligned): a quad's
// transpose gives each lane four channels of one pixel, and a store writes
// eight whole 128-byte pieces.
template <int kPolicy, int FM, int FN>
__device__ __forceinline__ void store_tile32_x4(const v16i (&acc)[FN][FM], __amdgpu_buffer_rsrc_t out,
                                                int rows, int px0, int oc0, int n, int lane) {
  const uint32_t pitch = uint32_t(n) * 4u;
  const int px = px0 + 4 * (lane >> 5) + (lane & 3), oc = oc0 + (lane & 28);
#pragma unroll
  for (int j = 0; j < FM; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int p = px + 32 * j + 8 * g;
      const uint32_t off = uint32_t(p) * pitch + uint32_t(oc) * 4u;
#pragma unroll
      for (int i = 0; i < FN; ++i) {
        const v4i v = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2],
                       acc[i][j][4 * g + 3]};
        __builtin_amdgcn_raw_buffer_store_b128(
            quad_transpose4(v, lane), out,
            p < rows && oc + 32 * i < n ? off + 128u * i : kOutOfRange, 0, kPolicy);
      }
    }
}

// One channel's requantization constants for the blocks of a wave: the
// odd-multiplier form where all of the wave's lanes allow it, else the exact
// one.
struct Requant32 {
  int32_t mult, shift;
  RequantOdd o;
  bool odd;
};
__device__ __forceinline__ Requant32 requant32_params(int32_t mult, int32_t shift, int32_t zp) {
  Requant32 r;
  r.mult = mult;
  r.shift = shift;
  r.o = requant_odd_params(mult, shift, zp);
  r.odd = __builtin_amdgcn_ballot_w64(!r.o.ok) == 0;
  return r;
}

// Four pixels of a lane's channel (a block's elements 4 g ..) requantized to
// int8, the first of them pixel px of the window.  Where n % 4 == 0 and the
// window is 4-byte aligned the lane packs their bytes, and the quad's
// transpose turns them into one pixel's four channels per lane, a 4-byte
// store; a pixel's 32 channels go out as one 32-byte piece.  kBytes (any n,
// any alignment): the same pieces, a byte per lane and store.
//
// `base` is the byte of the lane's first store at px == 0 (quad_int8_base),
// out of range for channels past n; pixels past the window's last row fall out
// of its bounds by themselves, so a store costs one add instead of a
// multiplication and two compares.
template <bool kBytes>
__device__ __forceinline__ uint32_t quad_int8_base(int oc0, int n, int lane) {
  const int px = 4 * (lane >> 5) + (kBytes ? 0 : lane & 3);
  const int oc = oc0 + (lane & (kBytes ? 31 : 28));
  return oc < n ? uint32_t(px) * uint32_t(n) + uint32_t(oc) : kOutOfRange;
}
template <bool kBytes, bool kOdd>
__device__ __forceinline__ void store_quad_int8(v4i acc, const Requant32 &r, int32_t zp,
                                                __amdgpu_buffer_rsrc_t out, uint32_t base, int px,
                                                int n, int lane) {
  uint32_t y[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    y[e] = uint32_t(kOdd ? requant1_odd(acc[e], r.o.mo, r.o.k, r.o.sh)
                         : requant1(acc[e], r.mult, r.shift, zp));
  }
  const uint32_t off = base + uint32_t(px) * uint32_t(n);
  if constexpr (kBytes) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      __builtin_amdgcn_raw_buffer_store_b8(uint8_t(y[e]), out, off + uint32_t(e) * uint32_t(n), 0, 0);
    return;
  }
  const uint32_t lo = __builtin_amdgcn_perm(y[1], y[0], 0x0c0c0400u);
  const uint32_t hi = __builtin_amdgcn_perm(y[3], y[2], 0x0c0c0400u);
  const uint32_t v = quad_transpose(__builtin_amdgcn_perm(hi, lo, 0x05040100u), lane);
  __builtin_amdgcn_raw_buffer_store_b32(v, out, off, 0, 0);
}

// One 32 x 32 block of a wave requantized to int8, px0 its first pixel.
template <bool kBytes, bool kOdd>
__device__ __forceinline__ void store_block32_int8(const v16i &acc, const Requant32 &r, int32_t zp,
                                                   __amdgpu_buffer_rsrc_t out, uint32_t base,
                                                   int px0, int n, int lane) {
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const v4i v = {acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
    store_quad_int8<kBytes, kOdd>(v, r, zp, out, base, px0 + 8 * g, n, lane);
  }
}

// The odd-multiplier form and the exact one apart, chosen once per block: the
// first is then short straight-line code and the exact form's 64-bit products
// lie out of its way.  With both in the code of every four values, fetching
// that code, once per launch, took a microsecond (us per launch of the
// pipelined GEMM: its 16 x 16 MFMA form, this one with both together, apart;
// 4 x 79x79, 256 -> 96 1x3: 7.8, 8.7, 6.7; 7 x 11x14, 512 -> 128 1x1: 6.9, 8.7,
// 6.1; 4 x 52x52, 256 -> 72: 5.5, 6.3, 5.2; exact form, 16 x 28x28, 512 -> 384:
// 14.6, 20.4, 12.7).  Chosen for a wave's blocks of 32 channels together the
// exact form spills where four waves share a SIMD (256 x 128 tile, 8 x 64x64,
// 256 -> 256: 25.3, 28.3 so).
template <bool kBytes>
__device__ __forceinline__ void requant_block32(const v16i &acc, const Requant32 &r, int32_t zp,
                                                __amdgpu_buffer_rsrc_t out, uint32_t base, int px0,
                                                int n, int lane) {
  if (__builtin_expect(r.odd, 1))
    store_block32_int8<kBytes, true>(acc, r, zp, out, base, px0, n, lane);
  else
    store_block32_int8<kBytes, false>(acc, r, zp, out, base, px0, n, lane);
}

#endif  // __HIPCC__

}  // namespace i8conv
