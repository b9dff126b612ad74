// The 32-key tile of the MFMA decode kernels (attn_decode.hip and the stream-K
// kernel of attn_rows.hip): its loads, the layout of its V rows in a wave's LDS
// stage, and P V for a tile whose values are not all finite.
#pragma once

#include "device_common.hpp"

namespace mi {
namespace dev {

constexpr int kDecodeTile = 32;  // keys per wave tile

__device__ __forceinline__ uint4 load16_nt(const uint16_t *ptr) {
  typedef unsigned u4_t __attribute__((ext_vector_type(4)));
  const u4_t x = __builtin_nontemporal_load(reinterpret_cast<const u4_t *>(ptr));
  return make_uint4(x.x, x.y, x.z, x.w);
}

// Key of LDS row r of a V tile: k-slot 8 g + i of the PV operand holds key
// 16 (i / 4) + 4 g + i % 4, the keys lane group g holds in the S accumulator.
__device__ __forceinline__ int decode_slot_key(int r) {
  return (((r >> 2) & 1) << 4) | (((r >> 3) & 3) << 2) | (r & 3);
}
// XOR applied to the 32-byte column pair of V row r: the 16 rows of one
// transposed read then fall on 8 distinct bank groups (D = 64: rows are half a
// bank row, so their parity already picks one of two halves).
template <int D>
__device__ __forceinline__ int decode_v_swizzle(int r) {
  return D == 128 ? ((r & 3) | (((r >> 3) & 1) << 2)) : (((r >> 1) & 1) | (((r >> 3) & 1) << 1));
}

// Whether any of a wave's `bytes` of LDS at `lds` (a multiple of 1 KB) is an f16
// infinity or NaN.
template <int BYTES>
__device__ __forceinline__ bool any_not_finite(const uint16_t *lds, int lane) {
  bool bad = false;
#pragma unroll 2
  for (int i = 0; i < BYTES / 1024; ++i) {
    const uint4 v = *reinterpret_cast<const uint4 *>(lds + (64 * i + lane) * 8);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < 4; ++e)
      bad |= (w[e] & 0x7c00u) == 0x7c00u || (w[e] & 0x7c000000u) == 0x7c000000u;
  }
  return __any(bad) != 0;
}

// O^T += V^T P^T for one tile on the vector units: lane (grp, col) adds keys
// 0 .. visible - 1 to its row's d = 16 dt + 4 grp + e. w[hf][e] is the lane's weight
// of key 16 hf + 4 grp + e; `spare` is 2 KB of the wave's own LDS.
template <int D, typename V4>
__device__ __forceinline__ void weigh_tile(V4 *o, const float (&w)[2][4], const uint16_t *stage, uint16_t *spare,
                                           int grp, int col, int visible) {
  float *weights = reinterpret_cast<float *>(spare);
#pragma unroll
  for (int hf = 0; hf < 2; ++hf)
#pragma unroll
    for (int e = 0; e < 4; ++e) weights[(16 * hf + 4 * grp + e) * 16 + col] = w[hf][e];
  // The reads below are of other lanes' stores: in order within the wave.
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll 4
  for (int key = 0; key < kDecodeTile; ++key) {
    const int r = 8 * ((key >> 2) & 3) + 4 * (key >> 4) + (key & 3);
    const float f = weights[key * 16 + col];
    const uint16_t *row = stage + r * D + 8 * (grp >> 1) + 4 * (grp & 1);
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt) {
      uint2 v = *reinterpret_cast<const uint2 *>(row + 16 * (dt ^ decode_v_swizzle<D>(r)));
      if (key >= visible) v = make_uint2(0, 0);
      o[dt][0] = fmaf(f, lo_f16(v.x), o[dt][0]);
      o[dt][1] = fmaf(f, hi_f16(v.x), o[dt][1]);
      o[dt][2] = fmaf(f, lo_f16(v.y), o[dt][2]);
      o[dt][3] = fmaf(f, hi_f16(v.y), o[dt][3]);
    }
  }
}

}  // namespace dev
}  // namespace mi
