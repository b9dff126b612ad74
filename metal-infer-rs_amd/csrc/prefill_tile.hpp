// LDS layouts of the 64-key tiles that the prefill and the tiled attention
// kernels load directly from global memory (D = 64, 128), and of their output
// rows.
#pragma once

#include "device_common.hpp"

namespace mi {
namespace dev {

// Direct-load tile layout (D = 64, 128): a tile row of D halves is 2D bytes
// in 16-byte chunks, the chunks of row r XOR-swizzled so that the K operand
// reads (16 rows, one chunk each) and the V^T transpose reads (four rows,
// eight bytes per lane) of 16 / 32 lanes fall on distinct banks. D = 128
// (256-byte rows span the 64 banks): K chunk ^ (r & 15), V chunk ^ 4 (r & 3).
// D = 64 (128-byte rows, two per bank row): rows 2m and 2m + 1 already sit
// in opposite bank halves, so K uses chunk ^ ((r >> 1) & 7) and V
// chunk ^ 4 ((r >> 1) & 1).
template <int D>
__device__ __forceinline__ int k_swizzle(int r) {
  return D == 128 ? (r & 15) : ((r >> 1) & 7);
}
template <int D>
__device__ __forceinline__ int v_swizzle(int r) {
  return D == 128 ? ((r & 3) << 2) : (((r >> 1) & 1) << 2);
}

// Output staging (the rows of one wave as f16 in LDS): 16-byte chunk c of
// row r sits at chunk c ^ out_swizzle(r), so that the writes (one chunk of
// 32 rows per instruction) and the reads (whole rows) spread over the banks.
template <int D>
__device__ __forceinline__ int out_swizzle(int r) {
  constexpr int CPR = D / 8, RB = D >= 128 ? 1 : 128 / D;  // rows per 256 bytes
  return (r / RB) & (CPR - 1);
}

}  // namespace dev
}  // namespace mi
