// o_proj of a short prompt, a chunk or a turn (33 to some thousand rows of x):
// out[m, n] = x[m, k] . w[n, k]^T, f16 in and out, f32 sums on MFMA, one output
// tile per CU.
//
// What bounds it: at these sizes one round of tiles is the whole launch, so the
// time is one workgroup's walk along k, its loads per step: 45 to 60 bytes per ns
// and CU in the traces, with two or more stages in flight. Whether that is the L2's
// rate or its latency under load is not told apart. So the k steps run through a ring
// of LDS stages filled by direct loads (96 to 147 KB), and the tile is the one
// with the least rows of x and w that still fits all tiles on the chip at once.
// Measured on MI355X (graph replays over rotated weights, hipBLASLt -> this):
// [128, 2048] x [1024, 2048]^T 8.4 -> 6.4 us, 48 x [1024, 1024] 8.1 -> 4.7, 100 x
// [2048, 2048] 8.4 -> 6.4, 1100 x [2048, 2048] 18.6 -> 16.8, 2048 x [1024, 2048]
// 14.7 -> 13.4, 256 x [5120, 8192] 72 -> 49.
//  - 8 waves: two groups of 2 x 2. Each group multiplies half of every step's
//    keys for the whole tile (two waves per SIMD hide each other's LDS reads at
//    the LDS traffic of 2 x 2), and the second group's sums are added through LDS.
//  - An LDS row is one row's BK halves; 16-byte piece c of row r lies at
//    c ^ swizzle(r), so the 16 rows of an operand read fall on all banks.
//  - Consecutive workgroups go to different XCDs, so tiles are dealt in
//    runs per XCD, up to 8 row tiles of a column first: an XCD's tiles share
//    x and weight rows in its L2 (2048 x [1024, 2048]: 16.2 us with 16 row tiles
//    first, 14.6 with 8).
//  - 128 keys per step where three stages fit, else 64 (128 x 64 tiles, six stages
//    of 64 -> three of 128 keys: 512 x [4096, 2048] 17.7 -> 17.0 us).
#include "device_common.hpp"
#include "kernels.hpp"

namespace mi {
namespace kernels {
namespace {

using namespace mi::dev;

typedef float f4_t __attribute__((ext_vector_type(4)));

constexpr uint32_t kXcds = 8;
constexpr uint32_t kBand = 8;  // row tiles walked together

// s_waitcnt: at most `vm` vector-memory accesses of the wave outstanding, and
// every LDS read returned (the stage it came from is overwritten next).
constexpr int wait_stage(int vm) { return (vm & 15) | ((vm >> 4) << 14) | 0x70; }

template <int BM, int BN, int BK, int S>
__global__ __launch_bounds__(512, 2) void gemm_tile_kernel(const MatvecParams p, uint32_t row_tiles,
                                                           uint32_t col_tiles) {
  constexpr int MT = BM / 32, NT = BN / 32;             // 16 x 16 blocks of a wave's tile
  constexpr int CPR = BK / 8, STAGE = (BM + BN) * BK;   // 16-byte pieces per row, halves per stage
  constexpr int LPW = STAGE / 512 / 8;                  // 1 KB loads per wave and stage
  constexpr int STEPS = BK / 64;                        // MFMA key steps per group and stage
  static_assert(STAGE % 4096 == 0 && S >= 3 && S <= 6 && (S - 2) * LPW < 64);
  static_assert(4 * 64 * ((MT * NT + 1) / 2) * 8 <= STAGE, "half the second group's sums fit a stage");
  __shared__ __attribute__((aligned(16))) uint16_t s0[STAGE], s1[STAGE], s2[STAGE],
      s3[S > 3 ? STAGE : 8], s4[S > 4 ? STAGE : 8], s5[S > 5 ? STAGE : 8];
  const uint32_t tile = (blockIdx.x % kXcds) * (gridDim.x / kXcds) + blockIdx.x / kXcds;
  if (tile >= row_tiles * col_tiles) return;
  const uint32_t band = tile / (kBand * col_tiles), in_band = tile % (kBand * col_tiles);
  const uint32_t band_rows = min(kBand, row_tiles - band * kBand);
  const uint32_t m0 = (band * kBand + in_band % band_rows) * BM, n0 = in_band / band_rows * BN;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int group = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
  const int r = lane & 15, kg = lane >> 4;
  auto swizzle = [](int row) { return BK == 128 ? row & 15 : (row >> 1) & 7; };
  // Stage rows: BM of x, then BN of w; rows past the last re-read it and are
  // not stored.
  const uint16_t *src[LPW];
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    const int row = (64 * (wave * LPW + i) + lane) / CPR;
    const int piece = (lane % CPR) ^ swizzle(row);
    src[i] = row < BM ? p.x + (int64_t)min(m0 + row, p.m - 1) * p.x_row + 8 * piece
                      : p.w + (int64_t)min(n0 + (row - BM), p.n - 1) * p.w_row + 8 * piece;
  }
  // Past the last step every lane loads the same 16 bytes, never read: without a
  // branch around the loads the compiler's own waits agree with the ones below.
  const uint32_t steps = p.k / BK;
  auto issue = [&](uint32_t t, uint16_t *stage) __attribute__((always_inline)) {
    const bool more = t < steps;
#pragma unroll
    for (int i = 0; i < LPW; ++i)
      load_lds16(more ? src[i] + (size_t)t * BK : p.x, stage + (wave * LPW + i) * 512);
  };
  // Operands: lane (kg, r) takes piece 4 s + kg of row r of a block; 16 rows on,
  // the swizzle is the same.
  int xat[STEPS], wat[STEPS];
#pragma unroll
  for (int s = 0; s < STEPS; ++s) {
    const int piece = ((4 * (group * STEPS + s) + kg) ^ swizzle(r)) * 8;
    xat[s] = (wm * (BM / 2) + r) * BK + piece;
    wat[s] = (BM + wn * (BN / 2) + r) * BK + piece;
  }
  f4_t acc[NT][MT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[j][i] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
  auto compute = [&](const uint16_t *stage) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      h8_t xv[MT], wv[NT];
#pragma unroll
      for (int i = 0; i < MT; ++i)
        xv[i] = as_h8(*reinterpret_cast<const uint4 *>(stage + xat[s] + i * 16 * BK));
#pragma unroll
      for (int j = 0; j < NT; ++j)
        wv[j] = as_h8(*reinterpret_cast<const uint4 *>(stage + wat[s] + j * 16 * BK));
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i)
          acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wv[j], xv[i], acc[j][i], 0, 0, 0);
    }
  };
  // One step: its stage has landed (each wave waits for its own loads, then all
  // meet; a bare barrier, since a fence would wait for the later stages too). Past
  // the barrier nobody reads the previous step's stage, which takes step t + S - 1.
  auto step = [&](uint32_t t, const uint16_t *stage, uint16_t *previous) __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(wait_stage((S - 2) * LPW));
    asm volatile("s_barrier" ::: "memory");
    issue(t + S - 1, previous);
    compute(stage);
  };
  uint16_t *const last = S == 3 ? s2 : S == 4 ? s3 : S == 5 ? s4 : s5;
  issue(0, s0);
  issue(1, s1);
  if constexpr (S > 3) issue(2, s2);
  if constexpr (S > 4) issue(3, s3);
  if constexpr (S > 5) issue(4, s4);
  // One turn of the ring from step t; whether steps are left.
  auto turn = [&](uint32_t t) __attribute__((always_inline)) {
    step(t, s0, last);
    if (t + 1 >= steps) return false;
    step(t + 1, s1, s0);
    if (t + 2 >= steps) return false;
    step(t + 2, s2, s1);
    if constexpr (S > 3) {
      if (t + 3 >= steps) return false;
      step(t + 3, s3, s2);
    }
    if constexpr (S > 4) {
      if (t + 4 >= steps) return false;
      step(t + 4, s4, s3);
    }
    if constexpr (S > 5) {
      if (t + 5 >= steps) return false;
      step(t + 5, s5, s4);
    }
    return t + S < steps;
  };
  // The compiler waits for every load once per iteration: two turns each.
  for (uint32_t t = 0; turn(t) && turn(t + S); t += 2 * S) {
  }
  __builtin_amdgcn_s_waitcnt(wait_stage(0));
  // The second group's sums, half of the blocks in each of two stages.
  constexpr int HALF = (MT * NT + 1) / 2;
  __syncthreads();
  f4_t *const slot[2] = {reinterpret_cast<f4_t *>(s0), reinterpret_cast<f4_t *>(s1)};
  auto at = [&](int f) { return slot[f / HALF] + ((wave & 3) * HALF + f % HALF) * 64 + lane; };
  if (group == 1)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int i = 0; i < MT; ++i) *at(j * MT + i) = acc[j][i];
  __syncthreads();
  if (group == 1) return;
  // Lane (kg, r) of block (j, i) holds features 4 kg .. 4 kg + 3 of x row r.
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const f4_t v = acc[j][i] + *at(j * MT + i);
      const uint32_t row = m0 + wm * (BM / 2) + 16 * i + r;
      const uint32_t col = n0 + wn * (BN / 2) + 16 * j + 4 * kg;
      if (row < p.m && col < p.n)
        *reinterpret_cast<uint2 *>(p.out + (int64_t)row * p.o_row + col) =
            make_uint2(pack_f16x2(v[0], v[1]), pack_f16x2(v[2], v[3]));
    }
}

template <int BM, int BN>
struct TileGrid {
  uint64_t row_tiles, col_tiles, tiles;
  TileGrid(const MatvecParams &p)
      : row_tiles((p.m + BM - 1ull) / BM), col_tiles((p.n + BN - 1ull) / BN), tiles(row_tiles * col_tiles) {}
  // Real rows of x in the row tiles, and real elements in all tiles, in percent.
  uint64_t row_fill(const MatvecParams &p) const { return 100ull * p.m / (row_tiles * BM); }
  uint64_t fill(const MatvecParams &p) const { return row_fill(p) * p.n / (col_tiles * BN); }
};

template <int BM, int BN, int BK, int S>
hipError_t run_tile(const MatvecParams &p, const Launch &l) {
  const TileGrid<BM, BN> g(p);
  return dispatch(gemm_tile_kernel<BM, BN, BK, S>, dim3((uint32_t)(g.tiles + kXcds - 1) / kXcds * kXcds), dim3(512),
                  0, l, p, (uint32_t)g.row_tiles, (uint32_t)g.col_tiles);
}

// The tile with the least rows of x and w together whose tiles fit the chip at once;
// None where the library measured faster (m = 33 to 3072 in 70 steps for 21 shapes of
// w from 1024 x 1024 to 8192 x 8192 and 4096 x 11008, and 16 others that drew no line;
// library / this in us). A tile's
// time goes by the real rows in it, the library's by its own larger tiles, so the
// lines are k, the share of the CUs and the share of real rows: where this says a
// tile, the worst is 5% (208 x [5120, 5120] 29.4 / 30.9; 224 of them 46.2 / 32.2).
//  - If none fits: 4096 x [5120, 8192] runs at 1.2 PFLOP/s in the library.
//  - 32 x 32: k up to 2048. 48 x [1536, 3072] 7.6 / 8.1, 64 x [1024, 4096] 8.3 / 9.8.
//  - 64 x 32: k up to 3584, or past 64 rows (64 x [5120, 4096] 17.6 / 18.4, 128 x [4096,
//    4096] 24.4 / 17.2).
//  - 64 x 64: from k = 4096 more than one row tile takes 60% of the CUs, up to 95 rows
//    70% (160 x [2816, 5632] 22.0 / 25.4; 90 x [5120, 5120] 22.0 / 25.3, [5120, 8192]
//    29.5 / 33.6; 96 of them 27.9 / 25.9).
//  - 64 x 96: k up to 2048, or 4096 for narrow w, two row tiles or less, or padding: 512 x
//    [2560, 4096] 23.7 / 25.2, 400 of them 24.8 / 23.1; 320 x [4096, 11008] 62 / 66, 700 x
//    [1536, 8960] 44.6 / 50.3.
//  - 128 x 64: past k = 1024 only on more than 3/4 of the CUs (384 x [4096, 4096] 24.9 /
//    28.2, 400 of them 25.7 / 24.9), past 4096 also not half empty (144 x [8192, 8192]
//    47.1 / 50.6).
//  - 192 x 64: three row tiles or more (300 x [6144, 2048] 17.9 / 19.2) and k up to 2048,
//    else to 5120 for wide w on nearly all CUs with some padding (768 x [3072, 3072]
//    27.4 / 30.2, 832 of them 27.4 / 25.9; 576 x [5120, 5120] 45.4 / 49.0).
enum class Tile { None, T32x32, T64x32, T64x64, T64x96, T128x64, T192x64 };

Tile pick_tile(const MatvecParams &p, uint64_t cus) {
  if (TileGrid<32, 32>(p).tiles <= cus) return p.k <= 2048 ? Tile::T32x32 : Tile::None;
  if (TileGrid<64, 32>(p).tiles <= cus) return p.k <= 3584 || (p.k <= 4096 && p.m > 64) ? Tile::T64x32 : Tile::None;
  if (const TileGrid<64, 64> g(p); g.tiles <= cus)
    return p.k < 4096 || p.m <= 64 || 10 * g.tiles >= (p.m < 96 ? 7 : 6) * cus ? Tile::T64x64 : Tile::None;
  if (const TileGrid<64, 96> g(p); g.tiles <= cus)
    return p.k <= 2048 || (p.k <= 4096 && p.n <= 1536) || p.m <= 128 || (p.k <= 8192 && (p.m <= 256 || g.fill(p) <= 92))
               ? Tile::T64x96
               : Tile::None;
  if (const TileGrid<128, 64> g(p); g.tiles <= cus)
    return p.k <= 1024 || (4 * g.tiles > 3 * cus && (p.k < 4096 || g.row_fill(p) >= 72)) ? Tile::T128x64
                                                                                        : Tile::None;
  if (const TileGrid<192, 64> g(p); g.tiles <= cus)
    return p.m > 384 && (p.k <= 2048 || (p.k <= 5120 && p.n >= 3072 && 100 * g.tiles >= 93 * cus &&
                                         g.row_fill(p) <= 92))
               ? Tile::T192x64
               : Tile::None;
  return Tile::None;
}

}  // namespace

bool gemm_tile_supported(const MatvecParams &p, uint32_t compute_units) {
  auto aligned = [](const void *ptr, uintptr_t to) { return reinterpret_cast<uintptr_t>(ptr) % to == 0; };
  return p.m > kSkinnyMaxRows && p.n > 0 && p.n % 4 == 0 && p.k > 0 && p.k % 128 == 0 &&
         p.x_row % 8 == 0 && p.w_row % 8 == 0 && p.o_row % 4 == 0 && aligned(p.x, 16) &&
         aligned(p.w, 16) && aligned(p.out, 8) && pick_tile(p, compute_units) != Tile::None;
}

hipError_t launch_gemm_tile(const MatvecParams &p, uint32_t compute_units, const Launch &l) {
  if (!gemm_tile_supported(p, compute_units)) return hipErrorInvalidValue;
  switch (pick_tile(p, compute_units)) {
    case Tile::T32x32: return run_tile<32, 32, 128, 6>(p, l);
    case Tile::T64x32: return run_tile<64, 32, 128, 6>(p, l);
    case Tile::T64x64: return run_tile<64, 64, 128, 4>(p, l);
    case Tile::T64x96: return run_tile<64, 96, 128, 3>(p, l);
    case Tile::T128x64: return run_tile<128, 64, 128, 3>(p, l);
    case Tile::T192x64: return run_tile<192, 64, 64, 4>(p, l);
    case Tile::None: break;
  }
  return hipErrorInvalidValue;
}

}  // namespace kernels
}  // namespace mi
