// Tiled attention of several query tokens on MFMA (AttentionKind::Tiled, D = 64
// and 128, more packed rows than the few-row kernel takes): a follow-up turn of
// 2 to 31 tokens on a cached conversation, and any longer Tiled call.
//
// Replaces attention_tiled_f16 (transformer.metal:1614-1665). The rows kernel
// serves a token per workgroup, so every token read the whole K/V range again
// (through L2) and paid vector arithmetic per (row, key). Here a workgroup owns
// 128 packed (token, head in group) rows of one KV head, as the flash prefill
// does, and walks 64-key K/V tiles staged into LDS by direct loads
// (prefill_tile.hpp); the differences from that kernel keep the Tiled kind's
// precision: probabilities are f32 values carried into P V as two f16 terms (hi +
// lo: 22 bits down to 2^-8 of the largest weight, 2^-31 of it below; twice the P V
// MFMAs), and split partials are f32.
//
// A few tokens give one row tile per KV head, so the keys are split over the
// chip and attn_tiled_merge_kernel, next on the stream, merges: with tens of
// partials of 128 rows (one KV head: over a hundred) an in-launch merge by the last
// arriver would read megabytes through one CU.
#include <type_traits>

#include "device_common.hpp"
#include "kernels.hpp"
#include "prefill_tile.hpp"

namespace mi {
namespace kernels {
namespace {

using namespace mi::dev;

constexpr int BN = kPrefillBlockN;
constexpr int BM = kPrefillBlockM;
// Added to every probability's exponent, so that the low f16 term of a weight of
// 2^-8 of the largest still has its 11 bits above f16's smallest value (2^-24); a
// smaller weight's pair is 2^-31 of the largest weight off at most. Weights are at
// most 2^(kBias + 8) (the lazy rescale).
constexpr float kBias = 6.0f;

typedef float f4_t __attribute__((ext_vector_type(4)));

template <int D>
__global__ __launch_bounds__(256, 2) void attn_tiled_kernel(const PrefillParams p) {
  constexpr int WAVES = 4, BPW = BN * D * 2 / 1024 / WAVES, CPR = D / 8, RPB = 1024 / (2 * D);
  constexpr int DC = D / 16, DT = D / 32;
  __shared__ __attribute__((aligned(16))) uint16_t k_lds_a[BN * D], k_lds_b[BN * D];
  __shared__ __attribute__((aligned(16))) uint16_t v_lds_a[BN * D], v_lds_b[BN * D];
  __shared__ uint32_t s_redo;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = lane & 31, h = lane >> 5;
  const uint32_t G = p.group;
  const uint32_t split = blockIdx.x, tile = p.row_tiles - 1 - blockIdx.y, kvh = blockIdx.z;
  const uint32_t row0 = tile * BM;
  const uint32_t my_row = row0 + wave * 32 + n;
  const uint32_t my_t = my_row / G, my_g = my_row % G;
  const bool row_ok = my_t < p.tokens;
  const uint32_t t_first = row0 / G, t_last = min(p.tokens - 1, (row0 + BM - 1) / G);
  const uint64_t L = p.kv_length, off = p.query_offset;
  const uint32_t kmax = p.causal != 0 ? (uint32_t)min(L, off + t_last + 1) : (uint32_t)L;
  const uint32_t n_tiles = (kmax + BN - 1) / BN;
  const uint32_t per_split = p.splits > 1 ? p.split_tiles : n_tiles;
  const uint32_t t_begin = split * per_split;
  if (t_begin >= n_tiles) return;  // the row tile needs fewer splits
  const uint32_t t_end = min(n_tiles, t_begin + per_split);
  // Last visible key of this lane's row, and of the tile's first row (below
  // which no key needs a mask).
  const uint64_t lim = p.causal != 0 ? min(L - 1, off + min(my_t, p.tokens - 1)) : L - 1;
  const uint64_t full_lim = p.causal != 0 ? min(L - 1, off + t_first) : L - 1;
  // Waves past the last row only load.
  const bool busy = (row0 + (uint32_t)__builtin_amdgcn_readfirstlane(wave) * 32) / G < p.tokens;

  const uint16_t *kbase = p.k + (int64_t)kvh * p.k_head;
  const uint16_t *vbase = p.v + (int64_t)kvh * p.v_head;
  // Direct loads of tile `ti`: each wave fills BPW 1 KB blocks (RPB tile rows
  // each) of the K and V stages, each lane the 16 bytes that belong at its
  // swizzled position.
  uint32_t k_off[BPW], v_off[BPW];
#pragma unroll
  for (int i = 0; i < BPW; ++i) {
    const int row = (wave * BPW + i) * RPB + lane / CPR, pc = lane % CPR;
    k_off[i] = (uint32_t)(row * p.k_pos + ((pc ^ k_swizzle<D>(row)) * 8)) * 2u;
    v_off[i] = (uint32_t)(row * p.v_pos + ((pc ^ v_swizzle<D>(row)) * 8)) * 2u;
  }
  auto issue_tile = [&](uint32_t ti, uint16_t *ks, uint16_t *vs) __attribute__((always_inline)) {
    const uint32_t j0 = ti * BN;
    const uint16_t *kt = kbase + (int64_t)j0 * p.k_pos;
    const uint16_t *vt = vbase + (int64_t)j0 * p.v_pos;
    if (j0 + BN <= kmax) {
#pragma unroll
      for (int i = 0; i < BPW; ++i) {
        const int blk = wave * BPW + i;
        load_lds16(reinterpret_cast<const uint16_t *>(reinterpret_cast<const char *>(kt) + k_off[i]),
                   ks + blk * 512);
        load_lds16(reinterpret_cast<const uint16_t *>(reinterpret_cast<const char *>(vt) + v_off[i]),
                   vs + blk * 512);
      }
      return;
    }
    // Partial last tile: rows past the last key re-read that key.
    const int last = (int)(kmax - 1 - j0);
#pragma unroll
    for (int i = 0; i < BPW; ++i) {
      const int blk = wave * BPW + i;
      const int row = blk * RPB + lane / CPR, pc = lane % CPR, rr = min(row, last);
      load_lds16(kt + (uint32_t)(rr * p.k_pos + ((pc ^ k_swizzle<D>(row)) * 8)), ks + blk * 512);
      load_lds16(vt + (uint32_t)(rr * p.v_pos + ((pc ^ v_swizzle<D>(row)) * 8)), vs + blk * 512);
    }
  };
  // Q^T as the B operand: lane (h, n) holds Q[row n][16c + 8h .. +8].
  h8_t qop[DC];
  {
    const uint16_t *qrow = p.q + (int64_t)min(my_t, p.tokens - 1) * p.q_tok +
                           (int64_t)(kvh * G + my_g) * p.q_head;
#pragma unroll
    for (int c = 0; c < DC; ++c)
      qop[c] = row_ok ? as_h8(*reinterpret_cast<const uint4 *>(qrow + 16 * c + 8 * h))
                      : as_h8(make_uint4(0, 0, 0, 0));
  }
  if (tid == 0) s_redo = 0;
  issue_tile(t_begin, k_lds_a, v_lds_a);
  if (t_begin + 1 < t_end) {
    issue_tile(t_begin + 1, k_lds_b, v_lds_b);
    static_assert(2 * BPW < 16, "vmcnt immediate");
    __builtin_amdgcn_s_waitcnt(kWaitVmcnt0 | (2 * BPW));
  } else {
    __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
  }
  // Bare barrier: a workgroup fence would wait for the second tile too. Each
  // wave has waited for its own part of the first, and for s_redo.
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

  float16_t o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.0f;
  float m_run = -INFINITY, l_run = 0.0f;  // raw-score reference max, this half-wave's row sum
  const float c2 = p.scale_log2;
  // Lane roles in the V^T transpose reads, as in the flash prefill.
  const int tr_g = lane >> 4, tr_a = lane & 3, tr_j = (lane >> 2) & 3;
  const int tr_key = 4 * (tr_g >> 1) + tr_j;
  const int tr_off = tr_key * D + 4 * (tr_a & 1);
  const int tr_chunk = 2 * (tr_g & 1) + (tr_a >> 1);

  // `finite` (a constant of each call): P V on MFMA, which every value has to be for.
  auto compute = [&](uint32_t it, const uint16_t *k_lds, const uint16_t *v_lds, bool finite) __attribute__((always_inline)) {
    const uint32_t j0 = it * BN;
    float16_t s[2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[mt][r] = 0.0f;
#pragma unroll
      for (int c = 0; c < DC; ++c) {
        const uint16_t *kp = k_lds + (32 * mt + n) * D + (((2 * c + h) ^ k_swizzle<D>(n)) * 8);
        s[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(as_h8(*reinterpret_cast<const uint4 *>(kp)), qop[c],
                                                       s[mt], 0, 0, 0);
      }
    }
    if ((uint64_t)j0 + BN - 1 > full_lim) {
      const int lim_rel = (int)max(min((int64_t)lim - (int64_t)j0, (int64_t)BN), (int64_t)-1);
      const int lim_lane = lim_rel - 4 * h;
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key_c = 32 * mt + 8 * (r >> 2) + (r & 3);
          s[mt][r] = key_c > lim_lane ? -INFINITY : s[mt][r];
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[mt][r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    // Lazy rescale: the reference max moves only when some row outgrows it by
    // 2^8 (always on a row's first visible tile).
    if (__any((mx - m_run) * c2 > 8.0f)) {
      const float m_new = fmaxf(m_run, mx);
      const float alpha = m_new == -INFINITY ? 1.0f : exp2_raw((m_run - m_new) * c2);
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
      m_run = m_new;
    }
    const float mc = m_run == -INFINITY ? 0.0f : m_run * c2 - kBias;
    float ps0 = 0.0f, ps1 = 0.0f;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        s[mt][r] = exp2_raw(fmaf(s[mt][r], c2, -mc));
        s[mt][r + 1] = exp2_raw(fmaf(s[mt][r + 1], c2, -mc));
        ps0 += s[mt][r];
        ps1 += s[mt][r + 1];
      }
    l_run += ps0 + ps1;
    if (!finite) {
      // P V on the vector units: the wave's weights go through LDS (the second
      // stage, 32 keys at a time), and each lane adds the keys that its row sees
      // to its d = 32 dt + 8 q + 4 h + e.
      float *weights = reinterpret_cast<float *>((wave < 2 ? k_lds_b : v_lds_b) + (wave & 1) * 2048);
      const int last = (int)max(min((int64_t)lim - (int64_t)j0, (int64_t)BN), (int64_t)-1);
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
#pragma unroll
        for (int r = 0; r < 16; ++r) weights[(8 * (r >> 2) + 4 * h + (r & 3)) * 32 + n] = s[mt][r];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma clang loop unroll_count(D == 64 ? 2 : 1)
        for (int key = 0; key < 32; ++key) {
          const float f = weights[key * 32 + n];
          const uint16_t *row = v_lds + (32 * mt + key) * D + 4 * h;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              uint2 v = *reinterpret_cast<const uint2 *>(row + ((4 * dt + q) ^ v_swizzle<D>(key)) * 8);
              if (32 * mt + key > last) v = make_uint2(0, 0);
              o[dt][4 * q] = fmaf(f, lo_f16(v.x), o[dt][4 * q]);
              o[dt][4 * q + 1] = fmaf(f, hi_f16(v.x), o[dt][4 * q + 1]);
              o[dt][4 * q + 2] = fmaf(f, lo_f16(v.y), o[dt][4 * q + 2]);
              o[dt][4 * q + 3] = fmaf(f, hi_f16(v.y), o[dt][4 * q + 3]);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      }
      return;
    }
    // O^T[d][row] += V^T[d][keys] P^T[keys][row], four 16-key chunks, P's low
    // terms first.
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      uint32_t ph[4], pl[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float p0 = s[c >> 1][8 * (c & 1) + 2 * w], p1 = s[c >> 1][8 * (c & 1) + 2 * w + 1];
        ph[w] = pack_f16x2(p0, p1);
        pl[w] = pack_f16x2(p0 - lo_f16(ph[w]), p1 - hi_f16(ph[w]));
      }
      const h8_t bh = as_h8(make_uint4(ph[0], ph[1], ph[2], ph[3]));
      const h8_t bl = as_h8(make_uint4(pl[0], pl[1], pl[2], pl[3]));
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const int sw = ((4 * dt + tr_chunk) ^ v_swizzle<D>(tr_key)) * 8;
        const uint16_t *v0 = v_lds + 16 * c * D + tr_off + sw;
        const uint2 l2 = read_tr16(v0), h2 = read_tr16(v0 + 8 * D);
        const h8_t a = as_h8(make_uint4(l2.x, l2.y, h2.x, h2.y));
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, bl, o[dt], 0, 0, 0);
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, bh, o[dt], 0, 0, 0);
      }
    }
  };
  // Tile t_begin + k lives in stage k & 1: after a tile its successor (issued a
  // tile ago) has landed, and past the barrier nobody reads this stage, which
  // takes the tile after that.
  for (uint32_t it = t_begin;; it += 2) {
    if (busy) compute(it, k_lds_a, v_lds_a, true);
    if (it + 1 >= t_end) break;
    __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
    __syncthreads();
    if (it + 2 < t_end) issue_tile(it + 2, k_lds_a, v_lds_a);
    if (busy) compute(it + 1, k_lds_b, v_lds_b, true);
    if (it + 2 >= t_end) break;
    __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
    __syncthreads();
    if (it + 3 < t_end) issue_tile(it + 3, k_lds_b, v_lds_b);
  }
  // An infinite or NaN value row times a zero weight (a masked key, an empty low
  // term) is NaN in the products above: a wave with an accumulator that is not
  // finite says so at the last tile's barrier.
  float sum = 0.0f;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) sum = fmaf(o[dt][r], 0.0f, sum);
  const bool bad = __any(!(sum == 0.0f));
  if (bad && lane == 0) s_redo = 1;
  __syncthreads();
  // Then the workgroup's tiles are loaded again, and the waves that have such an
  // accumulator take them again on the vector units, visible keys only and with whole f32
  // weights (MFMA for the tiles without such a value costs the main loop its
  // registers: 16 spilled).
  if (s_redo != 0) {
    const float l_sum = l_run;
    if (bad)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] = 0.0f;
#pragma unroll 1
    for (uint32_t it = t_begin; it < t_end; ++it) {
      issue_tile(it, k_lds_a, v_lds_a);
      __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
      __syncthreads();
      if (bad) compute(it, k_lds_a, v_lds_a, false);
      __syncthreads();
    }
    l_run = l_sum;
  }
  const float l_total = l_run + __shfl_xor(l_run, 32, 64);
  if (n_tiles > per_split) {
    // A partial, in the accumulator's order (512 or 1024 contiguous bytes per
    // store): per wave, slot 0 (8 bytes a lane) = (max in log2 units with the
    // weights' bias taken out, sum), then DT * 4 slots of four O values (16
    // bytes a lane), value r of d tile dt in slot 4 dt + r / 4.
    if (!busy) return;
    float *mine = p.partial + ((((size_t)split * p.row_tiles + tile) * p.kv_heads + kvh) * WAVES + wave) *
                                  64 * (D / 2 + 2);
    *reinterpret_cast<float2 *>(mine + 2 * lane) =
        make_float2(m_run == -INFINITY ? -INFINITY : m_run * c2 - kBias, l_total);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f4_t *>(mine + 128 + (4 * dt + q) * 256 + 4 * lane) =
            f4_t{o[dt][4 * q], o[dt][4 * q + 1], o[dt][4 * q + 2], o[dt][4 * q + 3]};
    return;
  }
  // Normalise and store through LDS, as the flash prefill: the wave's 32 rows as
  // f16 in its own region of the idle stages, then whole 16-byte chunks. The
  // loop's last barrier is behind every operand read.
  const float inv = 1.0f / l_total;
  constexpr int RPI = 64 / CPR;
  static_assert(2 * 32 * D <= BN * D, "output staging");
  uint16_t *rows_lds = (wave < 2 ? k_lds_a : k_lds_b) + (wave & 1) * 32 * D;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint2 v;
      v.x = pack_f16x2(o[dt][4 * q] * inv, o[dt][4 * q + 1] * inv);
      v.y = pack_f16x2(o[dt][4 * q + 2] * inv, o[dt][4 * q + 3] * inv);
      *reinterpret_cast<uint2 *>(rows_lds + n * D + ((4 * dt + q) ^ out_swizzle<D>(n)) * 8 + 4 * h) = v;
    }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 32 / RPI; ++i) {
    const int r = i * RPI + lane / CPR, c = lane % CPR;
    const uint4 v = *reinterpret_cast<const uint4 *>(rows_lds + r * D + (c ^ out_swizzle<D>(r)) * 8);
    const uint32_t prow = row0 + wave * 32 + r, t = prow / G, g = prow % G;
    if (t < p.tokens)
      *reinterpret_cast<uint4 *>(p.out + (int64_t)t * p.o_tok + (int64_t)(kvh * G + g) * p.o_head + c * 8) = v;
  }
}

// Merges the splits of attn_tiled_kernel in split order: one wave per (row tile,
// KV head, 32-row wave, slot of four O values), lane (h, n) taking row n's four
// values from every split, CH splits in flight.
template <int D>
__global__ __launch_bounds__(256) void attn_tiled_merge_kernel(const PrefillParams p) {
  constexpr int CH = 8;
  const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
  const uint32_t slot = blockIdx.y * 4 + (threadIdx.x >> 6);
  const uint32_t region = blockIdx.x, wave = region % 4, unit = region / 4;
  const uint32_t kvh = unit % p.kv_heads, tile = unit / p.kv_heads;
  const uint32_t row = tile * BM + wave * 32 + n, t = row / p.group, g = row % p.group;
  if ((tile * BM + wave * 32) / p.group >= p.tokens) return;
  const uint32_t t_last = min(p.tokens - 1, (tile * BM + BM - 1) / p.group);
  const uint32_t kmax = p.causal != 0
                            ? (uint32_t)min((uint64_t)p.kv_length, (uint64_t)p.query_offset + t_last + 1)
                            : p.kv_length;
  const uint32_t nsplits = ((kmax + BN - 1) / BN + p.split_tiles - 1) / p.split_tiles;
  if (nsplits <= 1) return;  // written by the split kernel
  const size_t stride = (size_t)p.row_tiles * p.kv_heads * 4 * 64 * (D / 2 + 2);
  const float *base = p.partial + (size_t)region * 64 * (D / 2 + 2);
  float M = -INFINITY, L = 0.0f;
  f4_t acc = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
  for (uint32_t s0 = 0; s0 < nsplits; s0 += CH) {
    float2 ml[CH];
    f4_t a[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      // Past the last split: re-read it (in bounds) with weight 0.
      const float *ps = base + (size_t)min(s0 + i, nsplits - 1) * stride;
      ml[i] = *reinterpret_cast<const float2 *>(ps + 2 * lane);
      a[i] = *reinterpret_cast<const f4_t *>(ps + 128 + slot * 256 + 4 * lane);
    }
    float cm = M;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      if (s0 + i >= nsplits) ml[i].x = -INFINITY;
      cm = fmaxf(cm, ml[i].x);
    }
    const float alpha = M == -INFINITY ? 0.0f : exp2_raw(M - cm);
    L *= alpha;
    acc *= alpha;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      if (ml[i].x == -INFINITY) continue;
      const float f = exp2_raw(ml[i].x - cm);
      L = fmaf(ml[i].y, f, L);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = fmaf(a[i][e], f, acc[e]);
    }
    M = cm;
  }
  if (t >= p.tokens) return;
  const float inv = 1.0f / L;
  uint2 v;
  v.x = pack_f16x2(acc[0] * inv, acc[1] * inv);
  v.y = pack_f16x2(acc[2] * inv, acc[3] * inv);
  *reinterpret_cast<uint2 *>(p.out + (int64_t)t * p.o_tok + (int64_t)(kvh * p.group + g) * p.o_head +
                             8 * slot + 4 * h) = v;
}

template <int D>
hipError_t launch_tiled_d(const PrefillParams &p, TiledPhase phase, const Launch &l) {
  if (phase == TiledPhase::Split)
    return dispatch(attn_tiled_kernel<D>, dim3(p.splits, p.row_tiles, p.kv_heads), dim3(256), 0, l, p);
  if (p.splits <= 1) return no_dispatch(l);
  return dispatch(attn_tiled_merge_kernel<D>, dim3(p.row_tiles * p.kv_heads * 4, D / 32), dim3(256), 0, l, p);
}

}  // namespace

hipError_t launch_tiled(const PrefillParams &p, uint32_t head_dim, TiledPhase phase, const Launch &l) {
  if (p.block_m != BM || p.splits == 0) return hipErrorInvalidValue;
  if (head_dim == 128) return launch_tiled_d<128>(p, phase, l);
  if (head_dim == 64) return launch_tiled_d<64>(p, phase, l);
  return hipErrorInvalidValue;
}

}  // namespace kernels
}  // namespace mi
