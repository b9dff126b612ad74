// Split-K attention of few query rows on MFMA (head_dim 64 and 128): up to 16
// packed (token, head in group) rows of one KV head per workgroup. Serves
// DecodeSplitKv, untuned FlashDecode, Tiled and the one-launch decode step
// where their rows kernel (attn_rows.hip) is bound by its vector arithmetic,
// which grows with rows x keys, or would read K/V once per head chunk or token.
//
// Replaces the same reference kernels as the rows kernel (transformer.metal:
// 1614-1665, 1824-2316). Probabilities are f32 values carried into the P V product
// as two f16 terms (hi + lo: 22 bits down to 2^-8 of the largest weight, 2^-31 of
// it below, where the rows kernel multiplies the 24), partials and their merge are
// f32; the error against 64 bits is the output's f16 rounding with both.
//  - One workgroup per (key split, KV head and head chunk, sequence). Its
//    waves take interleaved 32-key tiles, each with two register (K) and LDS
//    (V) stages, the next tile in flight while one is computed.
//  - S^T[key][row] = K Q^T on v_mfma_f32_16x16x32_f16, K rows loaded straight
//    into the A operand (lane (grp, col) holds key col, d 8 grp + 32 j). Each
//    lane then holds 8 keys of one row. O^T[d][row] += V^T P^T on the same
//    MFMA, once for P's hi and once for its lo terms: V rows land in the wave's
//    LDS stage by direct loads, in the key order of the S accumulator, and are
//    read transposed, so P is used in place.
//  - The last split of a unit to arrive merges all of them in split order in
//    the same launch (device_common.hpp, "Split partials"), one wave per row.
//
// What bounds it (per-workgroup timelines on MI355X, 32 heads, 4100 keys): the
// first tile's data at 3.5 us, the tile's dependent chain of QK, softmax and P V
// 1.2, wave merge 0.6, partial written through 0.9, arrival 0.4, the last
// arriver's merge 1.9. At 32768 keys and 64 heads (134 MB) the data phase runs
// at 7 TB/s and ends at 18 us. Graph replays over rotated caches, rows kernel ->
// this one: 32/8 heads, 4100 keys 15.3 -> 10.7 us; 40/8 23.5 -> 11.4; 64/8 24.5
// -> 12.0; 64/8, 32768 keys 137 -> 31 us; 32/8 of 64, 5000 keys 18.5 -> 8.5;
// Tiled, 4 tokens of 32/8 on 6000 keys 25.4 -> 15.7; the decode step, 64/8 heads,
// 20000 keys 31.9 -> 22.2. Eight waves in one workgroup per CU measured better
// than four in two (32768 keys: 31 against 42 us: half the partials to merge).
#include <type_traits>

#include "decode_tile.hpp"
#include "device_common.hpp"
#include "kernels.hpp"

namespace mi {
namespace kernels {
namespace {

using namespace mi::dev;

typedef float f4_t __attribute__((ext_vector_type(4)));

constexpr int KT = kDecodeTile;
// The exponent added to every probability: 2^(s - m_ref + kBias), so that the
// low f16 term of a weight of 2^-8 of the largest still has 22 bits above
// f16's smallest value. With the lazy rescale below a weight is at most
// 2^(kBias + 8).
constexpr float kBias = 6.0f;

// Wave slots of the workgroup merge: one per wave, and one for the new token of
// a decode step.
template <int D, bool STEP>
__global__ __launch_bounds__(kDecodeWaves * 64, 2) void attn_decode_kernel(const RowsParams p) {
  constexpr int WAVES = kDecodeWaves;
  constexpr int DC = D / 32, DB = D / 16, CPR = D / 8;  // QK chunks, O tiles, 16-byte chunks per row
  constexpr int THREADS = WAVES * 64, STAGE = KT * D, VL = KT * CPR / 64;
  constexpr int SLOTS = WAVES + (STEP ? 1 : 0);
  __shared__ __attribute__((aligned(16))) uint16_t v_lds_a[WAVES * STAGE];
  __shared__ __attribute__((aligned(16))) uint16_t v_lds_b[WAVES * STAGE];
  __shared__ float s_m[SLOTS][16], s_l[SLOTS][16];
  __shared__ float s_new[STEP ? D : 1];
  __shared__ float s_ang[STEP ? WAVES : 1][2][STEP ? D / 2 : 1];
  __shared__ uint32_t s_last;
  static_assert(16 * D * 4 <= STAGE * 2, "a wave's merged rows fit its stage");

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 15, grp = lane >> 4;
  const uint32_t split = blockIdx.x, b = blockIdx.z;
  uint32_t kvh = blockIdx.y, hc = 0, per_chunk = p.group;
  if (p.head_chunks != 1) {
    kvh = blockIdx.y / p.head_chunks, hc = blockIdx.y % p.head_chunks;
    per_chunk = (p.group + p.head_chunks - 1) / p.head_chunks;
  }
  const uint32_t unit = b * gridDim.y + blockIdx.y;
  const float c2 = p.scale_log2;
  // Rows of the unit: tokens x heads of the chunk (several chunks only with
  // one token), row r = token r / heads, head r % heads of the chunk.
  const uint32_t heads = min(per_chunk, p.group - hc * per_chunk);
  const uint32_t h0 = kvh * p.group + hc * per_chunk;
  const uint32_t rows = heads * p.tokens;
  uint32_t my_t = 0, my_g = min((uint32_t)col, rows - 1);
  if (p.tokens != 1) my_t = my_g / heads, my_g = my_g % heads;

  uint32_t len = p.kv_length, off = p.query_offset;
  if (p.lengths != nullptr) {
    len = min(p.lengths[b], p.kv_length);
    off = len >= p.tokens ? len - p.tokens : 0u;
  }
  // Visible cached keys: of the last token's row (the unit's), of the first
  // token's (below which no key needs a mask) and of this lane's. A decode
  // step's own key is not read from the cache.
  const uint64_t window = (uint64_t)off + (STEP ? 0 : 1);
  const bool causal = p.causal != 0 || STEP;
  const uint32_t available = causal ? (uint32_t)min((uint64_t)len, window + p.tokens - 1) : len;
  const uint32_t vis_first = causal ? (uint32_t)min((uint64_t)len, window) : len;
  const uint32_t vis = causal ? (uint32_t)min((uint64_t)len, window + my_t) : len;
  uint16_t *out = p.out + (int64_t)b * p.o_seq + (int64_t)h0 * p.o_head;
  auto out_row = [&](uint32_t r) -> uint16_t * {
    if (p.tokens == 1) return out + (int64_t)r * p.o_head;
    return out + (int64_t)(r / heads) * p.o_tok + (int64_t)(r % heads) * p.o_head;
  };
  if (!STEP && available == 0) {
    // No visible key: the reference divides 0 by 0.
    if (split == 0)
      for (uint32_t idx = tid; idx < rows * D; idx += THREADS) out_row(idx / D)[idx % D] = 0x7e00;
    return;
  }
  const uint32_t k0 = split * p.block_keys;
  if (split != 0 && k0 >= available) return;
  const uint32_t k1 = min(available, k0 + p.block_keys);
  const uint32_t ntiles = k1 > k0 ? (k1 - k0 + KT - 1) / KT : 0;

  const uint16_t *kb = p.k + (int64_t)b * p.k_seq + (int64_t)kvh * p.k_head;
  const uint16_t *vb = p.v + (int64_t)b * p.v_seq + (int64_t)kvh * p.v_head;
  // Loop-invariant byte offsets inside a full tile (its base is uniform). K:
  // lane (grp, col) loads key col (+ 16 for the second half), d 8 grp + 32 j.
  // V: direct-load instruction i writes 1 KB of LDS rows, lane L row (64 i + L) /
  // CPR and physical 16-byte chunk L % CPR.
  uint32_t v_off[VL], k_off[2];
#pragma unroll
  for (int i = 0; i < VL; ++i) {
    const int r = (64 * i + lane) / CPR, pc = lane % CPR;
    const int chunk = 2 * ((pc >> 1) ^ decode_v_swizzle<D>(r)) + (pc & 1);
    v_off[i] = (uint32_t)(decode_slot_key(r) * p.v_pos + chunk * 8) * 2u;
  }
#pragma unroll
  for (int hf = 0; hf < 2; ++hf) k_off[hf] = (uint32_t)((16 * hf + col) * p.k_pos + 8 * grp) * 2u;
  auto issue = [&](uint32_t ti, uint4 *kr, uint16_t *vst) __attribute__((always_inline)) {
    const uint32_t base = k0 + ti * KT;
    uint16_t *vdst = vst + wave * STAGE;
    if (base + KT <= k1) {
      const char *kt = reinterpret_cast<const char *>(kb + (int64_t)base * p.k_pos);
      const char *vt = reinterpret_cast<const char *>(vb + (int64_t)base * p.v_pos);
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int j = 0; j < DC; ++j)
          kr[hf * DC + j] = load16_nt(reinterpret_cast<const uint16_t *>(kt + k_off[hf] + 64 * j));
#pragma unroll
      for (int i = 0; i < VL; ++i)
        load_lds16_nt(reinterpret_cast<const uint16_t *>(vt + v_off[i]), vdst + i * 512);
    } else {
      // The split's last, partial tile: rows past it re-read its last key
      // (always in bounds) and are masked.
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        const uint32_t key = min(base + 16 * hf + col, k1 - 1);
#pragma unroll
        for (int j = 0; j < DC; ++j)
          kr[hf * DC + j] = load16_nt(kb + (int64_t)key * p.k_pos + 8 * grp + 32 * j);
      }
#pragma unroll
      for (int i = 0; i < VL; ++i) {
        const int r = (64 * i + lane) / CPR, pc = lane % CPR;
        const int chunk = 2 * ((pc >> 1) ^ decode_v_swizzle<D>(r)) + (pc & 1);
        const uint32_t key = min(base + (uint32_t)decode_slot_key(r), k1 - 1);
        load_lds16_nt(vb + (int64_t)key * p.v_pos + chunk * 8, vdst + i * 512);
      }
    }
  };
  // Q^T as the B operand: lane (grp, col) holds row col, d 8 grp + 32 j.
  uint4 qraw[DC];
  {
    const uint16_t *qb = p.q + (int64_t)b * p.q_seq + (int64_t)my_t * p.q_tok +
                         (int64_t)(h0 + my_g) * p.q_head + 8 * grp;
#pragma unroll
    for (int j = 0; j < DC; ++j) qraw[j] = *reinterpret_cast<const uint4 *>(qb + 32 * j);
  }
  // STEP: the new key row (in Q's layout, the same for every col), the norm
  // weights and the new value row, ahead of the cache rows.
  uint4 kraw[DC], wq[DC], wk[DC], vnew;
  if constexpr (STEP) {
#pragma unroll
    for (int j = 0; j < DC; ++j) {
      kraw[j] = *reinterpret_cast<const uint4 *>(p.step_k + (int64_t)kvh * p.step_k_head + 8 * grp + 32 * j);
      wq[j] = *reinterpret_cast<const uint4 *>(p.step_qw + 8 * grp + 32 * j);
      wk[j] = *reinterpret_cast<const uint4 *>(p.step_kw + 8 * grp + 32 * j);
    }
    vnew = *reinterpret_cast<const uint4 *>(p.step_v + (int64_t)kvh * p.step_v_head + 8 * (lane % CPR));
    __builtin_amdgcn_sched_barrier(0);
  }

  uint4 kra[2 * DC], krb[2 * DC];
  if ((uint32_t)wave < ntiles) issue(wave, kra, v_lds_a);
  const uint32_t nsplits = max(1u, (available + p.block_keys - 1) / p.block_keys);

  if constexpr (STEP) {
    // While the cache rows are in flight: qk_norm_rope_cache's transform of
    // the query rows and the key row (transformer.metal:1533-1577). A row is
    // spread over the four lane groups, and element d's RoPE partner d + D/2 is
    // chunk j + DC / 2 of the same lane. One angle per lane (pair = lane),
    // shared through the wave's own LDS.
#pragma clang fp contract(off)
    if (lane < D / 2) {
      const float frequency = powf(p.step_theta, -(float)(lane * 2) / (float)D);
      const float angle = (float)p.query_offset * frequency;
      s_ang[wave][0][lane] = cosf(angle);
      s_ang[wave][1][lane] = sinf(angle);
    }
    auto norm_rope = [&](uint4 *row, const uint4 *weight) __attribute__((always_inline)) {
      float n[DC][8];
      float sum = 0.0f;
#pragma unroll
      for (int j = 0; j < DC; ++j) {
        const uint32_t w[4] = {row[j].x, row[j].y, row[j].z, row[j].w};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          n[j][e] = (e & 1) ? hi_f16(w[e >> 1]) : lo_f16(w[e >> 1]);
          sum += n[j][e] * n[j][e];
        }
      }
      sum += __shfl_xor(sum, 16, 64);
      sum += __shfl_xor(sum, 32, 64);
      const float scale = 1.0f / sqrtf(sum / (float)D + p.step_eps);
#pragma unroll
      for (int j = 0; j < DC; ++j) {
        const uint32_t w[4] = {weight[j].x, weight[j].y, weight[j].z, weight[j].w};
#pragma unroll
        for (int e = 0; e < 8; ++e)
          n[j][e] = n[j][e] * scale * ((e & 1) ? hi_f16(w[e >> 1]) : lo_f16(w[e >> 1]));
      }
#pragma unroll
      for (int j = 0; j < DC / 2; ++j) {
        float lo[8], hi[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float c = s_ang[wave][0][32 * j + 8 * grp + e], s = s_ang[wave][1][32 * j + 8 * grp + e];
          const float x = n[j][e], y = n[j + DC / 2][e];
          lo[e] = x * c - y * s;
          hi[e] = x * s + y * c;
        }
        row[j] = make_uint4(pack_f16x2(lo[0], lo[1]), pack_f16x2(lo[2], lo[3]), pack_f16x2(lo[4], lo[5]),
                            pack_f16x2(lo[6], lo[7]));
        row[j + DC / 2] = make_uint4(pack_f16x2(hi[0], hi[1]), pack_f16x2(hi[2], hi[3]),
                                     pack_f16x2(hi[4], hi[5]), pack_f16x2(hi[6], hi[7]));
      }
    };
    norm_rope(qraw, wq);
    if (split != nsplits - 1 && tid < 16) s_m[WAVES][tid] = -INFINITY, s_l[WAVES][tid] = 0.0f;
    if (split != nsplits - 1 && tid < D) s_new[tid] = 0.0f;
    // The last split adds the new token: its score with every row as a wave
    // slot of the merge below, with weight 1 and its value row; and writes the
    // key and value rows into the caches, which no workgroup reads there.
    if (split == nsplits - 1 && wave == 0) {
      norm_rope(kraw, wk);
      float s = 0.0f;
#pragma unroll
      for (int j = 0; j < DC; ++j) {
        s = dot2(qraw[j].x, kraw[j].x, s);
        s = dot2(qraw[j].y, kraw[j].y, s);
        s = dot2(qraw[j].z, kraw[j].z, s);
        s = dot2(qraw[j].w, kraw[j].w, s);
      }
      s += __shfl_xor(s, 16, 64);
      s += __shfl_xor(s, 32, 64);
      if (grp == 0) {
        s_m[WAVES][col] = s * c2;
        s_l[WAVES][col] = 1.0f;
      }
      if (lane < CPR) {
        const uint32_t w[4] = {vnew.x, vnew.y, vnew.z, vnew.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) s_new[8 * lane + e] = (e & 1) ? hi_f16(w[e >> 1]) : lo_f16(w[e >> 1]);
      }
      if (hc == 0) {
        const int64_t pos = p.query_offset;
        if (col == 0)
#pragma unroll
          for (int j = 0; j < DC; ++j)
            *reinterpret_cast<uint4 *>(p.step_kc + (int64_t)kvh * p.k_head + pos * p.k_pos + 8 * grp +
                                       32 * j) = kraw[j];
        if (lane < CPR)
          *reinterpret_cast<uint4 *>(p.step_vc + (int64_t)kvh * p.v_head + pos * p.v_pos + 8 * lane) = vnew;
      }
    }
  }
  h8_t qop[DC];
#pragma unroll
  for (int j = 0; j < DC; ++j)
    qop[j] = as_h8((uint32_t)col < rows ? qraw[j] : make_uint4(0, 0, 0, 0));

  // Transposed V reads: lane (grp, mu) addresses row 8 grp + mu / 4 (and + 4),
  // d 16 dt + 4 (mu % 4).
  const int tr_row = 8 * grp + (col >> 2);
  const int tr_base = tr_row * D + 4 * (col & 1);
  const int tr_hi = (col & 3) >> 1, tr_f = decode_v_swizzle<D>(tr_row);
  f4_t o[DB];
#pragma unroll
  for (int dt = 0; dt < DB; ++dt) o[dt] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
  float m_run = -INFINITY, l_run = 0.0f;  // raw-score reference max, row sum

  // `finite` is a constant of the main loop: every value of the tile is.
  auto compute = [&](uint32_t ti, const uint4 *kr, const uint16_t *vst, bool finite) __attribute__((always_inline)) {
    const uint32_t base = k0 + ti * KT;
    f4_t s[2];  // s[hf][e]: row col, key 16 hf + 4 grp + e
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      s[hf] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < DC; ++j)
        s[hf] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_h8(kr[hf * DC + j]), qop[j], s[hf], 0, 0, 0);
    }
    if (base + KT > min(k1, vis_first)) {
      const uint32_t lim = min(k1, vis);
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (base + 16 * hf + 4 * grp + e >= lim) s[hf][e] = -INFINITY;
    }
    float mx = fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])),
                     fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    // Lazy rescale: the reference max moves only when some row outgrows it by
    // 2^8 (always on a row's first visible tile).
    if (__any((mx - m_run) * c2 > 8.0f)) {
      const float m_new = fmaxf(m_run, mx);
      const float alpha = m_new == -INFINITY ? 1.0f : exp2_raw((m_run - m_new) * c2);
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < DB; ++dt) o[dt] *= alpha;
      m_run = m_new;
    }
    const float mc = m_run == -INFINITY ? 0.0f : m_run * c2 - kBias;
    if (!finite) {
      float w[2][4];
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int e = 0; e < 4; ++e) w[hf][e] = exp2_raw(fmaf(s[hf][e], c2, -mc));
      const uint32_t lim = min(k1, vis);
      weigh_tile<D>(o, w, vst + wave * STAGE, v_lds_b + wave * STAGE, grp, col,
                    lim > base ? (int)min(lim - base, (uint32_t)KT) : 0);
      return;
    }
    // P as f16 pairs in the PV operand's key order: hi, and what it rounded off.
    uint32_t ph[4], pl[4];
    float ps = 0.0f;
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        const float p0 = exp2_raw(fmaf(s[hf][e], c2, -mc)), p1 = exp2_raw(fmaf(s[hf][e + 1], c2, -mc));
        const uint32_t h = pack_f16x2(p0, p1);
        ph[2 * hf + e / 2] = h;
        pl[2 * hf + e / 2] = pack_f16x2(p0 - lo_f16(h), p1 - hi_f16(h));
        ps += p0 + p1;
      }
    l_run += ps;
    const h8_t bh = as_h8(make_uint4(ph[0], ph[1], ph[2], ph[3]));
    const h8_t bl = as_h8(make_uint4(pl[0], pl[1], pl[2], pl[3]));
    const uint16_t *vw = vst + wave * STAGE;
#pragma unroll
    for (int dt = 0; dt < DB; ++dt) {
      const uint16_t *a0 = vw + tr_base + (2 * (dt ^ tr_f) + tr_hi) * 8;
      const uint2 lo = read_tr16(a0), hi = read_tr16(a0 + 4 * D);
      const h8_t a = as_h8(make_uint4(lo.x, lo.y, hi.x, hi.y));
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bl, o[dt], 0, 0, 0);
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bh, o[dt], 0, 0, 0);
    }
  };
  uint32_t ti = wave;
  while (ti < ntiles) {
    uint32_t nx = ti + WAVES;
    if (nx < ntiles) issue(nx, krb, v_lds_b);
    compute(ti, kra, v_lds_a, true);
    ti = nx;
    if (ti >= ntiles) break;
    nx = ti + WAVES;
    if (nx < ntiles) issue(nx, kra, v_lds_a);
    compute(ti, krb, v_lds_b, true);
    ti = nx;
  }
  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);

  // An infinite or NaN value row times a zero weight (a masked key, an empty low
  // term) is NaN in the products above. If any accumulator is not finite, the
  // wave takes its tiles again, those that hold such a value on the vector units
  // (visible keys only, whole f32 weights).
  {
    float bad = 0.0f;
#pragma unroll
    for (int dt = 0; dt < DB; ++dt) bad += (o[dt][0] + o[dt][1] + o[dt][2] + o[dt][3]) * 0.0f;
    if (__any(!(bad == 0.0f))) {
      const float l_sum = l_run;
#pragma unroll
      for (int dt = 0; dt < DB; ++dt) o[dt] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
      for (uint32_t t = wave; t < ntiles; t += WAVES) {
        issue(t, kra, v_lds_a);
        __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
        compute(t, kra, v_lds_a, !any_not_finite<2 * STAGE>(v_lds_a + wave * STAGE, lane));
      }
      l_run = l_sum;
    }
  }

  // Each wave's rows go to its own stage, the 16-byte chunks of row r at
  // chunk ^ r (a store instruction writes one chunk of 16 rows). Maxima in
  // log2 units with the weights' bias taken out.
  float *s_o = reinterpret_cast<float *>(v_lds_a) + wave * (STAGE / 2);
  if ((uint32_t)col < rows) {
    if (grp == 0) {
      s_m[wave][col] = m_run == -INFINITY ? -INFINITY : m_run * c2 - kBias;
      s_l[wave][col] = l_run;
    }
#pragma unroll
    for (int dt = 0; dt < DB; ++dt)
      *reinterpret_cast<f4_t *>(s_o + col * D + (((4 * dt + grp) ^ col) * 4)) = o[dt];
  }
  __syncthreads();
  const bool direct = nsplits == 1;
  float *part = p.partial + ((size_t)unit * p.max_splits + split) * p.rows * (D + 2);
  const uint32_t pairs = rows * (D / 2);
  for (uint32_t idx = tid; idx < pairs; idx += THREADS) {
    const uint32_t r = idx / (D / 2), d = 2 * (idx % (D / 2));
    const uint32_t at = r * D + (((d >> 2) ^ r) << 2) + (d & 3);
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < SLOTS; ++w) M = fmaxf(M, s_m[w][r]);
    float L = 0.0f, a0 = 0.0f, a1 = 0.0f;
#pragma unroll
    for (int w = 0; w < SLOTS; ++w) {
      const float f = s_m[w][r] == -INFINITY ? 0.0f : exp2_raw(s_m[w][r] - M);
      float2 v;
      if (w < WAVES)
        v = *reinterpret_cast<const float2 *>(reinterpret_cast<const float *>(v_lds_a) + w * (STAGE / 2) + at);
      else
        v = make_float2(s_new[d], s_new[d + 1]);
      L = fmaf(s_l[w][r], f, L);
      a0 = fmaf(v.x, f, a0);
      a1 = fmaf(v.y, f, a1);
    }
    if (direct) {
      const float inv = 1.0f / L;
      out_row(r)[d] = f32_to_f16(a0 * inv);
      out_row(r)[d + 1] = f32_to_f16(a1 * inv);
    } else {
      // A partial: the accumulators of every row, then (max, sum) per row.
      store_partial2(part + r * D + d, a0, a1);
      if (d == 0) store_partial2(part + p.rows * D + 2 * r, M, L);
    }
  }
  if (direct) return;
  // Every store of this workgroup has completed before the arrival counts.
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
  __syncthreads();
  if (tid == 0) {
    uint32_t *counter = p.counters + (size_t)unit * p.counter_stride;
    const bool last = arrive(counter) == nsplits - 1;
    if (last) {
      acquire_partials();
      __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    s_last = last;
  }
  __syncthreads();
  if (s_last == 0) return;

  // Log-sum-exp merge in split order, one wave per row: lane s loads split s's
  // (max, sum) and turns it into a weight, each lane EPL elements of every
  // split's accumulators, CH splits in flight per memory round trip. The weights
  // are wave-uniform per split (v_readlane), so a merge of up to CH splits
  // costs one round trip and one exponential per lane.
  constexpr int EPL = D / 64, CH = 32;
  const uint32_t stride = p.rows * (D + 2);
  const float *base = p.partial + (size_t)unit * p.max_splits * stride;
  for (uint32_t r = wave; r < rows; r += WAVES) {
    float M = -INFINITY, L = 0.0f, acc[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) acc[e] = 0.0f;
    for (uint32_t s0 = 0; s0 < nsplits; s0 += CH) {
      // Past the last split a lane re-reads it (in bounds) with weight 0.
      const uint32_t s = min(s0 + (lane & (CH - 1)), nsplits - 1);
      float2 ml = load_partial2(base + (size_t)s * stride + p.rows * D + 2 * r);
      float a[CH][EPL];
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const float *src = base + (size_t)min(s0 + i, nsplits - 1) * stride + r * D + EPL * lane;
        if constexpr (EPL == 2) {
          const float2 v = load_partial2(src);
          a[i][0] = v.x, a[i][1] = v.y;
        } else {
          a[i][0] = load_partial(src);
        }
      }
      if (s0 + (lane & (CH - 1)) >= nsplits) ml = make_float2(-INFINITY, 0.0f);
      // Both halves of the wave hold the same CH splits.
      float cm = ml.x;
      cm = fmaxf(cm, dpp_f32<kDppQuadXor1>(cm));
      cm = fmaxf(cm, dpp_f32<kDppQuadXor2>(cm));
      cm = fmaxf(cm, dpp_f32<kDppRowRor4>(cm));
      cm = fmaxf(cm, dpp_f32<kDppRowRor8>(cm));
      cm = fmaxf(cm, __shfl_xor(cm, 16, 64));
      cm = fmaxf(cm, M);
      const float f = ml.x == -INFINITY ? 0.0f : exp2_raw(ml.x - cm);
      const float alpha = M == -INFINITY ? 0.0f : exp2_raw(M - cm);
      L = L * alpha + lane_group_sum<32>(ml.y * f);
#pragma unroll
      for (int e = 0; e < EPL; ++e) acc[e] *= alpha;
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const float fi = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f), i));
        if (s0 + i < nsplits)
#pragma unroll
          for (int e = 0; e < EPL; ++e) acc[e] = fmaf(a[i][e], fi, acc[e]);
      }
      M = cm;
    }
    const float inv = 1.0f / L;
    uint16_t *dst = out_row(r) + EPL * lane;
#pragma unroll
    for (int e = 0; e < EPL; ++e) dst[e] = f32_to_f16(acc[e] * inv);
  }
}

}  // namespace

hipError_t launch_decode(const RowsParams &p, uint32_t head_dim, const Launch &l) {
  if (p.rows == 0 || p.rows > kDecodeRows) return hipErrorInvalidValue;
  const dim3 grid(p.max_splits, p.kv_heads * p.head_chunks, p.batch), block(kDecodeWaves * 64);
  if (head_dim == 128 && p.step_k != nullptr)
    return dispatch(attn_decode_kernel<128, true>, grid, block, 0, l, p);
  if (p.step_k != nullptr) return hipErrorInvalidValue;
  if (head_dim == 128) return dispatch(attn_decode_kernel<128, false>, grid, block, 0, l, p);
  if (head_dim == 64) return dispatch(attn_decode_kernel<64, false>, grid, block, 0, l, p);
  return hipErrorInvalidValue;
}

}  // namespace kernels
}  // namespace mi
