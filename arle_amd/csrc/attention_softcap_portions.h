// Prompt portions of the soft-capped attention at heads of 128: four waves share tiles of keys and values in LDS.
// Included by attention_softcap.hip behind its arguments and vector types.
#pragma once
#include "common.h"
#include "lds_loads.h"

namespace arle {

// A workgroup of four waves takes 128 rows (row = token * G + head of the kv head's group) of a request and kv head, 32 a
// wave, and walks the keys in tiles of 64 that are loaded from memory straight into LDS, the next one while this one is worked.
// The layouts of tiles, scores and probabilities are those of attn_prefill_dma_kernel (attention_portions_dma.h): a lane
// (row j = lane % 32, h = lane / 32) holds the scores of its row and the keys 32 t + 16 (r / 8) + 8 h + r % 8.
//
// What bounds it is arithmetic: a score takes the cap, the penalty, an exponential, a maximum and a sum, and quarter-rate
// instructions cost as much as four others.  So
//   * the cap is a polynomial where all scores of a wave's tile lie within half of it: cap tanh(x / cap) = x P((x / cap)^2) with the
//     minimax P of degree 4 for tanh(t) / t over |t| <= 0.5 (off by 2.6e-8, and t P from tanh by 1.3e-8; six multiply-adds where
//     the exponential and the reciprocal take 44 cycles), and the exponential form elsewhere;
//   * the distance penalties of a group of four heads come from a table in LDS, filled once a workgroup for windows of up
//     to 1,024 (PEN 1; the heads side by side, so that the lanes of a wave spread over the banks, and distances descending,
//     so that a lane's sixteen keys are one base and sixteen constants); other groups and windows compute them (PEN 2: the same layer
//     in groups of two 73 us, of eight 72, by waves of their own 107 and 106; without a window 89 and 162);
//   * masks are worked out in the tiles at the ends only, and sums are rescaled only where a maximum has grown by 2^8.
// A layer of 2,048 rows of 32 q heads and 8 kv heads, window 1,024, cap and penalty: 66 us, 110 with every wave fetching its tiles
// by itself into registers (attn_softcap_mfma_kernel, 32 rows a wave); without the penalty 60, with neither 50.  What a wave spends is
// the sum of its parts rather than the longest (leaving one out of the loads, the second product or the exponentials takes 5 to 6 us
// each): two waves a SIMD hide little of one another.
constexpr int kCpWaves = 4;
constexpr int kCpRows = 32 * kCpWaves;
constexpr int kCpD = 128;
constexpr int kCpKeys = 64;
constexpr int kCpStage = kCpKeys * kCpD * 2 * 2;      // keys and values of a tile
constexpr int kCpTableGroup = 4, kCpTableMax = 1024;  // q heads a kv head, and the longest window, that the penalties' table is for
constexpr int kCpTable = kCpTableGroup * kCpTableMax * static_cast<int>(sizeof(float));
static_assert(2 * (2 * kCpStage + kCpTable) <= 160 * 1024, "two workgroups a compute unit");
constexpr float kCpLazyBits = 8.0f;
typedef float f32x16_t __attribute__((ext_vector_type(16)));

template <int PEN>
__global__ __launch_bounds__(kCpWaves* kWave, 2) void cap_portions_kernel(const CapArgs a) {
  constexpr int D = kCpD;
  extern __shared__ __align__(16) unsigned char lds_all[];
  float* const table_lds = reinterpret_cast<float*>(lds_all + 2 * kCpStage);
  const int tid = threadIdx.x, lane = tid & 63, j = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = a.nq / a.nkv, P = a.page_size, ps = __builtin_ctz(static_cast<unsigned>(P)), pm = P - 1;
  // Neighbouring workgroups are kv heads, which the dies of the chip take in turn: with eight of them a die keeps to one, and
  // its keys and values to its level-two cache.  The last row blocks, which see the most keys, come first.
  const int kvh = static_cast<int>(blockIdx.x) % a.nkv;
  int left = static_cast<int>(blockIdx.x) / a.nkv, seg = -1;
  for (int s = a.segments - 1; s >= 0; --s) {
    const int blocks = ((a.seg_row0[s + 1] - a.seg_row0[s]) * G + kCpRows - 1) / kCpRows;
    if (left < blocks) {
      seg = s;
      left = blocks - 1 - left;
      break;
    }
    left -= blocks;
  }
  if (seg < 0) return;
  const int row0 = a.seg_row0[seg], rows = (a.seg_row0[seg + 1] - row0) * G, qlen = rows / G, start = a.seg_start[seg];
  const int wg_row = left * kCpRows;
  const int* table = a.block_table + static_cast<int64_t>(a.seg_slot[seg]) * a.table_stride;
  const int tok_min = wg_row / G, tok_max = (min(wg_row + kCpRows, rows) - 1) / G;
  const int kv_hi = start + tok_max + 1;
  const int kv_lo = a.window > 0 ? max(0, start + tok_min - a.window + 1) : 0;
  const int t0 = kv_lo / kCpKeys, t1 = (kv_hi + kCpKeys - 1) / kCpKeys;

  const int row_begin = wg_row + 32 * wave;
  const bool wave_has_rows = row_begin < rows;
  const int wave_tok_max = wave_has_rows ? (min(row_begin + 32, rows) - 1) / G : 0;
  const int wave_kv_hi = start + wave_tok_max + 1;                                           // the keys that any row of the wave sees
  const int wave_pos_min = start + min(row_begin, rows - 1) / G;
  const int wave_kv_lo = a.window > 0 ? max(0, wave_pos_min - a.window + 1) : 0;
  const int wave_win_lo = a.window > 0 ? max(0, start + wave_tok_max - a.window + 1) : 0;    // and from here to wave_pos_min all rows
  const int row = row_begin + j;
  const bool row_ok = row < rows;
  const int my_tok = min(row / G, qlen - 1), my_head = kvh * G + row % G, my_pos = start + my_tok;
  bf16x8_t qreg[D / 16];
  {
    const bf16* qp = a.q + static_cast<int64_t>(row0 + my_tok) * a.q_stride + my_head * D + 8 * h;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) qreg[s] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(qp + 16 * s));
  }
  const int jk = (j & 19) | ((j & 4) << 1) | ((j & 8) >> 1);   // row i of a score tile is the key with bits 2 and 3 of i exchanged

  // page ids of 64 consecutive logical pages in one register across the wave (lane i: page pg_base + i)
  const int pg_first = kv_lo >> ps, pg_last = (kv_hi - 1) >> ps;
  int pg_base = 0, pg_reg = 0;
  auto cover = [&](int tile, bool first) {
    const int lo = min(max(tile * kCpKeys >> ps, pg_first), pg_last), hi = min(max((tile * kCpKeys + kCpKeys - 1) >> ps, pg_first), pg_last);
    if (first || lo < pg_base || hi >= pg_base + kWave) {
      pg_base = lo;
      pg_reg = table[min(lo + lane, pg_last)];
    }
  };
  const int64_t page_elems = static_cast<int64_t>(a.nkv) * P * D, head_off = static_cast<int64_t>(kvh) * P * D;
  // Four loads of keys and four of values a wave and tile: piece q = 64 (4 wave + i) + lane of the keys is key q / 16,
  // position q % 16 in its row, of the values d row q / 8, position q % 8.
  // A page holds sixteen keys at least, so a wave's sixteen lie in one (a lookup for each of the four loads cost 3 us).
  auto fetch = [&](int tile, int stage) __attribute__((always_inline)) {
    const int base = tile * kCpKeys;
    unsigned char* at = lds_all + stage * kCpStage + (4 * wave) * 1024;
    int k_src = (lane >> 4) * D + 8 * ((lane & 15) ^ (lane >> 4)), v_key = 8 * ((lane & 7) ^ (lane >> 4));
    asm volatile("" : "+v"(k_src), "+v"(v_key));   // (not kept over the loop)
    int v_at[2], v_page[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {   // keys outside the request are fetched from the nearest page that is there, and masked
      v_at[i] = min(max(base + (v_key ^ (32 * i)), kv_lo & ~7), (kv_hi - 1) & ~7);
      v_page[i] = __shfl(pg_reg, (v_at[i] >> ps) - pg_base, kWave);
    }
    const int first_key = base + 16 * wave;
    const int page_at = min(max(first_key >> ps, pg_first), pg_last) - pg_base;
    const int page = __builtin_amdgcn_readlane(pg_reg, __builtin_amdgcn_readfirstlane(page_at));
    const bf16* kb = a.k_pages + page * page_elems + head_off + (first_key & pm) * D;
#pragma unroll
    for (int i = 0; i < 4; ++i) load_to_lds_16(kb, 2u * static_cast<uint32_t>((k_src ^ (32 * i)) + 4 * i * D), at + i * 1024);
    const bf16* vb[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
      vb[i] = a.v_pages + v_page[i] * page_elems + head_off + ((32 * wave + 8 * i + (lane >> 3)) * P + (v_at[i] & pm));
#pragma unroll
    for (int i = 0; i < 4; ++i) load_to_lds_16(vb[i & 1] + (i & 2) * 8 * P, at + kCpKeys * D * 2 + i * 1024);
  };
  cover(t0, true);
  fetch(t0, 0);

  // Scores are kept in units of ln 2, so that every exponential is one of base 2.
  constexpr float kLog2e = 1.4426950408889634f;
  const float pen1 = PEN ? load_as_float(a.r1, a.r_dtype, my_head) : 0.f, pen2 = PEN ? load_as_float(a.r2, a.r_dtype, my_head) : 0.f;
  const float scale2 = a.scale * kLog2e, cap2 = a.cap * kLog2e;
  const float to_exp = a.cap > 0.f ? 2.0f * kLog2e * a.scale / a.cap : 0.f;        // the exponential form: 1 / (1 + exp(2 x / cap))
  // the polynomial in the square of a product, its coefficients scaled for it
  const float in_cap = a.cap > 0.f ? a.scale / a.cap : 0.f, sq = in_cap * in_cap;
  const float within = in_cap > 0.f ? 0.5f / in_cap : -1.0f;      // products of up to so much (a cap below 0, none: never)
  const float c1 = -0.33333070f * sq * scale2, c2 = 0.13324780f * sq * sq * scale2, c3 = -0.05298607f * sq * sq * sq * scale2,
              c4 = 0.017135007f * sq * sq * sq * sq * scale2;
  const int span = PEN == 1 ? a.window : 0;                       // entry e * 4 + head: distance span - 1 - e
  if constexpr (PEN == 1) {
    const int hg = tid % kCpTableGroup;
    const float p1 = load_as_float(a.r1, a.r_dtype, kvh * G + hg), p2 = load_as_float(a.r2, a.r_dtype, kvh * G + hg);
    // (of the distances that occur between this workgroup's rows and keys; what a masked lane reads elsewhere is dropped)
    for (int e = max(0, span - (kv_hi - kv_lo)) + tid / kCpTableGroup; e < span; e += kCpWaves * kWave / kCpTableGroup)
      table_lds[e * kCpTableGroup + hg] = p1 * __builtin_amdgcn_logf(1.0f + p2 * static_cast<float>(span - 1 - e));
  }

  f32x16_t o[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  float m = -INFINITY, l = 0.f;
  // the query has to be there before the loop: a wait for it inside would wait for the tiles in flight too
#pragma unroll
  for (int s = 0; s < D / 16; ++s) asm volatile("" ::"v"(qreg[s]));

  for (int tile = t0; tile < t1; ++tile) {
    const int stage = (tile - t0) & 1;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's pieces of the tile have landed
    __syncthreads();                                   // everybody's have; and everybody is done with the other stage
    if (tile + 1 < t1) {
      cover(tile + 1, false);
      fetch(tile + 1, stage ^ 1);
    }
    const int key_base = tile * kCpKeys;
    if (!(wave_has_rows && key_base < wave_kv_hi && key_base + kCpKeys > wave_kv_lo)) continue;
    // piece c of a row lies at position c ^ (the row's own bits): a read's place is the first one's with a constant's bits
    // turned (worked out in every tile anew: kept over the loop they would not fit the registers)
    uint32_t k_at = stage * kCpStage + jk * (D * 2) + (h ^ (jk & 15)) * 16, v_at = stage * kCpStage + kCpKeys * D * 2 + j * (kCpKeys * 2) + (h ^ ((j >> 1) & 7)) * 16;
    asm volatile("" : "+v"(k_at), "+v"(v_at));

    f32x16_t st[2];
    {
      bf16x8_t kop[2][D / 16];
#pragma unroll
      for (int s = 0; s < D / 16; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          kop[t][s] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(lds_all + (k_at ^ (32 * s)) + 32 * t * (D * 2)));
        }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) st[t][r] = 0.f;
#pragma unroll
      for (int s = 0; s < D / 16; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t) st[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kop[t][s], qreg[s], st[t], 0, 0, 0);
      // a read four products ahead of the product that needs it
      constexpr int kAhead = 4, kOps = 2 * (D / 16);
      __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);
#pragma unroll
      for (int i = 0; i < kOps - kAhead; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, kAhead, 0);
    }
    const bool masked = key_base + kCpKeys - 1 > wave_pos_min || key_base < wave_win_lo;   // not every row sees every key
    const int first_key = key_base + 8 * h;    // st[t][r] is key first_key + 32 t + 16 (r / 8) + r % 8
    // cap, penalty and mask of the row's scores, eight keys in a row at a time (more at once would leave the registers)
    bool poly = false;
    if (!masked && a.cap > 0.f) {
      float most = 0.f;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) most = fmaxf(most, fabsf(st[t][r]));
      poly = __builtin_amdgcn_ballot_w64(!(most <= within)) == 0;
    }
    const int entry = PEN == 1 ? (span - 1 - (my_pos - first_key)) * kCpTableGroup + my_head % kCpTableGroup : 0;
    auto far_of = [&](int off) { return pen1 * __builtin_amdgcn_logf(1.0f + pen2 * static_cast<float>(my_pos - first_key - off)); };
    if (poly) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int run = 0; run < 2; ++run) {
          const int off = 32 * t + 16 * run;      // st[t][8 run + i] is key first_key + off + i
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const float x = st[t][8 * run + i], u = x * x, c = fmaf(fmaf(fmaf(fmaf(c4, u, c3), u, c2), u, c1), u, scale2);
            const float far = PEN == 1 ? table_lds[entry + (off + i) * kCpTableGroup] : PEN == 2 ? far_of(off + i) : 0.f;
            st[t][8 * run + i] = PEN ? fmaf(x, c, -far) : x * c;
          }
        }
    } else {
      const int lo = a.window > 0 ? my_pos - a.window + 1 : 0;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int run = 0; run < 2; ++run) {
          const int off = 32 * t + 16 * run;
          __builtin_amdgcn_sched_barrier(0);
          float x[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) x[i] = st[t][8 * run + i];
          if (a.cap > 0.f) {
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = fmaf(-2.0f * cap2, __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x[i] * to_exp)), cap2);
          } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] *= scale2;
          }
          if (PEN == 2)
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] -= far_of(off + i);
          if (!masked) {
            if (PEN == 1)
#pragma unroll
              for (int i = 0; i < 8; ++i) x[i] -= table_lds[entry + (off + i) * kCpTableGroup];
          } else {   // (a key that the row does not see lies outside the table)
            if (PEN == 1)
#pragma unroll
              for (int i = 0; i < 8; ++i) x[i] -= table_lds[min(max(entry + (off + i) * kCpTableGroup, 0), span * kCpTableGroup - 1)];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const int key = first_key + off + i;
              x[i] = (key >= lo) & (key <= my_pos) ? x[i] : -INFINITY;
            }
          }
#pragma unroll
          for (int i = 0; i < 8; ++i) st[t][8 * run + i] = x[i];
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    float bmax = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) bmax = fmaxf(bmax, st[t][r]);
    {
      const LanePair both = across32(bmax);
      bmax = fmaxf(both.lo, both.hi);
    }
    // m is what the row's exponentials are taken from, not its exact maximum: it moves when that has grown by more than kCpLazyBits
    const float m_new = bmax > m + kCpLazyBits ? bmax : m;
    const float m_use = m_new == -INFINITY ? 0.f : m_new;   // a row that has seen no key yet
    float psum = 0.f;
    bf16x8_t pb[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        u32x4_t packed;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float p0 = __builtin_amdgcn_exp2f(st[t][8 * u + 2 * e] - m_use), p1 = __builtin_amdgcn_exp2f(st[t][8 * u + 2 * e + 1] - m_use);
          psum += p0 + p1;
          packed[e] = pack_bf16x2(p0, p1);
        }
        pb[t][u] = __builtin_bit_cast(bf16x8_t, packed);
      }
    const float alpha = __builtin_amdgcn_exp2f(m - m_use);
    l = l * alpha + psum;      // of the lane's own keys: the halves of a row meet at the end
    if (__builtin_amdgcn_ballot_w64(m_new > m) != 0) {
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
    }
    m = m_new;

    // O^T += V^T . P^T, 16 keys a step
    __builtin_amdgcn_sched_barrier(0);   // (the values' reads stay behind the scores' registers)
    auto values = [&](int k, int dt) {
      return *reinterpret_cast<const u32x4_t*>(lds_all + (v_at ^ (32 * k)) + 32 * dt * (kCpKeys * 2));
    };
    if (masked) {
      // a value that no row of the wave sees may be anything, also NaN, and 0 * NaN is NaN
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        u32x4_t seen = {~0u, ~0u, ~0u, ~0u};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int key = first_key + 16 * k + e;
          if (key < wave_kv_lo || key >= wave_kv_hi) seen[e / 2] &= (e & 1) ? 0x0000ffffu : 0xffff0000u;
        }
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
          o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, values(k, dt) & seen), pb[k / 2][k % 2], o[dt], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      u32x4_t vop[4][D / 32];
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt) vop[k][dt] = values(k, dt);
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
          o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, vop[k][dt]), pb[k / 2][k % 2], o[dt], 0, 0, 0);
      constexpr int kAhead = 4, kOps = 4 * (D / 32);
      __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 1);
#pragma unroll
      for (int i = 0; i < kOps - kAhead; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, kAhead, 1);
    }
  }
  const LanePair both = across32(l);
  l = both.lo + both.hi;

  // o[dt][r] is O^T[d = 32 dt + 8 (r / 4) + 4 h + r % 4][this lane's row]
  if (!row_ok) return;
  const float inv_l = a.out_scale / l;
  bf16* op = a.out + static_cast<int64_t>(row0 + my_tok) * a.o_stride + my_head * D;
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      u32x2_t w;
      w[0] = pack_bf16x2(o[dt][4 * q] * inv_l, o[dt][4 * q + 1] * inv_l);
      w[1] = pack_bf16x2(o[dt][4 * q + 2] * inv_l, o[dt][4 * q + 3] * inv_l);
      *reinterpret_cast<u32x2_t*>(op + 32 * dt + 8 * q + 4 * h) = w;
    }
}

// Whether the kernel takes a step of these sizes.  Groups of two heads and more, by powers of two: a wave's 32 rows are then a
// half, a quarter, ... of sixteen tokens of the portion, and a value that is no number stays in the block of sixteen rows that sees it.
inline bool cap_portions_take(const CapArgs& a) {
  const int group = a.nq / a.nkv;
  return a.Dk == kCpD && a.Dv == kCpD && group >= 2 && (group & (group - 1)) == 0 && (a.page_size & (a.page_size - 1)) == 0 && a.chunk == 0 &&
         a.keep_first == 0 && a.sink == nullptr;
}

template <int PEN>
inline int launch_cap_portions(const CapArgs& a, int blocks, hipStream_t s) {
  constexpr int kBytes = 2 * kCpStage + (PEN == 1 ? kCpTable : 0);
  static OnceADevice asked;
  if (const int e = ask_lds(asked, kBytes, {reinterpret_cast<const void*>(&cap_portions_kernel<PEN>)})) return e;
  cap_portions_kernel<PEN><<<static_cast<unsigned>(blocks) * a.nkv, kCpWaves * kWave, kBytes, s>>>(a);
  return launch_status();
}

}  // namespace arle
