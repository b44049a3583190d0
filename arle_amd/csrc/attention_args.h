// What the attention kernels of attention_mfma.hip share: vector types, the launch's arguments, small helpers.
#pragma once
#include "common.h"

namespace arle {


typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct AttnArgs {
  const uint16_t* q;
  int64_t q_stride;
  uint16_t* out;
  int64_t o_stride;
  float* ws_o;   // [segment * ws_rows + token of the segment][q head][split][D]   (splits > 1)
  float* ws_ml;  // [segment * ws_rows + token of the segment][q head][split][2]
  const uint16_t* k_pages;  // [page][kv head][slot][D]
  const uint16_t* v_pages;  // [page][kv head][D][slot]
  const int* block_table;
  int table_stride;
  const int* seg_row0;   // [segments + 1] first token row of each segment
  const int* seg_slot;   // [segments]
  const int* seg_start;  // [segments] position of a segment's first token
  int nq, nkv, D, P;
  int p_shift;  // log2(P): page sizes are powers of two, so / and % by P are a shift and a mask
  float scale_log2;
  int window;  // 0: all earlier keys
  const float* sink;   // [q heads] or null: exp(sink_h) joins the softmax's denominator, with no value behind it
  float out_scale;     // a factor on the output, in 32 bits
  int splits;
  int segments;        // PREP with splits: how many segments share the waves of a kv head (gridDim.z of them)
  int* ws_plan;        // PREP with splits: [segments][2] a segment's first wave and its number of waves, then
                       // [waves][8] every wave's DecodeShare
  int plan_made;       // the plan is there already (an earlier layer of the same step made it); 0: this launch makes it
  int ws_rows;   // token rows that the split-KV workspace holds for a segment
  int portion_splits;  // parts into which the LDS kernel cuts the keys of a row block (1: whole; it writes out)
  float* pws_o;        // [token row][q head][part][D]   (portion_splits > 1)
  float* pws_ml;       // [token row][q head][part][2]
  int rows_max;  // the streaming kernel skips segments with more rows than this (0: takes all)
  long long plan_token;  // names the step for the portions kernels' list of work (0: no name, plan every time)
  // The kernel that prepares q, k and v itself (PREP; steps of single decoded tokens): the fused q|k|v projection
  // comes as a stack of float32 partial products [prep_n][token rows][(nq + 2 nkv) D], q is unused.
  const void* prep_parts;   // float32, or with prep_bf16 the projection itself in bfloat16 (prep_n 1)
  int prep_bf16;
  int prep_n;
  int64_t prep_part_stride, prep_row_stride;  // elements between the parts, and between the rows of a part
  const void* prep_qw;   // per-head norm weights [D] of q and k (null: no norm), float32 if prep_w_f32 else bfloat16
  const void* prep_kw;
  int prep_w_f32;
  const float* prep_cos;  // [positions][prep_rot / 2]
  const float* prep_sin;
  int prep_rot;           // rotated width: 0, or a multiple of 64 up to D
  float prep_eps;
  uint16_t* prep_k_pages;  // the pages again, to write the new token's key and value into
  uint16_t* prep_v_pages;
};

__device__ __forceinline__ bf16x8 load_bf16x8(const uint16_t* p) {
  return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p));
}

__device__ __forceinline__ bf16x8 zero_bf16x8() {
  uint4 z = {0u, 0u, 0u, 0u};
  return __builtin_bit_cast(bf16x8, z);
}

// The factor that turns a row's summed values into its output: m is what its exponentials (of base 2) are taken from, l their sum.
__device__ __forceinline__ float row_factor(const float* sink, float out_scale, int head, float m, float l) {
  if (sink) l += exp2f(sink[head] * 1.4426950408889634f - m);
  return l > 0.f ? out_scale / l : 0.f;
}

// Inclusive sum (or maximum) over the lanes 0 .. lane of a wave of 64, of values that are not negative: shifts inside
// the rows of 16, then a row's total handed on to the next ones; lane 63 holds the whole wave's.
#define ARLE_PREFIX(NAME, JOIN)                                                                              \
  __device__ __forceinline__ int NAME(int v) {                                                               \
    int u;                                                                                                   \
    u = __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false), v = JOIN; /* row_shr 1, 2, 4, 8 */        \
    u = __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false), v = JOIN;                                 \
    u = __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false), v = JOIN;                                 \
    u = __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false), v = JOIN;                                 \
    u = __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false), v = JOIN; /* lane 15 of a row to the next */ \
    u = __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false), v = JOIN; /* lane 31 to the upper half */ \
    return v;                                                                                                \
  }
ARLE_PREFIX(wave_prefix_sum, v + u)
ARLE_PREFIX(wave_prefix_max, max(v, u))
#undef ARLE_PREFIX

// How the blocks of 32 keys of a step of single decoded tokens are shared out over the `waves` waves that a kv head
// gets: every wave takes up to `per` blocks of one segment, per being the smallest number with which all segments'
// waves are no more than there are and no segment has more than 64 (which is what the merge takes).  Equal contexts
// get what an even split of each would give them.  waves is at least the number of segments.
struct DecodeShare {
  int seg, split, count;   // the wave's segment (-1: none), its place among the segment's waves, how many those are
  int first;               // the segment's first wave
  int per;
  int start, slot;         // the segment's position and its row of the block table
  int unused;
};
static_assert(sizeof(DecodeShare) == 8 * sizeof(int), "a plan keeps eight numbers a wave");
__device__ __forceinline__ int decode_blocks(int start, int window) {   // blocks of 32 that hold a key which the token sees
  const int lo = window > 0 ? max(0, start - window + 1) : 0;
  return start / 32 + 1 - lo / 32;
}
__device__ __forceinline__ DecodeShare decode_share(const int* seg_start, const int* seg_slot, int segments, int window, int waves,
                                                    int wave) {
  const int lane = threadIdx.x & (kWave - 1);
  // segment `at + lane`: up to 64 of them are one load, kept; further ones are read again where they are needed
  const int start0 = seg_start[min(lane, segments - 1)], slot0 = seg_slot[min(lane, segments - 1)];
  const int blocks0 = lane < segments ? decode_blocks(start0, window) : 0;
  auto blocks_at = [&](int at) {
    const int got = seg_start[min(at + lane, segments - 1)];
    return at + lane < segments ? decode_blocks(got, window) : 0;
  };
  auto last = [](int v) { return __builtin_amdgcn_readlane(v, kWave - 1); };
  int total = last(wave_prefix_sum(blocks0)), most = last(wave_prefix_max(blocks0));
  for (int at = kWave; at < segments; at += kWave) {
    const int b = blocks_at(at);
    total += last(wave_prefix_sum(b));
    most = max(most, last(wave_prefix_max(b)));
  }
  DecodeShare s;
  s.per = max(max((total + waves - 1) / waves, (most + kWave - 1) / kWave), 1);
  int mine0, incl0;
  for (;; ++s.per) {   // ends: with per = most a segment is one wave
    mine0 = (blocks0 + s.per - 1) / s.per;
    incl0 = wave_prefix_sum(mine0);
    int need = last(incl0);
    for (int at = kWave; at < segments; at += kWave) need += last(wave_prefix_sum((blocks_at(at) + s.per - 1) / s.per));
    if (need <= waves || s.per >= most) break;
  }
  s.seg = -1;
  s.split = s.count = s.first = s.start = s.slot = s.unused = 0;
  int before = 0;
  for (int at = 0; at < segments; at += kWave) {
    const int mine = at == 0 ? mine0 : (blocks_at(at) + s.per - 1) / s.per;
    const int incl = at == 0 ? incl0 : wave_prefix_sum(mine);
    const unsigned long long past = __ballot(before + incl > wave);
    if (past != 0) {   // the first segment whose waves reach beyond this one
      const int l = __builtin_ctzll(past);
      s.seg = at + l;
      s.count = __builtin_amdgcn_readlane(mine, l);
      s.first = before + __builtin_amdgcn_readlane(incl, l) - s.count;
      s.split = wave - s.first;
      s.start = at == 0 ? __builtin_amdgcn_readlane(start0, l) : seg_start[s.seg];
      s.slot = at == 0 ? __builtin_amdgcn_readlane(slot0, l) : seg_slot[s.seg];
      return s;
    }
    before += last(incl);
  }
  return s;
}

__device__ __forceinline__ float group_max4(float v) {  // over the 4 lanes i, i+16, i+32, i+48
  const LanePair near = across16(v), far = across32(fmaxf(near.lo, near.hi));
  return fmaxf(far.lo, far.hi);
}
__device__ __forceinline__ float group_sum4(float v) {
  const LanePair near = across16(v), far = across32(near.lo + near.hi);
  return far.lo + far.hi;
}

}  // namespace arle
