// Token selection from rows of 32-bit logits: argmax, and temperature sampling
// with min-p / top-k / top-p truncation; plus the repetition / frequency /
// presence penalties applied to logits beforehand.
//
// reference counterparts: crates/cuda-kernels/csrc/misc/sampling.cu:27-87,252-317
// (argmax: first maximum in index order) and :327-596 (temperature -> softmax ->
// top-k -> renormalise -> top-p -> renormalise -> inverse CDF with a uniform u
// drawn on the host); penalties infer/src/sampler.rs:100-140.
//
// Differences kept on purpose: the top-k and top-p thresholds are found exactly, ten or
// eleven bits of the bit pattern of the (non-negative) probabilities at a time, from
// histograms filled with integer atomics, instead of 32 halvings of a float interval;
// each thread owns a contiguous run of the vocabulary so the inverse CDF walks tokens
// in index order; one launch serves many rows with per-row parameters; and the
// log-probability of a chosen token (the reference has it for greedy rows only,
// sampling.cu:252-317) is a kernel of its own that serves greedy and sampled rows.
#include "common.h"
#include <cstring>
#include <type_traits>

namespace arle {

constexpr int kSampThreads = 1024;
constexpr int kSampWaves = kSampThreads / kWave;

struct ArgMax {
  float v;
  int i;
};

__device__ __forceinline__ ArgMax better(ArgMax a, ArgMax b) {
  // larger value wins; equal values: smaller index wins
  if (b.v > a.v || (b.v == a.v && b.i < a.i)) return b;
  return a;
}

__device__ __forceinline__ ArgMax block_argmax(ArgMax a, ArgMax* lds /* [kSampWaves] */) {
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    ArgMax o;
    o.v = __shfl_xor(a.v, off, kWave);
    o.i = __shfl_xor(a.i, off, kWave);
    a = better(a, o);
  }
  const int wave = threadIdx.x / kWave;
  if ((threadIdx.x % kWave) == 0) lds[wave] = a;
  __syncthreads();
  ArgMax r = lds[0];
  for (int i = 1; i < kSampWaves; ++i) r = better(r, lds[i]);
  __syncthreads();
  return r;
}

__device__ __forceinline__ ArgMax row_argmax(const float* x, int n, ArgMax* lds) {
  ArgMax a;
  a.v = -INFINITY;
  a.i = 0x7fffffff;
  for (int i = threadIdx.x; i < n; i += kSampThreads) {
    ArgMax c;
    c.v = x[i];
    c.i = i;
    // NaN never wins a comparison; a row of NaNs yields index 0 below.
    a = better(a, c);
  }
  ArgMax r = block_argmax(a, lds);
  if (r.i == 0x7fffffff) r.i = 0;
  return r;
}

__global__ __launch_bounds__(kSampThreads) void argmax_rows_kernel(const float* __restrict__ logits,
                                                                  int vocab, int* __restrict__ out) {
  __shared__ ArgMax lds[kSampWaves];
  const float* x = logits + static_cast<int64_t>(blockIdx.x) * vocab;
  ArgMax r = row_argmax(x, vocab, lds);
  if (threadIdx.x == 0) out[blockIdx.x] = r.i;
}

// A row cut into gridDim.x chunks, so that a few rows still fill the chip: every workgroup leaves the best
// (value, index) of its chunk in parts[row][chunk], and argmax_merge_kernel picks among them by the same rule.
constexpr int kChunkThreads = 256;

// clear_a, clear_b (null: nothing): so many 16-byte pieces a row that a sampling call wants zeroed, a row's chunks in turn.
struct ClearRows {
  uint4* a;
  uint4* b;
  int a_pieces, a_stride, b_pieces, b_stride;   // to clear, and from row to row
};

__global__ __launch_bounds__(kChunkThreads) void argmax_chunks_kernel(const float* __restrict__ logits, int vocab,
                                                                     int chunk_len, ArgMax* __restrict__ parts, const ClearRows clear) {
  __shared__ ArgMax lds[kChunkThreads / kWave];
  const int row = blockIdx.y, chunk = blockIdx.x;
  for (int i = chunk * kChunkThreads + static_cast<int>(threadIdx.x); i < clear.a_pieces; i += gridDim.x * kChunkThreads)
    clear.a[static_cast<int64_t>(row) * clear.a_stride + i] = uint4{0u, 0u, 0u, 0u};
  for (int i = chunk * kChunkThreads + static_cast<int>(threadIdx.x); i < clear.b_pieces; i += gridDim.x * kChunkThreads)
    clear.b[static_cast<int64_t>(row) * clear.b_stride + i] = uint4{0u, 0u, 0u, 0u};
  const float* x = logits + static_cast<int64_t>(row) * vocab;
  const int begin = chunk * chunk_len, end = min(vocab, begin + chunk_len);
  ArgMax a;
  a.v = -INFINITY;
  a.i = 0x7fffffff;
  auto take = [&](float v, int i) {
    ArgMax c;
    c.v = v;
    c.i = i;
    a = better(a, c);
  };
  // chunk_len is a multiple of 4: with a 16-byte aligned row, four logits a load
  if (reinterpret_cast<uintptr_t>(x) % 16 == 0) {
    const int whole = begin + (max(end - begin, 0) & ~3);
    for (int i = begin + 4 * static_cast<int>(threadIdx.x); i < whole; i += 4 * kChunkThreads) {
      const float4 v = *reinterpret_cast<const float4*>(x + i);
      take(v.x, i);
      take(v.y, i + 1);
      take(v.z, i + 2);
      take(v.w, i + 3);
    }
    for (int i = whole + static_cast<int>(threadIdx.x); i < end; i += kChunkThreads) take(x[i], i);
  } else {
    for (int i = begin + static_cast<int>(threadIdx.x); i < end; i += kChunkThreads) take(x[i], i);
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    ArgMax o;
    o.v = __shfl_xor(a.v, off, kWave);
    o.i = __shfl_xor(a.i, off, kWave);
    a = better(a, o);
  }
  if (threadIdx.x % kWave == 0) lds[threadIdx.x / kWave] = a;
  __syncthreads();
  if (threadIdx.x == 0) {
    ArgMax r = lds[0];
    for (int i = 1; i < kChunkThreads / kWave; ++i) r = better(r, lds[i]);
    parts[static_cast<int64_t>(row) * gridDim.x + chunk] = r;
  }
}

// What a sampling call of rows with a small top_k wants of the logits: the largest of every 64 tokens of a chunk (a NaN is no
// candidate; -inf of a group without tokens or with NaNs alone).  One read of the logits, kAhead pieces of 16 bytes a lane on
// their way at once: 64 rows of 151,936 8.6 us, which with the launch's ramp is what reading 39 MB takes (11.0 with the
// index of every chunk's largest beside it, which only greedy rows want and find in one group).
__device__ __forceinline__ float row16_max(float v);
__global__ __launch_bounds__(kChunkThreads) void group_max_kernel(const float* __restrict__ logits, int vocab, int chunk_len, int groups,
                                                                  float* __restrict__ group_max) {
  constexpr int kAhead = 5, kTokens = 64;
  const int row = blockIdx.y, chunk = blockIdx.x, lane = threadIdx.x & (kWave - 1);
  const int begin = chunk * chunk_len, len = min(vocab - begin, chunk_len);   // len: zero or less behind the row's end
  const float* x = logits + static_cast<int64_t>(row) * vocab + begin;
  float* gm = group_max + (static_cast<int64_t>(row) * gridDim.x + chunk) * groups;
  const bool wide = reinterpret_cast<uintptr_t>(x) % 16 == 0;
  for (int base = 4 * static_cast<int>(threadIdx.x); base < groups * kTokens; base += 4 * kChunkThreads * kAhead) {
    float4 v[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const int at = base + 4 * kChunkThreads * j;
      v[j] = float4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      if (wide && at + 4 <= len) {
        v[j] = *reinterpret_cast<const float4*>(x + at);
      } else {
        if (at < len) v[j].x = x[at];
        if (at + 1 < len) v[j].y = x[at + 1];
        if (at + 2 < len) v[j].z = x[at + 2];
        if (at + 3 < len) v[j].w = x[at + 3];
      }
    }
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const int at = base + 4 * kChunkThreads * j;
      // -inf among them: fmaxf of two NaNs is one
      const float most = row16_max(fmaxf(fmaxf(fmaxf(v[j].x, -INFINITY), fmaxf(v[j].y, -INFINITY)), fmaxf(fmaxf(v[j].z, -INFINITY), fmaxf(v[j].w, -INFINITY))));
      if ((lane & 15) == 0 && at < groups * kTokens) gm[at / kTokens] = most;
    }
  }
}

__global__ __launch_bounds__(kWave) void argmax_merge_kernel(const ArgMax* __restrict__ parts, int chunks,
                                                             int* __restrict__ out) {
  const ArgMax* p = parts + static_cast<int64_t>(blockIdx.x) * chunks;
  ArgMax a;
  a.v = -INFINITY;
  a.i = 0x7fffffff;
  for (int c = threadIdx.x; c < chunks; c += kWave) a = better(a, p[c]);
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    ArgMax o;
    o.v = __shfl_xor(a.v, off, kWave);
    o.i = __shfl_xor(a.i, off, kWave);
    a = better(a, o);
  }
  // a row of NaNs (no value ever wins) yields index 0, as in the one-workgroup kernel
  if (threadIdx.x == 0) out[blockIdx.x] = a.i == 0x7fffffff ? 0 : a.i;
}

// ---------------------------------------------------------------------------------------------
// Temperature sampling with min-p, top-k and top-p, many workgroups a row.
//
// e[i] = exp(x[i] / T - max) is kept unnormalised: every filter is "keep e[i] >= some threshold", and since
// e >= 0 the order of the values is the order of their bit patterns.
//   min_p:  e >= min_p                       (the largest e is exp(0) = 1)
//   top_k:  e >= the k-th largest e           (ties of the k-th stay)
//   top_p:  e >= the largest t whose kept mass reaches top_p of the mass kept so far
// The k-th largest value and the mass threshold are found digit by digit, 10 + 11 + 10 bits: a pass over the
// row fills a histogram with the next digit of the elements that match the digits found so far; scanning the bins
// from the top gives the digit in which the count (the mass) is reached.  Counts are integers and masses are summed as
// 64-bit fixed-point numbers (e * 2^40), so the histograms do not depend on the order in which workgroups add to
// them, and every workgroup that reads them finds the same digits.  The token is then drawn by the inverse CDF in
// token order: u * (kept mass) falls into a chunk, and inside the chunk into a token.
//
// What bounds a call of few rows is the chain of kernels, of many rows reading e once a pass.  So:
//   - the pass that makes e also fills the first histogram, of top_k, or of top_p where the row has no top_k;
//   - it leaves the largest e of every 64 tokens; the later passes read only groups that reach the threshold's known
//     digits (of 50 kept tokens in 151,936 at most 50 groups of 2,374);
//   - every workgroup finds the next digit by itself, with all its threads, from one histogram: the digits before it
//     and what is left to reach stand in the row's slot of the pass before.
// 64 rows of 151,936 logits, kernels back to back: with top_k 50 and top_p 0.9 184 us -> 98 us, top_p alone 136 -> 83,
// top_k alone 84 -> 71; one row 142 -> 80 (before: digits of eight bits, every pass read the whole row and scanned all
// digits before its own with one wave, and one thread added up 256 bins).
constexpr int kSelThreads = kChunkThreads;
constexpr int kSelWaves = kSelThreads / kWave;
constexpr int kGroup = kWave;                   // tokens that share a largest e
constexpr float kMassScale = 1099511627776.0f;  // 2^40
constexpr int kBins0 = 1024, kBins1 = 2048, kBins2 = 1024;   // a non-negative float has no bit 31: ten bits lead
constexpr int kRowBins = kBins0 + kBins1 + kBins2;

// What a pass has found of a row's threshold.
struct Slot {
  unsigned long long rest;   // rank (mass) still to reach inside the bin of the last digit
  unsigned int prefix;       // the digits so far
  unsigned int floor;        // what min_p (and, once it is known, top_k) asks of e
  unsigned int open;         // 1: the row does not reach the rank (the mass): everything above the floor stays
  unsigned int unused;
};
// The passes, in order.  FIRST, SECOND: digits 0 and 1 of top_k, or of top_p for a row without top_k.  FLOOR: the last
// digit of top_k, and top_p's first histogram.  THIRD, FOURTH: digits 0 and 1 of top_p for a row with top_k.
enum Pass { kFirst = 0, kSecond = 1, kFloor = 2, kThird = 3, kFourth = 4, kPasses = 5 };

struct SampleArgs {
  const float* logits;
  float* e;  // [rows, vocab]
  int vocab, chunk_len, chunks, groups;   // groups of kGroup tokens in a chunk
  const float* temperature;
  const int* top_k;
  const float* top_p;
  const float* min_p;
  const float* u;
  const ArgMax* part_max;          // [rows, chunks]
  unsigned int* hist_k;            // [rows, kRowBins] counts
  unsigned long long* hist_p;      // [rows, kRowBins] masses
  Slot* slots;                     // [rows, kPasses]
  float* group_max;                // [rows, chunks, groups]
  float* chunk_mass;               // [rows, chunks]
  unsigned int* threshold;         // [rows] bits of the final threshold
  int use_top_k, use_top_p;        // 0: no row of this call uses the filter (its passes are not launched)
  int* out;
  int* out_host;                   // pinned host memory that takes the tokens as well, or null
};

// A row's token, by one thread.  The copy for the host is a store over the bus that nothing waits for but the launch's end; as a copy behind the
// kernel it was a launch more and 9 us (64 rows of 151,936 logits, top_k 50, one call among others: 40.8 us with the copy, 34.3 without).
__device__ __forceinline__ void leave_token(const SampleArgs& a, int row, int token) {
  a.out[row] = token;
  if (a.out_host != nullptr) a.out_host[row] = token;
}

// The e of a logit, the same bits wherever it is computed; mx: the row's largest logit over the temperature.
__device__ __forceinline__ float weight_of(float x, float inv_t, float mx) { return expf(fmaf(x, inv_t, -mx)); }

// Where a row's e are read: in memory, as sample_exp_kernel left them with the largest e of every group, or made from the logits,
// with the groups' largest logits (group_max_kernel).  A larger logit may have an e that is smaller by the
// rounding of two exponentials (expf is off by one unit at most): a group is looked at where its largest is kSlack units short.
struct StoredWeights {
  const float* e;
  __device__ __forceinline__ float at(int i) const { return e[i]; }
  __device__ __forceinline__ float of(float stored) const { return stored; }
  __device__ __forceinline__ bool group_reaches(float most, unsigned int lower) const { return __float_as_uint(most) >= lower; }
  __device__ __forceinline__ const float* row() const { return e; }
};
struct MadeWeights {
  static constexpr unsigned int kSlack = 4;
  const float* x;
  float inv_t, mx;
  __device__ __forceinline__ float at(int i) const { return weight_of(x[i], inv_t, mx); }
  __device__ __forceinline__ float of(float logit) const { return weight_of(logit, inv_t, mx); }
  __device__ __forceinline__ bool group_reaches(float most, unsigned int lower) const {
    const float e = of(most);
    return e >= 0.f && __float_as_uint(e) + kSlack >= lower;
  }
  __device__ __forceinline__ const float* row() const { return x; }
};

struct RowParams {
  float inv_t, min_p, top_p;
  int k;
  bool greedy, k_active, p_active;
};

__device__ __forceinline__ RowParams row_params(const SampleArgs& a, float temp, int top_k, float top_p, float min_p) {
  RowParams r;
  r.k = top_k;
  r.top_p = top_p;
  r.min_p = min_p;
  // Greedy rule of the reference: (T <= 0 or top_k == 1) and no stochastic filter.
  r.greedy = (temp <= 0.f || r.k == 1) && r.top_p >= 1.f && r.min_p <= 0.f;
  r.inv_t = temp > 0.f ? 1.0f / temp : 1.0f;
  r.k_active = a.use_top_k && r.k > 0 && r.k < a.vocab;
  r.p_active = a.use_top_p && r.top_p < 1.f;
  return r;
}
__device__ __forceinline__ RowParams row_params(const SampleArgs& a, int row) {
  return row_params(a, a.temperature[row], a.top_k[row], a.top_p[row], a.min_p[row]);
}

__device__ __forceinline__ unsigned int min_p_bits(const RowParams& r) {
  return r.min_p > 0.f ? __float_as_uint(r.min_p) : 0u;
}

__device__ __forceinline__ unsigned int shfl_any(unsigned int v, int src) { return __shfl(v, src, kWave); }
__device__ __forceinline__ unsigned long long shfl_any(unsigned long long v, int src) {
  const unsigned int lo = __shfl(static_cast<unsigned int>(v), src, kWave);
  const unsigned int hi = __shfl(static_cast<unsigned int>(v >> 32), src, kWave);
  return (static_cast<unsigned long long>(hi) << 32) | lo;
}

struct SelectLds {
  unsigned long long wave_total[kSelWaves];
  unsigned long long rest;
  unsigned int digit, ok;
};

// What top_p asks of the kept mass, as a fixed-point number (at least 1).
__device__ __forceinline__ unsigned long long top_p_need(float top_p, unsigned long long total) {
  const unsigned long long need = static_cast<unsigned long long>(static_cast<double>(top_p) * static_cast<double>(total));
  return need < 1ull ? 1ull : need;
}

// The digit in which a histogram of BINS bins, counted from the top, reaches need(total) >= 1, and what is left to reach
// inside that bin.  False when the whole histogram does not.  Every thread of the workgroup calls it.
template <int BINS, typename T, typename Need>
__device__ __forceinline__ bool select_digit(const T* __restrict__ hist, Need need_of, SelectLds& lds, unsigned int& digit, T& rest) {
  constexpr int kPer = BINS / kSelThreads;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  T m[kPer];
  T own = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    m[j] = hist[kPer * threadIdx.x + j];
    own += m[j];
  }
  T suffix = own;  // over the bins of this thread and of the wave's threads above it
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const T other = shfl_any(suffix, min(lane + off, kWave - 1));
    if (lane + off < kWave) suffix += other;
  }
  if (lane == 0) lds.wave_total[wave] = static_cast<unsigned long long>(suffix);
  if (threadIdx.x == 0) lds.ok = 0u;
  __syncthreads();
  T above = suffix - own, total = 0;
#pragma unroll
  for (int w = 0; w < kSelWaves; ++w) {
    const T t = static_cast<T>(lds.wave_total[w]);
    total += t;
    if (w > wave) above += t;
  }
  const T need = need_of(total);
  if (above < need && above + own >= need) {   // one thread: the sums grow from thread to thread downwards
    unsigned int at = 0u;
    T left = 0;
#pragma unroll
    for (int j = kPer - 1; j >= 0; --j) {
      if (left == 0 && above + m[j] >= need) {
        at = kPer * threadIdx.x + j;
        left = need - above;  // >= 1
      }
      above += m[j];
    }
    lds.digit = at;
    lds.rest = static_cast<unsigned long long>(left);
    lds.ok = 1u;
  }
  __syncthreads();
  const bool ok = lds.ok != 0u;
  digit = lds.digit;
  rest = static_cast<T>(lds.rest);
  __syncthreads();  // lds may be used again
  return ok;
}

// Digit LEVEL of a threshold, from its histogram (the row's kRowBins bins) and what the pass before found.
template <int LEVEL, typename T, typename Need>
__device__ __forceinline__ Slot next_digit(const T* __restrict__ row_bins, Need first_need, Slot s, SelectLds& lds) {
  constexpr int kBins = LEVEL == 0 ? kBins0 : LEVEL == 1 ? kBins1 : kBins2;
  constexpr int kAt = LEVEL == 0 ? 0 : LEVEL == 1 ? kBins0 : kBins0 + kBins1;
  constexpr int kBits = LEVEL == 0 ? 10 : LEVEL == 1 ? 11 : 10;
  if (s.open) return s;  // the same for every thread
  unsigned int digit;
  T rest;
  const T left = static_cast<T>(s.rest);
  const bool ok = select_digit<kBins, T>(row_bins + kAt, [&](T total) { return LEVEL == 0 ? first_need(total) : left; }, lds,
                                         digit, rest);
  if (!ok) {
    s.open = 1u;
  } else {
    s.prefix = LEVEL == 0 ? digit : (s.prefix << kBits) | digit;
    s.rest = static_cast<unsigned long long>(rest);
  }
  return s;
}
template <int LEVEL>
__device__ __forceinline__ Slot next_k(const SampleArgs& a, int row, const RowParams& r, const Slot& s, SelectLds& lds) {
  return next_digit<LEVEL, unsigned int>(a.hist_k + static_cast<int64_t>(row) * kRowBins,
                                         [&](unsigned int) { return static_cast<unsigned int>(r.k); }, s, lds);
}
template <int LEVEL>
__device__ __forceinline__ Slot next_p(const SampleArgs& a, int row, const RowParams& r, const Slot& s, SelectLds& lds) {
  return next_digit<LEVEL, unsigned long long>(a.hist_p + static_cast<int64_t>(row) * kRowBins,
                                               [&](unsigned long long total) { return top_p_need(r.top_p, total); }, s, lds);
}

__device__ __forceinline__ float merged_max(const SampleArgs& a, int row, float* lds /* [kSelWaves] */) {
  float v = -INFINITY;
  for (int c = threadIdx.x; c < a.chunks; c += kSelThreads)
    v = fmaxf(v, a.part_max[static_cast<int64_t>(row) * a.chunks + c].v);
  return block_max<kSelWaves>(v, lds);
}

// Calls take(e) for the tokens of a chunk whose group of 64 reaches `lower` (bits); wave w has the groups w, w + 4, ..,
// in this order, a token a lane: a thread meets the tokens threadIdx.x, threadIdx.x + 256, .. of the chunk.
template <typename Take>
__device__ __forceinline__ void walk_chunk(const SampleArgs& a, int row, int chunk, unsigned int lower, Take take) {
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int begin = chunk * a.chunk_len, len = min(a.vocab - begin, a.chunk_len);
  const float* e = a.e + static_cast<int64_t>(row) * a.vocab + begin;
  const float* gm = a.group_max + (static_cast<int64_t>(row) * a.chunks + chunk) * a.groups;
  const int have = (max(len, 0) + kGroup - 1) / kGroup;
  for (int base = wave; base < have; base += kSelWaves * kWave) {
    const int g = base + kSelWaves * lane;
    const bool live = g < have && __float_as_uint(gm[min(g, have - 1)]) >= lower;
    unsigned long long mask = __ballot(live);
    while (mask != 0ull) {
      float v[4];
      bool in[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int at = mask != 0ull ? __builtin_ctzll(mask) : 0;
        const int i = (base + kSelWaves * at) * kGroup + lane;
        in[j] = mask != 0ull && i < len;
        mask &= mask - 1ull;   // 0 stays 0
        v[j] = in[j] ? e[i] : -1.0f;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (in[j]) take(v[j]);
    }
  }
}

// Adds digit LEVEL of the chunk's tokens that match the slot's digits and reach its floor to the row's histogram.
template <int LEVEL, bool MASS>
__device__ __forceinline__ void fill_bins(const SampleArgs& a, int row, int chunk, const Slot& s, void* lds_bins) {
  using T = std::conditional_t<MASS, unsigned long long, unsigned int>;
  constexpr int kBins = LEVEL == 0 ? kBins0 : LEVEL == 1 ? kBins1 : kBins2;
  constexpr int kAt = LEVEL == 0 ? 0 : LEVEL == 1 ? kBins0 : kBins0 + kBins1;
  constexpr int kHigh = LEVEL == 1 ? 21 : 10, kLow = LEVEL == 0 ? 21 : LEVEL == 1 ? 10 : 0;
  T* bins = static_cast<T*>(lds_bins);
#pragma unroll
  for (int j = 0; j < kBins / kSelThreads; ++j) bins[j * kSelThreads + threadIdx.x] = 0;
  __syncthreads();
  const unsigned int prefix = s.prefix, floor = s.floor;
  walk_chunk(a, row, chunk, LEVEL == 0 ? floor : max(floor, prefix << kHigh), [&](float v) {
    const unsigned int bits = __float_as_uint(v);
    if (!(v >= 0.f && bits >= floor && (LEVEL == 0 || (bits >> kHigh) == prefix))) return;
    const T n = MASS ? static_cast<T>(v * kMassScale) : static_cast<T>(1);
    if (n) atomicAdd(&bins[(bits >> kLow) & (kBins - 1)], n);
  });
  __syncthreads();
  T* to = (MASS ? reinterpret_cast<T*>(a.hist_p) : reinterpret_cast<T*>(a.hist_k)) + static_cast<int64_t>(row) * kRowBins + kAt;
#pragma unroll
  for (int j = 0; j < kBins / kSelThreads; ++j) {
    const T n = bins[j * kSelThreads + threadIdx.x];
    if (n) atomicAdd(to + j * kSelThreads + threadIdx.x, n);
  }
}

__device__ __forceinline__ float row16_max(float v) {   // over the 16 lanes of a row, into all of them
#define ARLE_ROR_MAX(n) \
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + n, 0xf, 0xf, true)));
  ARLE_ROR_MAX(8) ARLE_ROR_MAX(4) ARLE_ROR_MAX(2) ARLE_ROR_MAX(1)
#undef ARLE_ROR_MAX
  return v;
}

// e = exp(x / T - max) for the chunk, the largest e of its groups, and the first histogram: top_k's, or top_p's for a row
// without top_k.  A thread takes four tokens at a time.  Neighbouring tokens fall into the same few bins, so the workgroup
// keeps several copies of the histogram, lane by lane in turn, and adds them up at its end.
__global__ __launch_bounds__(kSelThreads) void sample_exp_kernel(const SampleArgs a) {
  constexpr int kCopiesK = 4, kCopiesP = 2;
  __shared__ float red[kSelWaves];
  __shared__ unsigned long long bins[kCopiesP * kBins0];
  static_assert(sizeof(bins) == kCopiesK * kBins0 * sizeof(unsigned int), "both histograms fill the same LDS");
  const int row = blockIdx.y, chunk = blockIdx.x;
  const RowParams r = row_params(a, row);
  if (r.greedy) return;
  const int lane = threadIdx.x & (kWave - 1);
  const bool by_mass = r.p_active && !r.k_active, any = r.k_active || r.p_active;
  const int begin = chunk * a.chunk_len, len = min(a.vocab - begin, a.chunk_len);
  const float* x = a.logits + static_cast<int64_t>(row) * a.vocab + begin;
  float* e = a.e + static_cast<int64_t>(row) * a.vocab + begin;
  float* gm = a.group_max + (static_cast<int64_t>(row) * a.chunks + chunk) * a.groups;
  const bool wide = reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(e) % 16 == 0;
  auto load = [&](int at) {
    float4 v = {0.f, 0.f, 0.f, 0.f};
    if (wide && at + 4 <= len) return *reinterpret_cast<const float4*>(x + at);
    if (at < len) v.x = x[at];
    if (at + 1 < len) v.y = x[at + 1];
    if (at + 2 < len) v.z = x[at + 2];
    if (at + 3 < len) v.w = x[at + 3];
    return v;
  };
  float4 next = load(4 * static_cast<int>(threadIdx.x));
  if (any)
#pragma unroll
    for (int j = 0; j < kCopiesP * kBins0 / kSelThreads; ++j) bins[j * kSelThreads + threadIdx.x] = 0ull;
  const float mx = merged_max(a, row, red) * r.inv_t;  // the block reduction also orders the LDS writes above
  const unsigned int mp = min_p_bits(r);
  unsigned int* counts = reinterpret_cast<unsigned int*>(bins);
  for (int base = 0; base < len; base += 4 * kSelThreads) {
    const int at = base + 4 * static_cast<int>(threadIdx.x);
    const float4 in = next;
    next = load(at + 4 * kSelThreads);
    const float v[4] = {weight_of(in.x, r.inv_t, mx), weight_of(in.y, r.inv_t, mx), weight_of(in.z, r.inv_t, mx),
                        weight_of(in.w, r.inv_t, mx)};
    float most = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (at + j < len) most = fmaxf(most, v[j]);
    if (wide && at + 4 <= len) {
      *reinterpret_cast<float4*>(e + at) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (at + j < len) e[at + j] = v[j];
    }
    if (any) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const unsigned int bits = __float_as_uint(v[j]);
        if (!(at + j < len && v[j] >= 0.f && bits >= mp)) continue;
        const unsigned int bin = (bits >> 21) & (kBins0 - 1);
        if (by_mass) {
          const unsigned long long n = static_cast<unsigned long long>(v[j] * kMassScale);
          if (n) atomicAdd(&bins[bin * kCopiesP + (lane & (kCopiesP - 1))], n);
        } else {
          atomicAdd(&counts[bin * kCopiesK + (lane & (kCopiesK - 1))], 1u);
        }
      }
    }
    most = row16_max(most);
    if ((lane & 15) == 0 && at < len) gm[at / kGroup] = most;
  }
  if (!any) return;
  __syncthreads();
  for (int bin = threadIdx.x; bin < kBins0; bin += kSelThreads) {
    if (by_mass) {
      unsigned long long n = 0ull;
#pragma unroll
      for (int c = 0; c < kCopiesP; ++c) n += bins[bin * kCopiesP + c];
      if (n) atomicAdd(a.hist_p + static_cast<int64_t>(row) * kRowBins + bin, n);
    } else {
      unsigned int n = 0u;
#pragma unroll
      for (int c = 0; c < kCopiesK; ++c) n += counts[bin * kCopiesK + c];
      if (n) atomicAdd(a.hist_k + static_cast<int64_t>(row) * kRowBins + bin, n);
    }
  }
}

// One pass: the next digit of the row's threshold, and the histogram of the one after it.
template <int PASS>
__global__ __launch_bounds__(kSelThreads) void sample_pass_kernel(const SampleArgs a) {
  __shared__ unsigned long long bins[kBins1];
  __shared__ SelectLds sel;
  const int row = blockIdx.y, chunk = blockIdx.x;
  const RowParams r = row_params(a, row);
  if (r.greedy) return;
  if (PASS >= kFloor ? !(r.k_active && r.p_active) : !(r.k_active || r.p_active)) return;
  Slot* slots = a.slots + static_cast<int64_t>(row) * kPasses;
  Slot s = {0ull, 0u, min_p_bits(r), 0u, 0u};
  if constexpr (PASS > 0) s = slots[PASS - 1];
  if constexpr (PASS == kFirst) s = r.k_active ? next_k<0>(a, row, r, s, sel) : next_p<0>(a, row, r, s, sel);
  if constexpr (PASS == kSecond) s = r.k_active ? next_k<1>(a, row, r, s, sel) : next_p<1>(a, row, r, s, sel);
  if constexpr (PASS == kFloor) {
    s = next_k<2>(a, row, r, s, sel);
    const unsigned int floor = s.open ? s.floor : max(s.floor, s.prefix);
    s = Slot{0ull, 0u, floor, 0u, 0u};
  }
  if constexpr (PASS == kThird) s = next_p<0>(a, row, r, s, sel);
  if constexpr (PASS == kFourth) s = next_p<1>(a, row, r, s, sel);
  if (chunk == 0 && threadIdx.x == 0) slots[PASS] = s;
  if (s.open) return;
  if constexpr (PASS == kFirst || PASS == kSecond) {
    if (r.k_active) fill_bins<PASS == kFirst ? 1 : 2, false>(a, row, chunk, s, bins);
    else fill_bins<PASS == kFirst ? 1 : 2, true>(a, row, chunk, s, bins);
  } else {
    fill_bins<PASS - kFloor, true>(a, row, chunk, s, bins);
  }
}

// The final threshold of the row and the kept mass of every chunk.
__global__ __launch_bounds__(kSelThreads) void sample_mass_kernel(const SampleArgs a) {
  __shared__ SelectLds sel;
  __shared__ float red[kSelWaves];
  const int row = blockIdx.y, chunk = blockIdx.x;
  const RowParams r = row_params(a, row);
  if (r.greedy) return;
  unsigned int thr = min_p_bits(r);
  if (r.k_active || r.p_active) {
    Slot s = a.slots[static_cast<int64_t>(row) * kPasses + (r.k_active && r.p_active ? kFourth : kSecond)];
    s = r.p_active ? next_p<2>(a, row, r, s, sel) : next_k<2>(a, row, r, s, sel);
    thr = s.open ? s.floor : max(s.floor, s.prefix);
  }
  if (chunk == 0 && threadIdx.x == 0) a.threshold[row] = thr;
  float mass = 0.f;
  walk_chunk(a, row, chunk, thr, [&](float v) {
    if (v >= 0.f && __float_as_uint(v) >= thr) mass += v;
  });
  mass = block_sum<kSelWaves>(mass, red);
  if (threadIdx.x == 0) a.chunk_mass[static_cast<int64_t>(row) * a.chunks + chunk] = mass;
}

__device__ __forceinline__ float lane_value(float v, int lane /* the same in every lane */) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

struct PickLds {
  ArgMax best[kSelWaves];
  alignas(16) float part[kSelThreads];
  float chunk_start, target;
  int chunk_of_target, chosen;
};

// What follows is the work of the first kSelThreads threads of a workgroup, whose others, if it has any, come along from barrier to
// barrier.

// A greedy row's token: the first maximum.
__device__ __forceinline__ void pick_greedy(const SampleArgs& a, int row, PickLds& l) {
  ArgMax m;
  m.v = -INFINITY;
  m.i = 0x7fffffff;
  const bool owns = threadIdx.x < kSelThreads;
  for (int c = threadIdx.x; owns && c < a.chunks; c += kSelThreads)
    m = better(m, a.part_max[static_cast<int64_t>(row) * a.chunks + c]);
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    ArgMax o;
    o.v = __shfl_xor(m.v, off, kWave);
    o.i = __shfl_xor(m.i, off, kWave);
    m = better(m, o);
  }
  if (owns && threadIdx.x % kWave == 0) l.best[threadIdx.x / kWave] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    ArgMax t = l.best[0];
    for (int w = 1; w < kSelWaves; ++w) t = better(t, l.best[w]);
    leave_token(a, row, t.i == 0x7fffffff ? 0 : t.i);
  }
}

// The chunk that u * (kept mass) falls into, and the mass in front of it.
__device__ __forceinline__ void find_target(const SampleArgs& a, float u, const float* masses, PickLds& l) {
  if (threadIdx.x < kWave) {   // wave 0: lane l has the masses 4 l .. 4 l + 3; lanes without any add nothing
    const int lane = threadIdx.x;
    float m[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) m[j] = 4 * lane + j < a.chunks ? masses[4 * lane + j] : 0.f;
    const unsigned long long some = __ballot(m[0] > 0.f || m[1] > 0.f || m[2] > 0.f || m[3] > 0.f);
    float total = 0.f;
    for (unsigned long long left = some; left != 0ull; left &= left - 1ull) {
      const int at = __builtin_ctzll(left);
#pragma unroll
      for (int j = 0; j < 4; ++j) total += lane_value(m[j], at);
    }
    const float target = u * total;
    float run = 0.f;
    int at = -1, last = 0;
    float start = 0.f, last_start = 0.f;
    for (unsigned long long left = some; left != 0ull && at < 0; left &= left - 1ull) {
      const int from = __builtin_ctzll(left);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float mass = lane_value(m[j], from);
        if (mass > 0.f) {
          last = 4 * from + j;
          last_start = run;
          if (at < 0 && target < run + mass) {
            at = last;
            start = run;
          }
        }
        run += mass;
      }
    }
    if (lane == 0) {
      l.chunk_of_target = at >= 0 ? at : last;  // u at or past the whole mass (rounding): the last chunk that holds any
      l.chunk_start = at >= 0 ? start : last_start;
      l.target = target;
      l.chosen = -1;
    }
  }
  __syncthreads();
}

// part[t], what thread t's tokens of the chunk weigh, becomes the mass in front of them (in the threads' order).
__device__ __forceinline__ void add_up_parts(PickLds& l, float before) {
  __syncthreads();
  if (threadIdx.x < kWave) {   // wave 0, four threads a lane; lanes without mass add nothing
    const int lane = threadIdx.x;
    const float4 c = *reinterpret_cast<const float4*>(&l.part[4 * lane]);
    float run = before;
    float4 own = {before, before, before, before};
    for (unsigned long long left = __ballot(c.x > 0.f || c.y > 0.f || c.z > 0.f || c.w > 0.f); left != 0ull; left &= left - 1ull) {
      const int from = __builtin_ctzll(left);
      float4 p;
      p.x = run;
      p.y = p.x + lane_value(c.x, from);
      p.z = p.y + lane_value(c.y, from);
      p.w = p.z + lane_value(c.z, from);
      run = p.w + lane_value(c.w, from);
      if (lane == from) own = p;
    }
    *reinterpret_cast<float4*>(&l.part[4 * lane]) = own;
  }
  __syncthreads();
}

// The token by the inverse CDF in token order, from e, the threshold and the chunks' kept masses.
template <typename Weights>
__device__ __forceinline__ void pick_token(const SampleArgs& a, int row, float u, unsigned int thr, const float* masses, const Weights& w, PickLds& l) {
  find_target(a, u, masses, l);
  const int chunk = l.chunk_of_target;
  const float target = l.target, before = l.chunk_start;
  const int begin = chunk * a.chunk_len, end = min(a.vocab, begin + a.chunk_len);
  // thread t owns the tokens [lo, hi) of the chunk, in token order
  const int per = (end - begin + kSelThreads - 1) / kSelThreads;
  const bool owns = threadIdx.x < kSelThreads;
  const int lo = owns ? min(begin + static_cast<int>(threadIdx.x) * per, end) : end, hi = min(lo + per, end);
  auto kept = [&](int i) {
    const float v = w.at(i);
    return (v >= 0.f && __float_as_uint(v) >= thr) ? v : 0.f;
  };
  const float* gm = a.group_max + (static_cast<int64_t>(row) * a.chunks + chunk) * a.groups;
  bool live = false;   // a group that the thread's tokens lie in reaches the threshold
  if (lo < hi)
    for (int g = (lo - begin) / kGroup; g <= (hi - 1 - begin) / kGroup; ++g) live |= w.group_reaches(gm[g], thr);
  float mine = 0.f;
  if (live)
#pragma unroll 4
    for (int i = lo; i < hi; ++i) mine += kept(i);
  if (owns) l.part[threadIdx.x] = mine;
  add_up_parts(l, before);
  const float start = owns ? l.part[threadIdx.x] : 0.f;
  if (target >= start && target < start + mine && hi > lo) {
    float run = start;
    int pick = -1;
    for (int i = lo; i < hi; ++i) {
      run += kept(i);
      if (target < run) {
        pick = i;
        break;
      }
    }
    if (pick < 0) {  // rounding left the target past this thread's end: its last kept token
      for (int i = hi - 1; i >= lo; --i)
        if (kept(i) > 0.f) {
          pick = i;
          break;
        }
    }
    if (pick >= 0) atomicMax(&l.chosen, pick);
  }
  __syncthreads();
  if (l.chosen < 0) {
    // the target lies outside what the threads found (rounding between the two ways of adding): the last kept
    // token of the chunk, or of the row when the chunk holds none
    int last = -1;
    for (int i = begin + static_cast<int>(threadIdx.x); i < end; i += blockDim.x)
      if (kept(i) > 0.f) last = max(last, i);
    __syncthreads();   // everybody has looked at `chosen`
    if (last >= 0) atomicMax(&l.chosen, last);
    __syncthreads();
    if (l.chosen < 0) {
      for (int i = threadIdx.x; i < a.vocab; i += blockDim.x)
        if (kept(i) > 0.f) last = max(last, i);
      __syncthreads();
      if (last >= 0) atomicMax(&l.chosen, last);
      __syncthreads();
    }
  }
  if (threadIdx.x == 0) leave_token(a, row, max(l.chosen, 0));
}

// The token: greedy rows take the first maximum; the others the inverse CDF in token order.
__global__ __launch_bounds__(kSelThreads) void sample_pick_kernel(const SampleArgs a) {
  __shared__ PickLds l;
  const int row = blockIdx.x;
  if (row_params(a, row).greedy) pick_greedy(a, row, l);
  else pick_token(a, row, a.u[row], a.threshold[row], a.chunk_mass + static_cast<int64_t>(row) * a.chunks, StoredWeights{a.e + static_cast<int64_t>(row) * a.vocab}, l);
}

// Rows with a small top_k: everything behind the groups' maxima (group_max_kernel) in one kernel, a workgroup a row.  The
// top_k-th largest of the maxima is a value that top_k tokens reach, and the tokens that do lie in the groups whose maxima do:
// some fifty groups of 2,374 for top_k 50.  Their e are made again from the logits, with the same function, and gathered into
// LDS; nothing else of the row is read and no e is written.  Of more than kDirectMost tokens the threshold's digits come from
// histograms of the list, and what does not reach it goes.  Each of the others is compared with all, which puts the list
// into the order of the tokens, for the chunks' masses and the token, and into that of the values, for the threshold of top_p (and
// gives that of top_k where it is not known yet).  The thresholds are the same values as by the passes (exact, counts and
// fixed-point masses); a chunk's mass is added in the order of sample_mass_kernel's threads
// and waves, a thread's in pick_token's, where what is not kept adds nothing: the same bits, the same token.
// Where more than kManyGroups maxima end in the threshold's value, the workgroup reads the row for the tokens above it: fewer
// than top_k, and their ties are counted and not listed.  A list that overflows all the same (or a row of fewer groups than top_k) is
// told from the row by digits.
// MI355X, rows of 151,936 normal logits, the kernels of a call in us, with the passes of many workgroups / with this kernel.  Spread 2.5
// (over the temperature), top_k 50 and top_p 0.9: one row 37 / 21, 64 rows 73 / 26; top_k 256 39 / 36, 76 / 40.  Spread 0.2: top_k 50 38 /
// 24, 74 / 28; top_k 256 40 / 38, 82 / 44.  Spread 0.05: top_k 50 39 / 24, 90 / 28; top_k 256 41 / 39, 94 / 44.  All logits equal:
// 53 / 69, 236 / 78.  (With a first histogram of all e in front of it, e written to memory and read again: 26, 41 and 39, 54 at
// spread 2.5, 61 and 82 for equal logits.)  The host needs 36 us for a call with one object of parameters, so that a call queued behind others takes 35 us for one row
// and 40 for 64; before 67 and 72.  What a spread row takes is trips through memory and steps in LDS; a flat one is
// bound by what a single workgroup reads, about 10 us a time.
constexpr int kFinishThreads = 1024, kFinishTopK = 256;
constexpr int kFinishMost = 4096, kDirectMost = 256, kKeptMost = 1024, kLiveMost = 4096;
constexpr int kFinishVocab = 1 << 28;      // a group's first token / 4 and its size share a word
static_assert(kFinishTopK <= kDirectMost, "a row that does not reach its rank has fewer tokens than that, and is not looked at by digits");
static_assert(kFinishMost % kFinishThreads == 0 && kKeptMost == kFinishThreads, "whole rounds of the threads, and one of those kept");

struct FinishLds {
  PickLds pick;
  int count, n_live;
  unsigned int threshold, ok, digit, left, found;
  unsigned int wave_total[kFinishThreads / kWave];
  float largest[kFinishThreads / kWave];
  unsigned long long wave_mass_total[kFinishThreads / kWave];
  float masses[256];
  int first[256], behind[256];            // of a chunk: its first token in the list, and the one behind its last
  uint2 raw[kFinishMost];                 // bits and token, as gathered
  union {
    unsigned int live[kLiveMost];         // groups that hold tokens for the list: 64 (first token / 4) + tokens - 1
    unsigned int bins[kBins1];
    struct {
      unsigned int bits[kKeptMost];       // in token order
      int token[kKeptMost];
      unsigned int value[kKeptMost];      // bits in descending order
    } list;
    float wave_mass[256][kSelWaves];
  };
};

// Appends the lanes' entries for which in[j] holds to a list of *count so far: put(place, j), one atomic a wave.
template <int N, typename Put>
__device__ __forceinline__ void append(const bool (&in)[N], int* count, Put put) {
  const int lane = threadIdx.x & (kWave - 1);
  unsigned long long some[N];
  int all = 0;
#pragma unroll
  for (int j = 0; j < N; ++j) some[j] = __ballot(in[j]), all += __builtin_popcountll(some[j]);
  if (all == 0) return;
  int at = 0;
  if (lane == 0) at = atomicAdd(count, all);
  at = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if (in[j]) put(at + __builtin_popcountll(some[j] & ((1ull << lane) - 1ull)), j);
    at += __builtin_popcountll(some[j]);
  }
}

// n / by and n % by by way of 1 / by (quotients below 2^20, so the estimate is one off at most; the whole division is some forty
// instructions).
__device__ __forceinline__ int quotient(int n, int by, float inverse, int& remainder) {
  int q = static_cast<int>(static_cast<float>(n) * inverse), r = n - q * by;
  if (r < 0) --q, r += by;
  else if (r >= by) ++q, r -= by;
  remainder = r;
  return q;
}

// From the top, the bin of a histogram in which `rest` (>= 1) tokens are reached, a run of bins a thread: the digit goes behind the
// prefix and `rest` becomes what is left inside the bin, `found` what is in it.  False when the whole histogram does not reach it.
template <int PER>
__device__ __forceinline__ bool reach_bin(const unsigned int (&m)[PER], int bits, unsigned int& prefix, unsigned int& rest,
                                          unsigned int& found, FinishLds& l) {
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  unsigned int own = 0u;
#pragma unroll
  for (int j = 0; j < PER; ++j) own += m[j];
  unsigned int suffix = own;   // over the wave's bins from these up
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const unsigned int other = __shfl(suffix, min(lane + off, kWave - 1), kWave);
    if (lane + off < kWave) suffix += other;
  }
  if (lane == 0) l.wave_total[wave] = suffix;
  if (tid == 0) l.ok = 0u;
  __syncthreads();
  unsigned int above = suffix - own;
#pragma unroll
  for (int w = 0; w < kFinishThreads / kWave; ++w)
    if (w > wave) above += l.wave_total[w];
  if (above < rest && above + own >= rest) {
#pragma unroll
    for (int j = PER - 1; j >= 0; --j) {
      if (above < rest && above + m[j] >= rest) l.ok = 1u, l.digit = PER * tid + j, l.left = rest - above, l.found = m[j];
      above += m[j];
    }
  }
  __syncthreads();
  const bool ok = l.ok != 0u;
  if (ok) prefix = (prefix << bits) | l.digit, rest = l.left, found = l.found;
  __syncthreads();   // l may be used again
  return ok;
}

// Digit `level` of 31 bits, ten, eleven and ten at a time from the top (a run-time number: the three digits share their code).
struct Digit {
  int low, bits, high;
  __device__ __forceinline__ explicit Digit(int level) : low(level == 0 ? 21 : level == 1 ? 10 : 0), bits(level == 1 ? 11 : 10), high(low + bits) {}
  __device__ __forceinline__ int bin(unsigned int v) const { return static_cast<int>((v >> low) & ((1u << bits) - 1u)); }
};
__device__ __forceinline__ void clear_bins(FinishLds& l) {
#pragma unroll
  for (int j = 0; j < kBins1 / kFinishThreads; ++j) l.bins[j * kFinishThreads + threadIdx.x] = 0u;
  __syncthreads();
}
// The digit of a threshold from the counts in l.bins (those behind a digit's last bin are zero).
__device__ __forceinline__ bool digit_of_bins(const Digit& d, unsigned int& prefix, unsigned int& rest, unsigned int& found, FinishLds& l) {
  constexpr int kPer = kBins1 / kFinishThreads;
  static_assert(kBins0 <= kBins1 && kBins2 <= kBins1, "the bins of any digit");
  __syncthreads();
  unsigned int m[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) m[j] = l.bins[kPer * threadIdx.x + j];
  return reach_bin<kPer>(m, d.bits, prefix, rest, found, l);
}

// The digit from the whole row.  Every lane has kAhead 16-byte pieces on their way at once, because one workgroup's share of the
// memory's rate is what it has in flight; a wave whose values are all alike counts them as one.
__device__ __forceinline__ bool digit_of_row(const Digit& d, const MadeWeights& w, int vocab, unsigned int floor, unsigned int& prefix,
                                             unsigned int& rest, unsigned int& found, FinishLds& l) {
  constexpr int kAhead = 8;
  const float* __restrict__ x = w.row();
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  // neither NaN nor -1: they are beyond any prefix
  const unsigned int from = max(floor, prefix << d.high), behind = min((prefix + 1u) << d.high, 0x7f800000u);
  clear_bins(l);
  auto count = [&](float v) {
    const unsigned int bits = __float_as_uint(v);
    if (bits >= from && bits < behind) atomicAdd(&l.bins[d.bin(bits)], 1u);
  };
  const int head = min(vocab, static_cast<int>((4u - (static_cast<unsigned int>(reinterpret_cast<uintptr_t>(x)) / 4u) % 4u) % 4u));
  const int pieces = (vocab - head) / 4, tail = head + 4 * pieces;
  if (tid < head) count(w.at(tid));
  if (tid < vocab - tail) count(w.at(tail + tid));
  const float4* at = reinterpret_cast<const float4*>(x + head);
  for (int base = 0; base < pieces; base += kAhead * kFinishThreads) {
    float4 v[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) v[j] = at[min(base + j * kFinishThreads + tid, pieces - 1)];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const bool in = base + j * kFinishThreads + tid < pieces;
      const unsigned int lead = __builtin_amdgcn_readfirstlane(__float_as_int(v[j].x));
      const bool alike = in && __float_as_uint(v[j].x) == lead && __float_as_uint(v[j].y) == lead && __float_as_uint(v[j].z) == lead && __float_as_uint(v[j].w) == lead;
      if (__ballot(alike) == ~0ull) {
        const unsigned int bits = __float_as_uint(w.of(__uint_as_float(lead)));
        if (lane == 0 && bits >= from && bits < behind) atomicAdd(&l.bins[d.bin(bits)], 4u * kWave);
      } else if (in) {
        count(w.of(v[j].x)), count(w.of(v[j].y)), count(w.of(v[j].z)), count(w.of(v[j].w));
      }
    }
  }
  return digit_of_bins(d, prefix, rest, found, l);
}

// The row's tokens above `tie`, into l.raw; how many there are, and in `reach` those from `tie` on.
__device__ __forceinline__ int above_tie(const MadeWeights& w, int vocab, unsigned int tie, int& reach, FinishLds& l) {
  constexpr int kAhead = 8;
  const float* __restrict__ x = w.row();
  const int tid = threadIdx.x;
  if (tid == 0) l.count = l.n_live = 0;
  __syncthreads();
  int mine = 0;
  auto take = [&](const float (&v)[4], int token, bool in) {      // every lane of the wave; token: the first of four
    bool more[4];
    float e[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      e[j] = w.of(v[j]);
      const bool ok = in && e[j] >= 0.f;
      mine += ok && __float_as_uint(e[j]) >= tie;
      more[j] = ok && __float_as_uint(e[j]) > tie;
    }
    append(more, &l.count, [&](int at, int j) { if (at < kFinishMost) l.raw[at] = uint2{__float_as_uint(e[j]), static_cast<unsigned int>(token + j)}; });
  };
  const int head = min(vocab, static_cast<int>((4u - (static_cast<unsigned int>(reinterpret_cast<uintptr_t>(x)) / 4u) % 4u) % 4u));
  const int pieces = (vocab - head) / 4, tail = head + 4 * pieces;
  const float none = -INFINITY;
  unsigned int last = 0x7fc00000u, lead_bits = 0x7fc00000u;   // a NaN, and its e
  take({tid < head ? x[tid] : none, none, none, none}, tid, tid < head);
  take({tid < vocab - tail ? x[tail + tid] : none, none, none, none}, tail + tid, tid < vocab - tail);
  const float4* at = reinterpret_cast<const float4*>(x + head);
  for (int base = 0; base < pieces; base += kAhead * kFinishThreads) {
    float4 v[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) v[j] = at[min(base + j * kFinishThreads + tid, pieces - 1)];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const int piece = base + j * kFinishThreads + tid;
      const bool in = piece < pieces;
      const unsigned int lead = __builtin_amdgcn_readfirstlane(__float_as_int(v[j].x));
      const bool alike = in && __float_as_uint(v[j].x) == lead && __float_as_uint(v[j].y) == lead && __float_as_uint(v[j].z) == lead && __float_as_uint(v[j].w) == lead;
      if (__builtin_expect(lead != last, 0)) last = lead, lead_bits = __float_as_uint(w.of(__uint_as_float(lead)));
      const unsigned int bits = lead_bits;
      if (__ballot(alike) == ~0ull && bits <= tie)
        mine += bits == tie ? 4 : 0;
      else
        take({v[j].x, v[j].y, v[j].z, v[j].w}, head + 4 * piece, in);
    }
  }
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) mine += __shfl_xor(mine, off, kWave);
  if ((tid & (kWave - 1)) == 0 && mine != 0) atomicAdd(&l.n_live, mine);
  __syncthreads();
  reach = l.n_live;
  return l.count;
}

// The digit from the list.
__device__ __forceinline__ bool digit_of_list(const Digit& d, int n, unsigned int& prefix, unsigned int& rest, unsigned int& found, FinishLds& l) {
  clear_bins(l);
  for (int i = threadIdx.x; i < n; i += kFinishThreads) {
    const unsigned int bits = l.raw[i].x;
    if ((bits >> d.high) == prefix) atomicAdd(&l.bins[d.bin(bits)], 1u);
  }
  return digit_of_bins(d, prefix, rest, found, l);
}

// The digit of the rank-th largest of the groups' largest e.  `most`: the first groups' largest logits, fetched by the caller.
constexpr int kGroupsAhead = 4;
__device__ __forceinline__ bool digit_of_groups(const Digit& d, const MadeWeights& w, const float* gm, int groups, const float (&most)[kGroupsAhead],
                                                unsigned int& prefix, unsigned int& rest, unsigned int& found, FinishLds& l) {
  clear_bins(l);
  for (int base = 0; base < groups; base += kGroupsAhead * kFinishThreads) {
#pragma unroll
    for (int j = 0; j < kGroupsAhead; ++j) {
      const int g = base + j * kFinishThreads + static_cast<int>(threadIdx.x);
      const float e = w.of(base == 0 ? most[j] : gm[min(g, groups - 1)]);
      const unsigned int bits = __float_as_uint(e);
      // (a wave whose lanes all fall into one bin adds them at once: flat rows)
      const bool in = g < groups && e >= 0.f && (bits >> d.high) == prefix;
      const int bin = d.bin(bits), lead = __builtin_amdgcn_readfirstlane(bin);
      const unsigned long long some = __ballot(in);
      if (some == __ballot(in && bin == lead)) {
        if ((threadIdx.x & (kWave - 1)) == 0 && some != 0ull) atomicAdd(&l.bins[lead], static_cast<unsigned int>(__builtin_popcountll(some)));
      } else if (in) {
        atomicAdd(&l.bins[bin], 1u);
      }
    }
  }
  return digit_of_bins(d, prefix, rest, found, l);
}

// The row's tokens from `lower` on, into l.raw; how many there are (more than kFinishMost: some are not listed).  `most`: the
// largest logits of the first groups, fetched by the caller.
__device__ __forceinline__ int gather(const SampleArgs& a, unsigned int lower, const MadeWeights& w, const float* gm, int groups,
                                      const float (&most)[kGroupsAhead], FinishLds& l) {
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const float inverse = 1.0f / static_cast<float>(a.groups);
  static_assert(kGroupsAhead * kFinishThreads <= kLiveMost, "a round's groups fit the list");
  if (tid == 0) l.count = l.n_live = 0;
  __syncthreads();
  for (int base = 0; base < groups; base += kGroupsAhead * kFinishThreads) {
    bool live[kGroupsAhead];
    unsigned int entry[kGroupsAhead];
#pragma unroll
    for (int j = 0; j < kGroupsAhead; ++j) {
      const int g = base + j * kFinishThreads + tid;
      const float m = base == 0 ? most[j] : gm[min(g, groups - 1)];
      int in_chunk;
      const int chunk = quotient(g, a.groups, inverse, in_chunk), first = chunk * a.chunk_len + in_chunk * kGroup;
      const int tokens = min(min(a.chunk_len - in_chunk * kGroup, a.vocab - first), kGroup);
      // (a chunk's last groups may lie past its end)
      live[j] = g < groups && tokens > 0 && w.group_reaches(m, lower);
      entry[j] = static_cast<unsigned int>(first) / 4u * kGroup + static_cast<unsigned int>(tokens - 1);
    }
    append(live, &l.n_live, [&](int at, int j) { l.live[at] = entry[j]; });
    __syncthreads();
    const int n_live = l.n_live;
    constexpr int kEach = 8;
    for (int from = kEach * wave; from < n_live; from += kEach * kFinishThreads / kWave) {
      float v[kEach];
      int token[kEach];
      bool in[kEach];
#pragma unroll
      for (int j = 0; j < kEach; ++j) {
        const unsigned int entry = l.live[min(from + j, n_live - 1)];
        in[j] = from + j < n_live && lane <= static_cast<int>(entry % kGroup);
        token[j] = static_cast<int>(entry / kGroup * 4u) + min(lane, static_cast<int>(entry % kGroup));
        v[j] = w.row()[token[j]];
      }
#pragma unroll
      for (int j = 0; j < kEach; ++j) v[j] = w.of(v[j]);
#pragma unroll
      for (int j = 0; j < kEach; ++j) in[j] = in[j] && v[j] >= 0.f && __float_as_uint(v[j]) >= lower;
      append(in, &l.count, [&](int at, int j) { if (at < kFinishMost) l.raw[at] = uint2{__float_as_uint(v[j]), static_cast<unsigned int>(token[j])}; });
    }
    __syncthreads();
    if (tid == 0) l.n_live = 0;
    if (base + kGroupsAhead * kFinishThreads < groups) __syncthreads();
  }
  __syncthreads();
  return l.count;
}

// What of the list reaches `lower` stays; how many that are.
__device__ __forceinline__ int keep_from(unsigned int lower, int n, FinishLds& l) {
  constexpr int kEach = kFinishMost / kFinishThreads;
  uint2 mine[kEach];
  bool in[kEach];
#pragma unroll
  for (int j = 0; j < kEach; ++j) {
    const int i = j * kFinishThreads + static_cast<int>(threadIdx.x);
    mine[j] = l.raw[min(i, n - 1)];
    in[j] = i < n && mine[j].x >= lower;
  }
  __syncthreads();
  if (threadIdx.x == 0) l.count = 0;
  __syncthreads();
  append(in, &l.count, [&](int at, int j) { l.raw[at] = mine[j]; });
  __syncthreads();
  return l.count;
}

// The kept mass of every chunk from the row, in the order of sample_mass_kernel: 256 threads a chunk, kAhead chunks of theirs at once.
__device__ __forceinline__ void masses_of_row(const SampleArgs& a, const MadeWeights& w, unsigned int thr, FinishLds& l) {
  constexpr int kAhead = 4, kUnroll = 9, kGroups = kFinishThreads / kSelThreads;
  const float* x = w.row();
  float last = __uint_as_float(0x7fc00000u), last_kept = 0.f;   // rows of many ties: an exponential only where a lane's logit is another than before
  auto kept = [&](float logit) {
    if (__builtin_expect(__ballot(logit != last) != 0ull, 0)) {
      asm volatile("");   // a branch, not two values to choose from
      const float e = w.of(logit);
      last = logit, last_kept = e >= 0.f && __float_as_uint(e) >= thr ? e : 0.f;
    }
    return last_kept;
  };
  const int t = threadIdx.x % kSelThreads, lane = threadIdx.x & (kWave - 1), wave = t / kWave;
  for (int c0 = threadIdx.x / kSelThreads; c0 < a.chunks; c0 += kAhead * kGroups) {
    float mass[kAhead] = {};
    for (int i = t; i < a.chunk_len; i += kUnroll * kSelThreads) {
      float v[kAhead][kUnroll];
#pragma unroll
      for (int j = 0; j < kAhead; ++j)
#pragma unroll
        for (int k = 0; k < kUnroll; ++k) v[j][k] = x[min(min(c0 + j * kGroups, a.chunks - 1) * a.chunk_len + i + k * kSelThreads, a.vocab - 1)];
#pragma unroll
      for (int j = 0; j < kAhead; ++j)
#pragma unroll
        for (int k = 0; k < kUnroll; ++k) {
          const bool in = i + k * kSelThreads < min(a.chunk_len, a.vocab - (c0 + j * kGroups) * a.chunk_len);
          const float e = kept(v[j][k]);
          if (in) mass[j] += e;
        }
    }
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const float sum = wave_sum(mass[j]);
      if (lane == 0 && c0 + j * kGroups < a.chunks) l.wave_mass[c0 + j * kGroups][wave] = sum;
    }
  }
  __syncthreads();
  if (static_cast<int>(threadIdx.x) < a.chunks) {
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < kSelWaves; ++w) total += l.wave_mass[threadIdx.x][w];
    l.masses[threadIdx.x] = total;
  }
  __syncthreads();
}

// The first token with the row's largest logit: in the first group that has it; where the largest is -inf a group of NaNs alone
// looks the same, and the whole row is searched.
__device__ __forceinline__ void first_of(const SampleArgs& a, int row, float largest, const float* gm, int groups, FinishLds& l) {
  const float* x = a.logits + static_cast<int64_t>(row) * a.vocab;
  constexpr int kNone = 0x7fffffff;
  if (threadIdx.x == 0) l.count = l.n_live = kNone;
  __syncthreads();
  int group = kNone;
  for (int g = threadIdx.x; g < groups && group == kNone; g += kFinishThreads)
    if (gm[g] == largest) group = g;
  if (group != kNone) atomicMin(&l.count, group);
  __syncthreads();
  group = l.count;
  int from = 0, to = a.vocab;
  if (largest > -INFINITY) {
    const int chunk = group / a.groups, in_chunk = group % a.groups;
    from = chunk * a.chunk_len + in_chunk * kGroup;
    to = min(min(from + kGroup, (chunk + 1) * a.chunk_len), a.vocab);
  }
  for (int i = from + static_cast<int>(threadIdx.x); i < to; i += kFinishThreads)
    if (x[i] == largest) {
      atomicMin(&l.n_live, i);
      break;
    }
  __syncthreads();
  if (threadIdx.x == 0) leave_token(a, row, l.n_live == kNone ? 0 : l.n_live);
}

constexpr unsigned int kManyGroups = 512;
// The parameters of up to kInlineRows rows as an argument of the kernel: no copy to the GPU in front of it.
constexpr int kInlineRows = 64;
struct InlineRows {
  float temperature[kInlineRows], top_p[kInlineRows], min_p[kInlineRows], u[kInlineRows];
  int top_k[kInlineRows];
};
struct NoRows {};

template <typename Rows>
__global__ __launch_bounds__(kFinishThreads) void sample_finish_kernel(const SampleArgs a, const Rows rows) {
  __shared__ FinishLds l;
  const int row = blockIdx.x, tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  // what is wanted of the row and does not hang on anything else: all on its way at once
  const float* gm = a.group_max + static_cast<int64_t>(row) * a.chunks * a.groups;
  const int groups = a.chunks * a.groups;
  float most[kGroupsAhead];
#pragma unroll
  for (int j = 0; j < kGroupsAhead; ++j) most[j] = gm[min(j * kFinishThreads + tid, groups - 1)];
  RowParams r;
  float u;
  if constexpr (std::is_same_v<Rows, InlineRows>) {
    r = row_params(a, rows.temperature[row], rows.top_k[row], rows.top_p[row], rows.min_p[row]);
    u = rows.u[row];
  } else {
    r = row_params(a, row);
    u = a.u[row];
  }
  float largest = -INFINITY;
#pragma unroll
  for (int j = 0; j < kGroupsAhead; ++j) largest = fmaxf(largest, most[j]);
  for (int g = kGroupsAhead * kFinishThreads + tid; g < groups; g += kFinishThreads) largest = fmaxf(largest, gm[g]);
  largest = block_max<kFinishThreads / kWave>(largest, l.largest);
  if (r.greedy) {
    first_of(a, row, largest, gm, groups, l);
    return;
  }
  const MadeWeights w{a.logits + static_cast<int64_t>(row) * a.vocab, r.inv_t, largest * r.inv_t};
  const unsigned int mp = min_p_bits(r), k = static_cast<unsigned int>(r.k);
  if (tid == 0) l.threshold = mp;
  for (int c = tid; c < 256; c += kFinishThreads) l.first[c] = l.behind[c] = 0, l.masses[c] = 0.f;
  // The top_k-th largest of the groups' largest e, or a digit's lower end that not many more groups reach: top_k tokens are there
  // or above, and those that are lie in these groups.  (An e of zero weighs nothing and is never drawn: where the rank is
  // only reached among those, most logits -inf, say, the others all stay, which is what the list then gives.)
  unsigned int prefix = 0u, rest = k, found = 0u;
  auto few = [&] { return (k - rest) + found <= max(2u * k, 128u); };
  int digits = 0;
  while (digits < 3 && (digits == 0 || !few()) && digit_of_groups(Digit(digits), w, gm, groups, most, prefix, rest, found, l)) ++digits;
  const unsigned int reached = digits == 0 ? 0u : prefix << Digit(digits - 1).low;   // 0 where fewer groups than that are there
  const unsigned int reaching = digits == 3 ? (k - rest) + found : 0u;   // groups whose largest reaches the threshold of the groups
  unsigned int lower = max(max(mp, reached), 1u), thr = mp, ties = 0u;   // ties: tokens at the threshold that are not listed
  bool known = false;
  int n;
  if (reaching > kManyGroups && lower == reached) {
    // so many groups end in one value that it is most likely the threshold: those above it are the list
    int reach;
    n = above_tie(w, a.vocab, lower, reach, l);
    if (static_cast<unsigned int>(n) < k) thr = lower, ties = static_cast<unsigned int>(reach - n), known = true;
  } else {
    n = gather(a, lower, w, gm, groups, most, l);
  }
  rest = k, found = 0u, prefix = 0u;
  if (n > kFinishMost) {      // the row by digits: the rank is reached from `lower` on (fewer than top_k tokens otherwise)
    auto listed = [&] { return (k - rest) + found <= static_cast<unsigned int>(kFinishMost); };
    int row_digits = 0;
    while (row_digits < 3 && (row_digits == 0 || !listed()) && digit_of_row(Digit(row_digits), w, a.vocab, lower, prefix, rest, found, l)) ++row_digits;
    if (row_digits > 0) lower = max(lower, prefix << Digit(row_digits - 1).low);
    if (row_digits == 3) {
      thr = max(mp, prefix), known = true;
      if (!listed()) ties = found, lower = prefix + 1u;
    }
    n = gather(a, lower, w, gm, groups, most, l);
    rest = k, found = 0u, prefix = 0u;
  }
  if (n > kDirectMost && !known) {
    int list_digits = 0;
    while (list_digits < 3 && digit_of_list(Digit(list_digits), n, prefix, rest, found, l)) ++list_digits;
    if (list_digits == 3) thr = max(mp, prefix);
    known = true;
    const int all = n;
    n = keep_from(max(thr, 1u), all, l);
  }
  if (n > kKeptMost) {      // ties
    const int all = n;
    n = keep_from(thr + 1u, n, l);
    ties += static_cast<unsigned int>(all - n);
  }
  // four threads a token compare it with all
  const int quarter = tid & 3;
  for (int i = tid / 4; i < n; i += kFinishThreads / 4) {
    const uint2 own_pair = l.raw[i];
    const unsigned int bits = own_pair.x, token = own_pair.y;
    unsigned int rank = 0, above = 0, reach = 0, before = 0;      // before: of the same value, further ahead in the tokens' order
#pragma unroll 4
    for (int j = quarter; j < n; j += 4) {
      const uint2 other = l.raw[j];
      const bool ahead = other.y < token;
      rank += ahead;
      above += other.x > bits;
      reach += other.x >= bits;
      before += ahead && other.x == bits;
    }
    auto four = [](unsigned int& v) { v += __shfl_xor(v, 1, kWave), v += __shfl_xor(v, 2, kWave); };
    four(rank), four(above), four(reach), four(before);
    if (quarter == 0) {
      l.list.bits[rank] = bits;
      l.list.token[rank] = static_cast<int>(token);
      l.list.value[above + before] = bits;
      if (!known && above < k && k <= reach) l.threshold = max(mp, bits);   // the k-th largest, and its ties
    }
  }
  if (tid == 0) l.ok = 0u;
  __syncthreads();
  if (!known) thr = l.threshold;
  if (r.p_active) {
    // from the largest value down, one a thread, until the mass is reached
    const unsigned int bits = tid < n ? l.list.value[tid] : 0u;
    auto mass_of = [](unsigned int b) { return static_cast<unsigned long long>(__uint_as_float(b) * kMassScale); };
    const unsigned long long mass = tid < n && bits >= thr ? mass_of(bits) : 0ull;
    unsigned long long upto = mass;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const unsigned long long other = shfl_any(upto, max(lane - off, 0));
      if (lane >= off) upto += other;
    }
    if (lane == kWave - 1) l.wave_mass_total[wave] = upto;
    __syncthreads();
    unsigned long long total = static_cast<unsigned long long>(ties) * mass_of(thr);
#pragma unroll
    for (int w = 0; w < kFinishThreads / kWave; ++w) {
      const unsigned long long of_wave = l.wave_mass_total[w];
      total += of_wave;
      if (w < wave) upto += of_wave;
    }
    const unsigned long long need = top_p_need(r.top_p, total);
    if (mass > 0ull && upto - mass < need && need <= upto) l.digit = bits, l.ok = 2u;
    __syncthreads();
    if (l.ok == 2u) thr = l.digit, ties = 0u;      // among those, above the ties
  }
  if (ties > 0u) {
    __syncthreads();   // the list is done with
    masses_of_row(a, w, thr, l);
    pick_token(a, row, u, thr, l.masses, w, l.pick);
    return;
  }
  const float per_chunk = 1.0f / static_cast<float>(a.chunk_len);
  auto chunk_of = [&](int i) { int in_chunk; return quotient(l.list.token[i], a.chunk_len, per_chunk, in_chunk); };
  if (tid < n) {
    const int chunk = chunk_of(tid);
    if (tid == 0 || chunk_of(tid - 1) != chunk) l.first[chunk] = tid;
    if (tid == n - 1 || chunk_of(tid + 1) != chunk) l.behind[chunk] = tid + 1;
  }
  __syncthreads();
  for (int c = wave; c < a.chunks; c += kFinishThreads / kWave) {
    const int from = l.first[c], to = l.behind[c];
    if (from == to) continue;
    float mass[kSelWaves] = {};      // what the waves of the chunk's workgroup would have found
    for (int i = from; i < to; ++i) {
      const unsigned int bits = l.list.bits[i];
      const int slot = (l.list.token[i] - c * a.chunk_len) % kSelThreads;
#pragma unroll
      for (int w = 0; w < kSelWaves; ++w)
        if (bits >= thr && slot == w * kWave + lane) mass[w] += __uint_as_float(bits);
    }
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < kSelWaves; ++w) total += wave_sum(mass[w]);
    if (lane == 0) l.masses[c] = total;
  }
  __syncthreads();

  // pick_token's steps on the list
  find_target(a, u, l.masses, l.pick);
  const int chunk = l.pick.chunk_of_target;
  const float target = l.pick.target;
  const int begin = chunk * a.chunk_len, end = min(a.vocab, begin + a.chunk_len);
  const int per = (end - begin + kSelThreads - 1) / kSelThreads;
  const bool owns = tid < kSelThreads;
  const int lo = owns ? min(begin + tid * per, end) : end, hi = owns ? min(lo + per, end) : end;
  const int from = l.first[chunk], to = l.behind[chunk];
  auto mine_is = [&](int i) { return l.list.bits[i] >= thr && l.list.token[i] >= lo && l.list.token[i] < hi; };
  float mine = 0.f;
  for (int i = from; i < to; ++i)
    if (mine_is(i)) mine += __uint_as_float(l.list.bits[i]);
  if (owns) l.pick.part[tid] = mine;
  add_up_parts(l.pick, l.pick.chunk_start);
  const float start = owns ? l.pick.part[tid] : 0.f;
  if (target >= start && target < start + mine && hi > lo) {
    float run = start;
    int pick = -1, last = -1;
    for (int i = from; i < to && pick < 0; ++i) {
      if (!mine_is(i)) continue;
      const float v = __uint_as_float(l.list.bits[i]);
      run += v;
      if (v > 0.f) last = l.list.token[i];
      if (target < run) pick = l.list.token[i];
    }
    if (pick < 0) pick = last;
    if (pick >= 0) atomicMax(&l.pick.chosen, pick);
  }
  __syncthreads();
  if (l.pick.chosen < 0) {
    int in_chunk = -1, in_row = -1;
    for (int i = tid; i < n; i += kFinishThreads)
      if (l.list.bits[i] >= thr && l.list.bits[i] > 0u) {
        in_row = max(in_row, l.list.token[i]);
        if (l.list.token[i] >= begin && l.list.token[i] < end) in_chunk = max(in_chunk, l.list.token[i]);
      }
    __syncthreads();
    if (in_chunk >= 0) atomicMax(&l.pick.chosen, in_chunk);
    __syncthreads();
    const bool none = l.pick.chosen < 0;
    __syncthreads();
    if (none && in_row >= 0) atomicMax(&l.pick.chosen, in_row);
    __syncthreads();
  }
  if (tid == 0) leave_token(a, row, max(l.pick.chosen, 0));
}

// logits[row, tok] for each (tok, count) listed for the row:
//   l = l >= 0 ? l / rep : l * rep;   l -= freq * count + presence
__global__ void apply_penalties_kernel(float* __restrict__ logits, int vocab,
                                       const int* __restrict__ indptr, const int* __restrict__ tok,
                                       const int* __restrict__ count, const float* __restrict__ rep,
                                       const float* __restrict__ freq,
                                       const float* __restrict__ pres) {
  const int row = blockIdx.x;
  float* x = logits + static_cast<int64_t>(row) * vocab;
  for (int e = indptr[row] + threadIdx.x; e < indptr[row + 1]; e += blockDim.x) {
    const int id = tok[e];
    const int c = count[e];
    if (id < 0 || id >= vocab || c <= 0) continue;
    float l = x[id];
    const float r = rep[row];
    if (r != 1.0f) l = l >= 0.f ? l / r : l * r;
    x[id] = l - freq[row] * static_cast<float>(c) - pres[row];
  }
}

}  // namespace arle

using namespace arle;

// parts: scratch of arle_argmax_chunks(rows, vocab) * rows pairs of 8 bytes, or null when that count is 1.
extern "C" int arle_argmax_chunks(int rows, int vocab) {
  if (rows <= 0 || vocab < 8192) return 1;
  const int wanted = (2048 + rows - 1) / rows;           // about 2048 workgroups of 256 threads in all
  const int most = vocab / 2048;                         // at least 2048 logits a chunk
  return max(1, min(min(wanted, most), 256));
}

extern "C" int arle_argmax_rows(const float* logits, int rows, int vocab, int* out, void* parts, void* stream) {
  if (rows == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int chunks = arle_argmax_chunks(rows, vocab);
  if (chunks == 1) {
    argmax_rows_kernel<<<rows, kSampThreads, 0, s>>>(logits, vocab, out);
    return launch_status();
  }
  if (parts == nullptr) return static_cast<int>(hipErrorInvalidValue);
  const int chunk_len = (((vocab + chunks - 1) / chunks) + 3) & ~3;
  argmax_chunks_kernel<<<dim3(chunks, rows), kChunkThreads, 0, s>>>(logits, vocab, chunk_len,
                                                                    static_cast<ArgMax*>(parts), ClearRows{nullptr, nullptr, 0, 0, 0, 0});
  argmax_merge_kernel<<<rows, kWave, 0, s>>>(static_cast<const ArgMax*>(parts), chunks, out);
  return launch_status();
}

// Scratch of a sampling call, in bytes: the histograms of top_k and of top_p, the passes' slots, the chunk maxima and masses,
// the groups' maxima and the thresholds.
static inline int sample_chunk_len(int vocab, int chunks) { return (((vocab + chunks - 1) / chunks) + 3) & ~3; }
static inline int sample_groups(int vocab, int chunks) { return (sample_chunk_len(vocab, chunks) + kGroup - 1) / kGroup; }
extern "C" long long arle_sample_hist_k_bytes(int rows) { return static_cast<long long>(rows) * kRowBins * sizeof(unsigned int); }
extern "C" long long arle_sample_hist_p_bytes(int rows) { return static_cast<long long>(rows) * kRowBins * sizeof(unsigned long long); }
// finish != 0: for calls that the finishing kernel takes (arle_sample_rows), which keep the groups' maxima alone.
extern "C" long long arle_sample_scratch_bytes(int rows, int vocab, int finish) {
  const int chunks = arle_argmax_chunks(rows, vocab);
  if (finish) return static_cast<long long>(static_cast<size_t>(rows) * chunks * sample_groups(vocab, chunks) * sizeof(float));
  return arle_sample_hist_k_bytes(rows) + arle_sample_hist_p_bytes(rows) +
         static_cast<long long>(static_cast<size_t>(rows) * kPasses * sizeof(Slot) +
                                static_cast<size_t>(rows) * chunks *
                                    (sizeof(ArgMax) + sizeof(float) + sample_groups(vocab, chunks) * sizeof(float)) +
                                rows * sizeof(unsigned int));
}

// The largest top_k that the finishing kernel is for.
extern "C" int arle_sample_finish_most() { return kFinishTopK; }

// One token id per row of logits [rows, vocab] (float32).  probs is scratch [rows, vocab] float32; scratch holds
// arle_sample_scratch_bytes(rows, vocab, whether two kernels do all) bytes, 16-byte aligned.  use_top_k / use_top_p == 0 promise that no row of the call has
// the filter switched on (top_k in 1..vocab-1, top_p < 1); its passes are then left out.  small_k != 0 promises that every row is
// greedy or has a top_k of 1 to arle_sample_finish_most(), below vocab: with vocab up to 2^28 two kernels then do all, probs may be
// null, and with on_host != 0 temperature is a host array [5][rows] of the temperatures, top_p, min_p, u and the bits of top_k of up to
// arle_sample_host_rows() rows (the other four pointers are not looked at), which travel with the launch.  out_host: pinned host
// memory of `rows` numbers that takes the tokens too, or null.
extern "C" int arle_sample_host_rows() { return kInlineRows; }
extern "C" int arle_sample_rows(const float* logits, int rows, int vocab, float* probs,
                                const float* temperature, const int* top_k, const float* top_p,
                                const float* min_p, const float* u, int* out, void* scratch, int use_top_k,
                                int use_top_p, int small_k, int on_host, int* out_host, void* stream) {
  if (rows == 0) return 0;
  if (scratch == nullptr || reinterpret_cast<uintptr_t>(scratch) % 16 != 0 || rows > 65535)
    return static_cast<int>(hipErrorInvalidValue);
  hipStream_t s = static_cast<hipStream_t>(stream);
  SampleArgs a;
  a.logits = logits;
  a.e = probs;
  a.vocab = vocab;
  a.chunks = arle_argmax_chunks(rows, vocab);
  a.chunk_len = sample_chunk_len(vocab, a.chunks);
  a.groups = sample_groups(vocab, a.chunks);
  a.temperature = temperature;
  a.top_k = top_k;
  a.top_p = top_p;
  a.min_p = min_p;
  a.u = u;
  a.use_top_k = use_top_k;
  a.use_top_p = use_top_p;
  a.out = out;
  a.out_host = out_host;
  const dim3 grid(a.chunks, rows);
  if (small_k && use_top_k && vocab <= kFinishVocab) {
    if (on_host && rows > kInlineRows) return static_cast<int>(hipErrorInvalidValue);
    a.group_max = static_cast<float*>(scratch);
    group_max_kernel<<<grid, kChunkThreads, 0, s>>>(logits, vocab, a.chunk_len, a.groups, a.group_max);
    if (on_host) {
      InlineRows values;
      float* const to[4] = {values.temperature, values.top_p, values.min_p, values.u};
      for (int i = 0; i < 4; ++i) std::memcpy(to[i], temperature + static_cast<size_t>(i) * rows, rows * sizeof(float));
      std::memcpy(values.top_k, temperature + static_cast<size_t>(4) * rows, rows * sizeof(int));
      sample_finish_kernel<InlineRows><<<rows, kFinishThreads, 0, s>>>(a, values);
    } else {
      sample_finish_kernel<NoRows><<<rows, kFinishThreads, 0, s>>>(a, NoRows{});
    }
    return launch_status();
  }
  if (on_host || probs == nullptr) return static_cast<int>(hipErrorInvalidValue);
  unsigned char* at = static_cast<unsigned char*>(scratch);
  a.hist_k = reinterpret_cast<unsigned int*>(at);
  at += arle_sample_hist_k_bytes(rows);
  a.hist_p = reinterpret_cast<unsigned long long*>(at);
  at += arle_sample_hist_p_bytes(rows);
  a.slots = reinterpret_cast<Slot*>(at);
  at += static_cast<size_t>(rows) * kPasses * sizeof(Slot);
  ArgMax* part_max = reinterpret_cast<ArgMax*>(at);
  a.part_max = part_max;
  at += static_cast<size_t>(rows) * a.chunks * sizeof(ArgMax);
  a.chunk_mass = reinterpret_cast<float*>(at);
  at += static_cast<size_t>(rows) * a.chunks * sizeof(float);
  a.group_max = reinterpret_cast<float*>(at);
  at += static_cast<size_t>(rows) * a.chunks * a.groups * sizeof(float);
  a.threshold = reinterpret_cast<unsigned int*>(at);
  // the histograms of the filters that are on start at zero
  const int k_row = kRowBins * sizeof(unsigned int) / 16, p_row = kRowBins * sizeof(unsigned long long) / 16;
  const ClearRows clear{reinterpret_cast<uint4*>(a.hist_k), reinterpret_cast<uint4*>(a.hist_p), use_top_k ? k_row : 0, k_row,
                        use_top_p ? p_row : 0, p_row};
  argmax_chunks_kernel<<<grid, kChunkThreads, 0, s>>>(logits, vocab, a.chunk_len, part_max, clear);
  sample_exp_kernel<<<grid, kSelThreads, 0, s>>>(a);
  if (use_top_k || use_top_p) {
    sample_pass_kernel<kFirst><<<grid, kSelThreads, 0, s>>>(a);
    sample_pass_kernel<kSecond><<<grid, kSelThreads, 0, s>>>(a);
  }
  if (use_top_k && use_top_p) {
    sample_pass_kernel<kFloor><<<grid, kSelThreads, 0, s>>>(a);
    sample_pass_kernel<kThird><<<grid, kSelThreads, 0, s>>>(a);
    sample_pass_kernel<kFourth><<<grid, kSelThreads, 0, s>>>(a);
  }
  sample_mass_kernel<<<grid, kSelThreads, 0, s>>>(a);
  sample_pick_kernel<<<rows, kSelThreads, 0, s>>>(a);
  return launch_status();
}

// out[r] = logits[r][token[r]] - logsumexp(logits[r]): the natural-log probability of the chosen token under
// the softmax of the row (for the largest logit this is the reference's -log(sum exp(x - max)),
// crates/cuda-kernels/csrc/misc/sampling.cu:299-316).  One workgroup a row, fixed order of additions.
__global__ __launch_bounds__(kSampThreads) void token_logprob_kernel(const float* __restrict__ logits, int vocab,
                                                                    const int* __restrict__ token,
                                                                    float* __restrict__ out) {
  __shared__ float lds[kSampWaves];
  const float* x = logits + static_cast<int64_t>(blockIdx.x) * vocab;
  float m = -INFINITY;
  for (int i = threadIdx.x; i < vocab; i += kSampThreads) m = fmaxf(m, x[i]);
  m = block_max<kSampWaves>(m, lds);
  float sum = 0.f;
  for (int i = threadIdx.x; i < vocab; i += kSampThreads) sum += expf(x[i] - m);
  sum = block_sum<kSampWaves>(sum, lds);
  if (threadIdx.x == 0) {
    const int t = token[blockIdx.x];
    out[blockIdx.x] = (t >= 0 && t < vocab) ? x[t] - m - logf(sum) : -INFINITY;
  }
}

extern "C" int arle_token_logprobs(const float* logits, int rows, int vocab, const int* token, float* out,
                                   void* stream) {
  if (rows == 0) return 0;
  if (vocab <= 0) return static_cast<int>(hipErrorInvalidValue);
  token_logprob_kernel<<<rows, kSampThreads, 0, static_cast<hipStream_t>(stream)>>>(logits, vocab, token, out);
  return launch_status();
}

extern "C" int arle_apply_penalties(float* logits, int rows, int vocab, const int* indptr,
                                    const int* tok, const int* count, const float* rep,
                                    const float* freq, const float* pres, void* stream) {
  if (rows == 0) return 0;
  apply_penalties_kernel<<<rows, 256, 0, static_cast<hipStream_t>(stream)>>>(
      logits, vocab, indptr, tok, count, rep, freq, pres);
  return launch_status();
}
