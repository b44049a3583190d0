// A short causal convolution over time on every channel of the rows of a packed step, continued across
// steps through a per-request state of the last taps-1 inputs.
//
//   y_t[c] = (ADD ? u_t[c] : 0) + sum_{j < taps} w[c][j] * u_(t - taps + 1 + j)[c],    u := input (+ bias)
//   (out_bias: added to y in front of the silu.)
//   (SILU: y <- y / (1 + exp(-y)) on the way out.  The entry point's `add_input` holds both: bit 0 ADD, bit 1 SILU.)
//
// The rows of one request are consecutive in the step; an input further back than the request's first row of
// this step comes from its state [slots][taps-1][channels] (the most recent input last), which is all zeros
// when the request starts, so inputs before position 0 count as zero without a test.  The sums are 32-bit.
// `conv_state_update` then shifts each request's state by the rows it brought.  The update is a kernel of its
// own because the convolution of a step reads the old state of every request; where one workgroup a request does all of that
// reading (causal_conv_rows_kernel) it moves the state on itself.
#include "common.h"

namespace arle {

constexpr int kConvMaxTaps = 16;
constexpr int kConvManyRows = 128;   // rows of a step from which on a lane takes several
constexpr int kConvAdd = 1, kConvSilu = 2;

__device__ __forceinline__ float conv_out(float y, int flags) { return (flags & kConvSilu) ? y / (1.0f + expf(-y)) : y; }

__global__ void causal_conv_kernel(const void* __restrict__ u, long long u_stride, int u_dtype,
                                   const void* __restrict__ bias, int bias_dtype, const void* __restrict__ out_bias,
                                   int ob_dtype, const void* __restrict__ w, int w_dtype,
                                   const void* __restrict__ state, int state_dtype,
                                   const int* __restrict__ slot_of_token, void* __restrict__ out,
                                   long long out_stride, int out_dtype, int channels, int taps, int add_input) {
  const int t = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  const int slot = slot_of_token[t];
  const float b = bias ? load_as_float(bias, bias_dtype, c) : 0.f;
  const float now = load_as_float(u, u_dtype, t * u_stride + c) + b;
  if (!w) {   // no convolution: the input with its bias
    store_from_float(out, out_dtype, t * out_stride + c, now);
    return;
  }
  // rows of the same request right before this one in the step (at most taps-1 matter)
  int mine = 0;
  while (mine < taps - 1 && t - mine - 1 >= 0 && slot_of_token[t - mine - 1] == slot) ++mine;
  float acc = ((add_input & kConvAdd) ? now : 0.f) + (out_bias ? load_as_float(out_bias, ob_dtype, c) : 0.f);
  acc = fmaf(load_as_float(w, w_dtype, static_cast<int64_t>(c) * taps + taps - 1), now, acc);
  for (int back = 1; back < taps; ++back) {
    float v;
    if (back <= mine) {
      v = load_as_float(u, u_dtype, (t - back) * u_stride + c) + b;
    } else {  // state row taps-1 - (back - mine): the (back - mine)-th most recent input before the step
      const int64_t row = static_cast<int64_t>(slot) * (taps - 1) + (taps - 1 - (back - mine));
      v = load_as_float(state, state_dtype, row * channels + c);
    }
    acc = fmaf(load_as_float(w, w_dtype, static_cast<int64_t>(c) * taps + taps - 1 - back), v, acc);
  }
  store_from_float(out, out_dtype, t * out_stride + c, conv_out(acc, add_input));
}

// One element type T throughout and channels in whole groups of four: a lane takes four channels of a row with one
// access each for the input, the taps - 1 rows before it (the step's, or the state's) and the weights; none of the
// loads stands under a condition on data (which rows are the step's is the same for the whole workgroup).
template <typename T, int TAPS>
__global__ void causal_conv_vec_kernel(const T* __restrict__ u, long long u_stride, const T* __restrict__ bias,
                                       const T* __restrict__ out_bias, const T* __restrict__ w, const T* __restrict__ state,
                                       const int* __restrict__ slot_of_token, T* __restrict__ out, long long out_stride,
                                       int channels, int add_input) {
  const int t = blockIdx.x;
  const int c = (blockIdx.y * blockDim.x + threadIdx.x) * 4;
  if (c >= channels) return;
  const int slot = slot_of_token[t];
  int mine = 0;
  while (mine < TAPS - 1 && t - mine - 1 >= 0 && slot_of_token[t - mine - 1] == slot) ++mine;
  const float4 b = bias ? ld4<T>(bias + c) : float4{0.f, 0.f, 0.f, 0.f};
  float4 in[TAPS];     // in[back]: the input `back` rows before this one
#pragma unroll
  for (int back = 0; back < TAPS; ++back) {
    if (back <= mine) {
      const float4 v = ld4<T>(u + (t - back) * u_stride + c);
      in[back] = float4{v.x + b.x, v.y + b.y, v.z + b.z, v.w + b.w};
    } else {
      const int64_t row = static_cast<int64_t>(slot) * (TAPS - 1) + (TAPS - 1 - (back - mine));
      in[back] = ld4<T>(state + row * channels + c);
    }
  }
  float wt[4][TAPS];   // four channels' taps are 4 * TAPS consecutive elements
#pragma unroll
  for (int j = 0; j < TAPS; ++j) {
    const float4 v = ld4<T>(w + static_cast<int64_t>(c) * TAPS + 4 * j);
    const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) wt[(4 * j + i) / TAPS][(4 * j + i) % TAPS] = e[i];
  }
  const float4 ob = out_bias ? ld4<T>(out_bias + c) : float4{0.f, 0.f, 0.f, 0.f};
  float acc[4] = {ob.x, ob.y, ob.z, ob.w};
  const float now[4] = {in[0].x, in[0].y, in[0].z, in[0].w};
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = fmaf(wt[i][TAPS - 1], now[i], ((add_input & kConvAdd) ? now[i] : 0.f) + acc[i]);
#pragma unroll
  for (int back = 1; back < TAPS; ++back) {
    const float v[4] = {in[back].x, in[back].y, in[back].z, in[back].w};
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = fmaf(wt[i][TAPS - 1 - back], v[i], acc[i]);
  }
  st4<T>(out + t * out_stride + c, float4{conv_out(acc[0], add_input), conv_out(acc[1], add_input), conv_out(acc[2], add_input),
                                         conv_out(acc[3], add_input)});
}

// The same for steps of many rows whose segments are known: a lane takes kConvRows rows of its four channels, whose inputs it slides over (each is
// fetched once, not once a tap), where they and the rows they look back on belong to one request; else row by row.
//
// The first TAPS - 1 rows of a segment, the only ones that look back on its state, are left to a workgroup of the segment's own
// behind those of the rows, which reads that state, makes those rows and writes the state moved on: the update is no kernel of its own
// (4.9 us for a few kilobytes, twelve times in a prompt of eight Gufasun layers).  No other workgroup reads a state: with that branch
// beside it, for steps without segments, the kernel took 9.9 / 15.6 us where it takes 8.7 / 14.7 (2,048 x 2,560 / 6,144, bfloat16).
//
// What bounds it is a chain of trips to memory, not its bytes (21 MB at 2,048 x 2,560, 3.7 us): all inputs and slots of a lane's rows are asked
// for at once, before the weights and before anything is looked at, and SILU is known here, or every lane takes the exponential and the
// divide.  MI355X, 2,048 x 2,560 / 6,144 with the states: slots one by one, weights first, silu by the flags 9.4 / 15.6 us; silu known
// 9.1 / 15.3; inputs and slots first 8.7 / 14.6 (four rows a lane 8.3 / 14.8, sixteen 11.5 / 18.3).
constexpr int kConvRows = 8;

template <typename T, int TAPS, bool SILU>
__global__ void causal_conv_rows_kernel(const T* __restrict__ u, long long u_stride, const T* __restrict__ bias,
                                        const T* __restrict__ out_bias, const T* __restrict__ w, T* state,
                                        const int* __restrict__ slot_of_token, T* __restrict__ out, long long out_stride,
                                        int tokens, int channels, int add_input, const int* __restrict__ seg_row0,
                                        const int* __restrict__ seg_slot, int row_blocks) {
  const int t0 = blockIdx.x * kConvRows, rows = min(kConvRows, tokens - t0);
  const int c = (blockIdx.y * blockDim.x + threadIdx.x) * 4;
  if (c >= channels) return;
  // All that the rows of one request need is asked for before anything is looked at; nothing of it stands under a condition.
  const int first_back = t0 - (TAPS - 1);
  auto row_at = [&](int r) { return min(max(first_back + r, 0), tokens - 1); };
  float4 raw[kConvRows + TAPS - 1];
  int slots[kConvRows + TAPS - 1];
#pragma unroll
  for (int r = 0; r < kConvRows + TAPS - 1; ++r) raw[r] = ld4<T>(u + static_cast<int64_t>(row_at(r)) * u_stride + c), slots[r] = slot_of_token[row_at(r)];
  const float4 b = bias ? ld4<T>(bias + c) : float4{0.f, 0.f, 0.f, 0.f};
  const float4 ob = out_bias ? ld4<T>(out_bias + c) : float4{0.f, 0.f, 0.f, 0.f};
  float wt[4][TAPS];   // four channels' taps are 4 * TAPS consecutive elements
#pragma unroll
  for (int j = 0; j < TAPS; ++j) {
    const float4 v = ld4<T>(w + static_cast<int64_t>(c) * TAPS + 4 * j);
    const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) wt[(4 * j + i) / TAPS][(4 * j + i) % TAPS] = e[i];
  }
  auto row_out = [&](int t, const float4 (&in)[TAPS]) {      // in[back]: the input `back` rows before row t
    float acc[4] = {ob.x, ob.y, ob.z, ob.w};
    const float now[4] = {in[0].x, in[0].y, in[0].z, in[0].w};
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = fmaf(wt[i][TAPS - 1], now[i], ((add_input & kConvAdd) ? now[i] : 0.f) + acc[i]);
#pragma unroll
    for (int back = 1; back < TAPS; ++back) {
      const float v[4] = {in[back].x, in[back].y, in[back].z, in[back].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = fmaf(wt[i][TAPS - 1 - back], v[i], acc[i]);
    }
    constexpr int kFlags = SILU ? kConvSilu : 0;
    st4<T>(out + t * out_stride + c, float4{conv_out(acc[0], kFlags), conv_out(acc[1], kFlags), conv_out(acc[2], kFlags), conv_out(acc[3], kFlags)});
  };
  if (static_cast<int>(blockIdx.x) >= row_blocks) {
    const int seg = static_cast<int>(blockIdx.x) - row_blocks;
    const int row0 = seg_row0[seg], len = seg_row0[seg + 1] - row0;
    T* mine = state + static_cast<int64_t>(seg_slot[seg]) * (TAPS - 1) * channels + c;
    float4 old[TAPS - 1], first[TAPS - 1], fresh[TAPS - 1];
    auto input = [&](int at) {     // row `at` of the segment, at a place that exists
      const float4 v = ld4<T>(u + static_cast<int64_t>(min(max(row0 + at, 0), tokens - 1)) * u_stride + c);
      return float4{v.x + b.x, v.y + b.y, v.z + b.z, v.w + b.w};
    };
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j) old[j] = ld4<T>(mine + static_cast<int64_t>(j) * channels), first[j] = input(j), fresh[j] = input(len - (TAPS - 1) + j);
#pragma unroll
    for (int r = 0; r < TAPS - 1; ++r) {
      float4 in[TAPS];
#pragma unroll
      for (int back = 0; back < TAPS; ++back) in[back] = back <= r ? first[r - back] : old[TAPS - 1 - (back - r)];
      if (r < len) row_out(row0 + r, in);
    }
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j) {
      const int at = len - (TAPS - 1) + j;      // place among the segment's rows; negative: still in the old state
      float4 v = fresh[j];
#pragma unroll
      for (int back = 1; back < TAPS; ++back)
        if (at == -back) v = old[TAPS - 1 - back];
      st4<T>(mine + static_cast<int64_t>(j) * channels, v);
    }
    return;
  }
  bool one = first_back >= 0;
#pragma unroll
  for (int r = 0; r < kConvRows + TAPS - 1; ++r) {
    one = one & ((slots[r] == slots[TAPS - 1]) | (r - (TAPS - 1) >= rows));
    asm volatile("" : "+v"(raw[r].x));      // or the load moves down to the one row that needs it, and is waited for there
  }
  if (one) {
#pragma unroll
    for (int r = 0; r < kConvRows + TAPS - 1; ++r) raw[r] = float4{raw[r].x + b.x, raw[r].y + b.y, raw[r].z + b.z, raw[r].w + b.w};
#pragma unroll
    for (int r = 0; r < kConvRows; ++r) {
      float4 in[TAPS];
#pragma unroll
      for (int back = 0; back < TAPS; ++back) in[back] = raw[r + TAPS - 1 - back];
      if (r < rows) row_out(t0 + r, in);
    }
    return;
  }
  for (int r = 0; r < rows; ++r) {
    const int t = t0 + r, mine_slot = slot_of_token[t];
    int mine = 0;
    while (mine < TAPS - 1 && t - mine - 1 >= 0 && slot_of_token[t - mine - 1] == mine_slot) ++mine;
    if (mine < TAPS - 1) continue;      // the segment's workgroup makes it
    float4 in[TAPS];
#pragma unroll
    for (int back = 0; back < TAPS; ++back) {
      const float4 v = ld4<T>(u + (t - back) * u_stride + c);
      in[back] = float4{v.x + b.x, v.y + b.y, v.z + b.z, v.w + b.w};
    }
    row_out(t, in);
  }
}

// A step of single rows, one a request: a lane's four channels of the state belong to nobody else in the step, so it
// writes them back moved on by its row, and no second kernel has to wait for this one (decode steps of the Gufasun design had
// twelve of these pairs, 4.4 + 3.9 us each at 8 requests; together 4.6; the eight behind a norm are in the norm's kernel now).  PARTS: the input is a stack of float32 partial sums, added in order and
// rounded to T as the kernel that adds such stacks does.
// Four channels of a row from c on: the convolution's outputs (before a silu), and their state moved on (`live`: else nothing is
// written, and c is a group that exists).
template <typename T, int TAPS, bool PARTS>
__device__ __forceinline__ float4 conv_step_channels(const void* __restrict__ u, long long u_stride, int parts, long long part_stride,
                                                     const T* __restrict__ bias, const T* __restrict__ out_bias,
                                                     const T* __restrict__ w, T* __restrict__ state, int64_t slot, int64_t t, int c,
                                                     int channels, int flags, bool live) {
  T* mine = state + slot * (TAPS - 1) * channels + c;
  float4 in[TAPS];     // in[back]: the input `back` rows before this one
#pragma unroll
  for (int back = 1; back < TAPS; ++back) in[back] = ld4<T>(mine + static_cast<int64_t>(TAPS - 1 - back) * channels);
  if constexpr (PARTS) {
    const float* at = static_cast<const float*>(u) + t * u_stride + c;
    float4 v = ld4<float>(at);
    for (int s0 = 1; s0 < parts; s0 += 7) {      // seven more at a time; a jump that all lanes take together waits for no load
      float4 e[7];
#pragma unroll
      for (int j = 0; j < 7; ++j)
        if (s0 + j < parts) e[j] = ld4<float>(at + (s0 + j) * part_stride);
#pragma unroll
      for (int j = 0; j < 7; ++j)
        if (s0 + j < parts) v = float4{v.x + e[j].x, v.y + e[j].y, v.z + e[j].z, v.w + e[j].w};
    }
    in[0] = float4{to_float(from_float<T>(v.x)), to_float(from_float<T>(v.y)), to_float(from_float<T>(v.z)), to_float(from_float<T>(v.w))};
  } else {
    in[0] = ld4<T>(static_cast<const T*>(u) + t * u_stride + c);
  }
  const float4 b = bias ? ld4<T>(bias + c) : float4{0.f, 0.f, 0.f, 0.f};
  in[0] = float4{in[0].x + b.x, in[0].y + b.y, in[0].z + b.z, in[0].w + b.w};
  float wt[4][TAPS];   // four channels' taps are 4 * TAPS consecutive elements
#pragma unroll
  for (int j = 0; j < TAPS; ++j) {
    const float4 v = ld4<T>(w + static_cast<int64_t>(c) * TAPS + 4 * j);
    const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) wt[(4 * j + i) / TAPS][(4 * j + i) % TAPS] = e[i];
  }
  const float4 ob = out_bias ? ld4<T>(out_bias + c) : float4{0.f, 0.f, 0.f, 0.f};
  float acc[4] = {ob.x, ob.y, ob.z, ob.w};
  const float now[4] = {in[0].x, in[0].y, in[0].z, in[0].w};
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = fmaf(wt[i][TAPS - 1], now[i], ((flags & kConvAdd) ? now[i] : 0.f) + acc[i]);
#pragma unroll
  for (int back = 1; back < TAPS; ++back) {
    const float v[4] = {in[back].x, in[back].y, in[back].z, in[back].w};
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = fmaf(wt[i][TAPS - 1 - back], v[i], acc[i]);
  }
  if (live) {
#pragma unroll
    for (int back = 0; back < TAPS - 1; ++back) st4<T>(mine + static_cast<int64_t>(TAPS - 2 - back) * channels, in[back]);
  }
  return float4{acc[0], acc[1], acc[2], acc[3]};
}

template <typename T, int TAPS, bool PARTS>
__global__ void conv_step_kernel(const void* __restrict__ u, long long u_stride, int parts, long long part_stride,
                                 const T* __restrict__ bias, const T* __restrict__ out_bias, const T* __restrict__ w,
                                 T* __restrict__ state, const int* __restrict__ slot_of_token, T* __restrict__ out,
                                 long long out_stride, int channels, int flags) {
  const int64_t t = blockIdx.x;
  const int c = (blockIdx.y * blockDim.x + threadIdx.x) * 4;
  if (c >= channels) return;
  const float4 y = conv_step_channels<T, TAPS, PARTS>(u, u_stride, parts, part_stride, bias, out_bias, w, state, slot_of_token[t], t, c,
                                                      channels, flags, true);
  st4<T>(out + t * out_stride + c, float4{conv_out(y.x, flags), conv_out(y.y, flags), conv_out(y.z, flags), conv_out(y.w, flags)});
}

// The same with what an attention makes of its channels, q's, k's and v's one after the other: every head of q and k over the root
// mean square of its outputs, times the norm's weight and q's factor for its position, k and v into the request's pages (k a row, v
// turned).  A head of q or k is 4 * LPH channels, LPH lanes.  One kernel less to wait for in a step of single rows, which is a chain
// of such kernels: 8 rows of 6,144 channels, a convolution of 4.5 us and norms and stores of 4.5 became one of 5.3 on MI355X (a step of 8 requests
// of the Gufasun design 719 -> 709 us).
struct ConvHeads {
  const bf16* q_weight;      // [4 * LPH] or null
  const bf16* k_weight;
  float eps, temp_coef;
  int temp_every;
  const int* positions;
  const int* block_table;
  int table_stride;
  bf16* k_pages;             // [page, nkv, page_size, key_dim]
  bf16* v_pages;             // [page, nkv, value_dim, page_size]
  int nq, nkv, value_dim, page_size;
};

template <int TAPS, bool PARTS, int LPH>
__global__ __launch_bounds__(256) void conv_step_store_kernel(const void* __restrict__ u, long long u_stride, int parts,
                                                              long long part_stride, const bf16* __restrict__ bias,
                                                              const bf16* __restrict__ w, bf16* __restrict__ state,
                                                              const int* __restrict__ slot_of_token, bf16* __restrict__ q,
                                                              int channels, const ConvHeads a) {
  constexpr int Dk = 4 * LPH;
  const int64_t t = blockIdx.x;
  const int at = (blockIdx.y * blockDim.x + threadIdx.x) * 4;
  const bool live = at < channels;      // lanes behind the last channel take part in the sums below
  const int c = live ? at : channels - 4;
  const int q_end = a.nq * Dk, k_end = q_end + a.nkv * Dk;
  const int pos = a.positions[t], slot = slot_of_token[t];
  const int64_t page = a.nkv ? a.block_table[static_cast<int64_t>(slot) * a.table_stride + pos / a.page_size] : 0;
  const bool is_q = c < q_end, is_k = !is_q && c < k_end;
  const bf16* weight = is_q ? a.q_weight : a.k_weight;
  const int d = c % Dk;                 // of a head of q or k: they end on whole heads
  const float4 wv = weight ? ld4<bf16>(weight + d) : float4{1.f, 1.f, 1.f, 1.f};
  const float4 y = conv_step_channels<bf16, TAPS, PARTS>(u, u_stride, parts, part_stride, bias, nullptr, w, state, slot, t, c, channels, 0, live);
  // what the convolution alone would have written
  const float x[4] = {to_float(from_float<bf16>(y.x)), to_float(from_float<bf16>(y.y)), to_float(from_float<bf16>(y.z)),
                      to_float(from_float<bf16>(y.w))};
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) ss = fmaf(x[e], x[e], ss);
  ss = lanes_sum<LPH>(ss);
  if (!live) return;
  float f = 1.0f / sqrtf(ss / static_cast<float>(Dk) + a.eps);
  if (is_q) {
    if (a.temp_coef != 0.f) f *= 1.0f + a.temp_coef * logf(static_cast<float>((pos + 1) / a.temp_every + 1));
    st4<bf16>(q + t * q_end + c, float4{x[0] * f * wv.x, x[1] * f * wv.y, x[2] * f * wv.z, x[3] * f * wv.w});
  } else if (is_k) {
    const int64_t row = (page * a.nkv + (c - q_end) / Dk) * a.page_size + pos % a.page_size;
    st4<bf16>(a.k_pages + row * Dk + d, float4{x[0] * f * wv.x, x[1] * f * wv.y, x[2] * f * wv.z, x[3] * f * wv.w});
  } else {
    // channel j of v: element j % value_dim of kv head j / value_dim
    bf16* v = a.v_pages + (page * a.nkv * a.value_dim + (c - k_end)) * a.page_size + pos % a.page_size;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[static_cast<int64_t>(e) * a.page_size] = from_float<bf16>(x[e]);
  }
}

// One thread a (segment, channel): the new state is the last taps-1 of (old state, this step's inputs).
__global__ void conv_state_update_kernel(const void* __restrict__ u, long long u_stride, int u_dtype,
                                         const void* __restrict__ bias, int bias_dtype, void* __restrict__ state,
                                         int state_dtype, const int* __restrict__ seg_row0,
                                         const int* __restrict__ seg_slot, int channels, int taps) {
  const int seg = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= channels) return;
  const int row0 = seg_row0[seg], len = seg_row0[seg + 1] - row0;
  const int keep = taps - 1;
  const int64_t base = static_cast<int64_t>(seg_slot[seg]) * keep;
  const float b = bias ? load_as_float(bias, bias_dtype, c) : 0.f;
  float fresh[kConvMaxTaps];
#pragma unroll
  for (int j = 0; j < kConvMaxTaps; ++j) {
    if (j < keep) {
      const int at = len - keep + j;   // place among this step's rows; negative: still in the old state
      fresh[j] = at >= 0 ? load_as_float(u, u_dtype, (row0 + at) * u_stride + c) + b
                         : load_as_float(state, state_dtype, (base + j + len) * channels + c);
    }
  }
#pragma unroll
  for (int j = 0; j < kConvMaxTaps; ++j)
    if (j < keep) store_from_float(state, state_dtype, (base + j) * channels + c, fresh[j]);
}

}  // namespace arle

using namespace arle;

extern "C" int arle_conv_state_update(const void* u, long long u_stride, int u_dtype, const void* bias,
                                      int bias_dtype, void* state, int state_dtype, const int* seg_row0,
                                      const int* seg_slot, int segments, int channels, int taps, void* stream);

// u [T, channels] rows u_stride apart; out likewise; w [channels, taps] or null (then out = u + bias);
// state [slots, taps-1, channels]; slot_of_token int32 [T].
// seg_row0 int32 [segments + 1], seg_slot (or null): the segments' states are moved on by their rows (what arle_conv_state_update does).
extern "C" int arle_causal_conv(const void* u, long long u_stride, int u_dtype, const void* bias, int bias_dtype,
                                const void* out_bias, int ob_dtype, const void* w, int w_dtype,
                                void* state, int state_dtype,
                                const int* slot_of_token, void* out, long long out_stride, int out_dtype, int tokens,
                                int channels, int taps, int add_input, const int* seg_row0, const int* seg_slot, int segments,
                                void* stream) {
  const bool moves = seg_row0 != nullptr;
  if (moves && (!seg_slot || segments < 0 || !w || !state)) return static_cast<int>(hipErrorInvalidValue);
  if (tokens == 0 || channels == 0) return 0;
  if (w && (taps < 1 || taps > kConvMaxTaps)) return static_cast<int>(hipErrorInvalidValue);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const auto moved_on = [&]() {      // behind the convolution, in a kernel of its own
    const int e = launch_status();
    return e != 0 || !moves ? e
                            : arle_conv_state_update(u, u_stride, u_dtype, bias, bias_dtype, state, state_dtype, seg_row0, seg_slot, segments,
                                                     channels, taps, stream);
  };
  const auto at16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (w && taps >= 2 && taps <= 4 && channels % 4 == 0 && u_stride % 4 == 0 && out_stride % 4 == 0 && at16(u) && at16(out) &&
      at16(state) && at16(w) && at16(bias) && at16(out_bias) && u_dtype == out_dtype && w_dtype == out_dtype && state_dtype == out_dtype &&
      (!bias || bias_dtype == out_dtype) && (!out_bias || ob_dtype == out_dtype)) {
    if (tokens >= kConvManyRows && moves) {
      const int row_blocks = (tokens + kConvRows - 1) / kConvRows;
      const dim3 rgrid(static_cast<unsigned>(row_blocks + segments), (channels / 4 + 255) / 256);
#define ARLE_CONV_ROWS_AS(T, TAPS, SILU)                                                                            \
  causal_conv_rows_kernel<T, TAPS, SILU><<<rgrid, 256, 0, s>>>(static_cast<const T*>(u), u_stride, static_cast<const T*>(bias), \
                                                               static_cast<const T*>(out_bias), static_cast<const T*>(w), \
                                                               static_cast<T*>(state), slot_of_token,               \
                                                               static_cast<T*>(out), out_stride, tokens, channels, add_input, \
                                                               seg_row0, seg_slot, row_blocks)
#define ARLE_CONV_ROWS(T, TAPS)                                                                                     \
  do {                                                                                                              \
    if (add_input & kConvSilu) ARLE_CONV_ROWS_AS(T, TAPS, true); else ARLE_CONV_ROWS_AS(T, TAPS, false);            \
  } while (0)
      if (out_dtype == kF32) {
        if (taps == 2) ARLE_CONV_ROWS(float, 2); else if (taps == 3) ARLE_CONV_ROWS(float, 3); else ARLE_CONV_ROWS(float, 4);
      } else {
        if (taps == 2) ARLE_CONV_ROWS(bf16, 2); else if (taps == 3) ARLE_CONV_ROWS(bf16, 3); else ARLE_CONV_ROWS(bf16, 4);
      }
#undef ARLE_CONV_ROWS
#undef ARLE_CONV_ROWS_AS
      return launch_status();
    }
    dim3 vgrid(tokens, (channels / 4 + 255) / 256);
#define ARLE_CONV(T, TAPS)                                                                                          \
  causal_conv_vec_kernel<T, TAPS><<<vgrid, 256, 0, s>>>(static_cast<const T*>(u), u_stride, static_cast<const T*>(bias), \
                                                        static_cast<const T*>(out_bias), static_cast<const T*>(w), static_cast<const T*>(state), \
                                                        slot_of_token, static_cast<T*>(out), out_stride, channels,    \
                                                        add_input)
    if (out_dtype == kF32) {
      if (taps == 2) ARLE_CONV(float, 2); else if (taps == 3) ARLE_CONV(float, 3); else ARLE_CONV(float, 4);
    } else {
      if (taps == 2) ARLE_CONV(bf16, 2); else if (taps == 3) ARLE_CONV(bf16, 3); else ARLE_CONV(bf16, 4);
    }
#undef ARLE_CONV
    return moved_on();
  }
  dim3 grid(tokens, (channels + 255) / 256);
  causal_conv_kernel<<<grid, 256, 0, static_cast<hipStream_t>(stream)>>>(
      u, u_stride, u_dtype, bias, bias_dtype, out_bias, ob_dtype, w, w_dtype, state, state_dtype, slot_of_token, out, out_stride,
      out_dtype, channels, taps, add_input);
  return moved_on();
}

extern "C" int arle_conv_state_update(const void* u, long long u_stride, int u_dtype, const void* bias,
                                      int bias_dtype, void* state, int state_dtype, const int* seg_row0,
                                      const int* seg_slot, int segments, int channels, int taps, void* stream) {
  if (segments == 0 || channels == 0 || taps <= 1) return 0;
  if (taps > kConvMaxTaps) return static_cast<int>(hipErrorInvalidValue);
  dim3 grid(segments, (channels + 255) / 256);
  conv_state_update_kernel<<<grid, 256, 0, static_cast<hipStream_t>(stream)>>>(
      u, u_stride, u_dtype, bias, bias_dtype, state, state_dtype, seg_row0, seg_slot, channels, taps);
  return launch_status();
}

// A step of single rows, no slot twice: the convolution of each and its request's state moved on.  u [T, channels] of `dtype`
// with rows u_stride apart, or, with parts > 0, a stack of so many float32 [T, channels] part_stride apart (u_stride its rows').
// bias, out_bias [channels] or null, w [channels, taps], state [slots, taps - 1, channels] and out [T, channels] of `dtype`;
// taps 2 to 4, channels % 4 == 0, everything on the 16-byte grid.
extern "C" int arle_conv_step(const void* u, long long u_stride, int parts, long long part_stride, int dtype, const void* bias,
                              const void* out_bias, const void* w, void* state, const int* slot_of_token, void* out,
                              long long out_stride, int tokens, int channels, int taps, int flags, void* stream) {
  if (tokens == 0 || channels == 0) return 0;
  const auto at16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (taps < 2 || taps > 4 || channels % 4 != 0 || u_stride % 4 != 0 || part_stride % 4 != 0 || out_stride % 4 != 0 || parts < 0 ||
      !at16(u) || !at16(out) || !at16(state) || !at16(w) || !at16(bias) || !at16(out_bias))
    return static_cast<int>(hipErrorInvalidValue);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid(tokens, (channels / 4 + 255) / 256);
#define ARLE_CONV_STEP(T, TAPS, PARTS)                                                                                       \
  conv_step_kernel<T, TAPS, PARTS><<<grid, 256, 0, s>>>(u, u_stride, parts, part_stride, static_cast<const T*>(bias),        \
                                                        static_cast<const T*>(out_bias), static_cast<const T*>(w),           \
                                                        static_cast<T*>(state), slot_of_token, static_cast<T*>(out),         \
                                                        out_stride, channels, flags)
#define ARLE_CONV_STEP_TAPS(T, PARTS)                                                                                        \
  do {                                                                                                                       \
    if (taps == 2) ARLE_CONV_STEP(T, 2, PARTS); else if (taps == 3) ARLE_CONV_STEP(T, 3, PARTS); else ARLE_CONV_STEP(T, 4, PARTS); \
  } while (0)
  if (dtype == kF32) {
    if (parts > 0) ARLE_CONV_STEP_TAPS(float, true); else ARLE_CONV_STEP_TAPS(float, false);
  } else {
    if (parts > 0) ARLE_CONV_STEP_TAPS(bf16, true); else ARLE_CONV_STEP_TAPS(bf16, false);
  }
#undef ARLE_CONV_STEP_TAPS
#undef ARLE_CONV_STEP
  return launch_status();
}

// arle_conv_step in bfloat16 with q's and k's head norm and the store behind it (conv_step_store_kernel): channels = (nq + nkv) *
// key_dim + nkv * value_dim, key_dim 64, 128 or 256, value_dim a multiple of 4; nkv 0: q alone, no pages.  q [T, nq * key_dim].
extern "C" int arle_conv_step_store(const void* u, long long u_stride, int parts, long long part_stride, const void* bias, const void* w,
                                    void* state, const int* slot_of_token, void* q, int tokens, int taps, const void* q_weight,
                                    const void* k_weight, float eps, float temp_coef, int temp_every, const int* positions,
                                    const int* block_table, int table_stride, void* k_pages, void* v_pages, int nq, int nkv, int key_dim,
                                    int value_dim, int page_size, void* stream) {
  if (tokens == 0) return 0;
  const auto at16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (taps < 2 || taps > 4 || u_stride % 4 != 0 || part_stride % 4 != 0 || parts < 0 || !at16(u) || !at16(q) || !at16(state) || !at16(w) ||
      !at16(bias) || !at16(q_weight) || !at16(k_weight) || !at16(k_pages) || nq < 1 || nkv < 0 || value_dim % 4 != 0 ||
      (key_dim != 64 && key_dim != 128 && key_dim != 256) || (nkv > 0 && (page_size < 1 || !k_pages || !v_pages || !block_table)) ||
      (temp_coef != 0.f && temp_every < 1))
    return static_cast<int>(hipErrorInvalidValue);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int channels = (nq + nkv) * key_dim + nkv * value_dim;
  const ConvHeads heads{static_cast<const bf16*>(q_weight), static_cast<const bf16*>(k_weight), eps, temp_coef, temp_every, positions,
                        block_table, table_stride, static_cast<bf16*>(k_pages), static_cast<bf16*>(v_pages), nq, nkv, value_dim, page_size};
  const dim3 grid(tokens, (channels / 4 + 255) / 256);
#define ARLE_STORE(TAPS, PARTS, LPH)                                                                                          \
  conv_step_store_kernel<TAPS, PARTS, LPH><<<grid, 256, 0, s>>>(u, u_stride, parts, part_stride, static_cast<const bf16*>(bias), \
                                                                static_cast<const bf16*>(w), static_cast<bf16*>(state), slot_of_token, \
                                                                static_cast<bf16*>(q), channels, heads)
#define ARLE_STORE_DIM(TAPS, PARTS)                                                                                           \
  do {                                                                                                                        \
    if (key_dim == 64) ARLE_STORE(TAPS, PARTS, 16); else if (key_dim == 128) ARLE_STORE(TAPS, PARTS, 32); else ARLE_STORE(TAPS, PARTS, 64); \
  } while (0)
#define ARLE_STORE_TAPS(PARTS)                                                                                                \
  do {                                                                                                                        \
    if (taps == 2) ARLE_STORE_DIM(2, PARTS); else if (taps == 3) ARLE_STORE_DIM(3, PARTS); else ARLE_STORE_DIM(4, PARTS);     \
  } while (0)
  if (parts > 0) ARLE_STORE_TAPS(true); else ARLE_STORE_TAPS(false);
#undef ARLE_STORE_TAPS
#undef ARLE_STORE_DIM
#undef ARLE_STORE
  return launch_status();
}
