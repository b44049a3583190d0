// Layer norm over rows (its own bias optional), with the residual adds of a parallel block fused in and one or two
// outputs from one pass.
//
//   x      = residual + (term_0 + bias_0) + (term_1 + bias_1)         (32-bit, written back)
//   mu     = mean_j x_j;   var = mean_j (x_j - mu)^2                   (two passes over registers)
//   out_a  = (x - mu) / sqrt(var + eps) * w_a + c_a;   out_b likewise with w_b, c_b (optional; c: the norm's own bias,
//            of the weight's type, optional)
//
// A block whose mixer and feed-forward both read the same residual hands on two deltas, each of which may be
// a stack of float32 partial products (added in the order of the stack) and may carry the bias of the
// projection that made it; the next block's two norms are of that same sum, so they share the statistics.
// With `rows` given (the final norm before the head) the rows named there are read for the last time and
// the sum is not written back.
#include "common.h"

#include <type_traits>

namespace arle {

constexpr int kLnThreads = 256;
constexpr int kLnWaves = kLnThreads / kWave;

struct LnTerm {
  const void* data;     // [n_stack][T][width], or null
  int n_stack;
  long long stack_stride;
  int dtype;
  const void* bias;     // [width] or null
  int bias_dtype;
};

// PER elements a thread (width <= kLnThreads * PER), the row stays in registers.
template <int PER>
__global__ __launch_bounds__(kLnThreads) void add_layernorm_kernel(
    float* __restrict__ residual, LnTerm t0, LnTerm t1, const void* __restrict__ wa, const void* __restrict__ wb,
    int w_dtype, void* __restrict__ out_a, void* __restrict__ out_b, int out_dtype, const int* __restrict__ rows,
    int width, float eps, const void* __restrict__ ca, const void* __restrict__ cb) {
  __shared__ float lds[kLnWaves];
  const int r = blockIdx.x;
  const int64_t src = rows ? rows[r] : r;
  float* res = residual + src * width;
  float x[PER];
  float sum = 0.f;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = threadIdx.x + k * kLnThreads;
    float v = 0.f;
    if (i < width) {
      v = res[i];
      if (t0.data) {
        float d = load_as_float(t0.data, t0.dtype, src * width + i);
        for (int s = 1; s < t0.n_stack; ++s) d += load_as_float(t0.data, t0.dtype, s * t0.stack_stride + src * width + i);
        if (t0.bias) d += load_as_float(t0.bias, t0.bias_dtype, i);
        v += d;
      }
      if (t1.data) {
        float d = load_as_float(t1.data, t1.dtype, src * width + i);
        for (int s = 1; s < t1.n_stack; ++s) d += load_as_float(t1.data, t1.dtype, s * t1.stack_stride + src * width + i);
        if (t1.bias) d += load_as_float(t1.bias, t1.bias_dtype, i);
        v += d;
      }
      if (!rows && (t0.data || t1.data)) res[i] = v;
    }
    x[k] = v;
    sum += v;
  }
  const float mu = block_sum<kLnWaves>(sum, lds) / static_cast<float>(width);
  float sq = 0.f;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = threadIdx.x + k * kLnThreads;
    const float d = i < width ? x[k] - mu : 0.f;
    x[k] = d;
    sq += d * d;
  }
  const float inv = 1.0f / sqrtf(block_sum<kLnWaves>(sq, lds) / static_cast<float>(width) + eps);
  const int64_t o = static_cast<int64_t>(r) * width;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = threadIdx.x + k * kLnThreads;
    if (i < width) {
      const float n = x[k] * inv;
      store_from_float(out_a, out_dtype, o + i, fmaf(n, load_as_float(wa, w_dtype, i), ca ? load_as_float(ca, w_dtype, i) : 0.f));
      if (out_b) store_from_float(out_b, out_dtype, o + i, fmaf(n, load_as_float(wb, w_dtype, i), cb ? load_as_float(cb, w_dtype, i) : 0.f));
    }
  }
}

// The same for the usual types: terms that are float32 (a projection's 32-bit output or its stack of partial
// products), biases, weights and outputs of one type TA, a width that is a multiple of 4.  Four elements a lane and
// access, every load of a row issued without a condition on data, before anything is stored.  Bound by the latency of that one trip to
// memory and of two reductions for few rows, by the memory for many (2,048 rows of 2,560, terms of one and two parts: 5.9 TB/s).
//
// CT > 0: the rows are single ones of different requests, and the first norm's output goes through a causal convolution of CT taps
// with its input added before it is written (LnConv): a lane holds the same four channels of the row, of the taps and of the
// request's state, which it moves on, and everything it needs is on its way before the reductions.  One kernel less to
// wait for in front of every layer; decode steps of 8 rows of 2,560, MI355X: norm 4.8 + convolution 4.4 us before.
// Four consecutive elements as they are stored: widened where they are used, as a conversion waits for its load.
template <typename T>
using Raw4 = std::conditional_t<std::is_same<T, float>::value, float4, uint2>;

template <typename T>
__device__ __forceinline__ Raw4<T> ld_raw(const T* p) { return *reinterpret_cast<const Raw4<T>*>(p); }
template <typename T>
__device__ __forceinline__ float4 widen(const Raw4<T>& v) { return ld4<T>(reinterpret_cast<const T*>(&v)); }

template <typename TA>
struct LnConv {
  const TA* w;         // [width, CT]
  TA* state;           // [slots, CT - 1, width]
  const int* slot;     // of every row
};

template <typename TA, int NT, int PER4, int CT, int U>
__global__ __launch_bounds__(NT) void add_layernorm_vec_kernel(
    float* __restrict__ residual, const float* __restrict__ t0, int n0, long long s0, const TA* __restrict__ b0,
    const float* __restrict__ t1, int n1, long long s1, const TA* __restrict__ b1, const TA* __restrict__ wa,
    const TA* __restrict__ wb, TA* __restrict__ out_a, TA* __restrict__ out_b, const int* __restrict__ rows, int width,
    float eps, const TA* __restrict__ ca, const TA* __restrict__ cb, const LnConv<TA> conv) {
  __shared__ float lds[2][(NT / kWave)];
  const int r = blockIdx.x;
  const int64_t src = rows ? rows[r] : r;
  const int64_t base = src * width;
  const int last = width - 4, tid = threadIdx.x;
  float4 x[PER4];
#pragma unroll
  for (int k = 0; k < PER4; ++k) x[k] = ld4<float>(residual + base + min((tid + k * NT) * 4, last));
  // U > 0: both terms have at most U parts, and all that there are are on their way with the row (a condition that is the same for
  // the whole workgroup is a jump and waits for no load, as long as nothing is made of the value in front of its use)
  [[maybe_unused]] float4 e0[U > 0 ? U : 1][PER4], e1[U > 0 ? U : 1][PER4];
  if constexpr (U > 0) {
    const float *p0 = t0 + base, *p1 = t1 + base;
    const int last0 = t0 ? n0 - 1 : -1, last1 = t1 ? n1 - 1 : -1;
#pragma unroll
    for (int j = 0; j < U; ++j)
      if (j <= last0)
#pragma unroll
        for (int k = 0; k < PER4; ++k) e0[j][k] = ld4<float>(p0 + j * s0 + min((tid + k * NT) * 4, last));
#pragma unroll
    for (int j = 0; j < U; ++j)
      if (j <= last1)
#pragma unroll
        for (int k = 0; k < PER4; ++k) e1[j][k] = ld4<float>(p1 + j * s1 + min((tid + k * NT) * 4, last));
  }
  [[maybe_unused]] Raw4<TA> bias0[PER4], bias1[PER4];
  if constexpr (U > 0) {
#pragma unroll
    for (int k = 0; k < PER4; ++k) {
      if (t0 && b0) bias0[k] = ld_raw<TA>(b0 + min((tid + k * NT) * 4, last));
      if (t1 && b1) bias1[k] = ld_raw<TA>(b1 + min((tid + k * NT) * 4, last));
    }
  }
  [[maybe_unused]] auto add_fetched = [&](const auto& e, int n, const Raw4<TA> (&bias)[PER4], bool biased) {
#pragma unroll
    for (int k = 0; k < PER4; ++k) {
      float4 d = e[0][k];
#pragma unroll
      for (int j = 1; j < U; ++j)
        if (j < n) d.x += e[j][k].x, d.y += e[j][k].y, d.z += e[j][k].z, d.w += e[j][k].w;
      if (biased) {
        const float4 b = widen<TA>(bias[k]);
        d.x += b.x; d.y += b.y; d.z += b.z; d.w += b.w;
      }
      x[k].x += d.x; x[k].y += d.y; x[k].z += d.z; x[k].w += d.w;
    }
  };
  [[maybe_unused]] auto add_term = [&](const float* t, int n, long long stride, const TA* bias) {
    float4 d[PER4];
#pragma unroll
    for (int k = 0; k < PER4; ++k) d[k] = ld4<float>(t + base + min((tid + k * NT) * 4, last));
    // the parts of a stack are fetched several at a time without a condition (a part past the last is the last one again, fetched
    // and dropped), so that their loads are in flight together; they are added in the stack's order.  Two at a time where a lane
    // has eight elements and their taps besides: more do not fit the registers of 1,024 lanes (8 rows of 8,192, taps 4, two terms of
    // 4 and 2 parts, us, eight / four / two at a time: bfloat16 12.4 / 9.1 / 8.6, float32 24.7 / 13.5 / 9.8, which spill; 5,120 wide 8.2 /
    // 7.1 / 6.7 and 9.6 / 7.6 / 7.4)
    constexpr int G = PER4 == 2 && NT > 256 && CT > 0 ? 2 : PER4 <= 4 ? 8 : (PER4 <= 8 ? 4 : 2);
    for (int s0 = 1; s0 < n; s0 += G) {
      float4 e[G][PER4];
#pragma unroll
      for (int j = 0; j < G; ++j) {
        const long long at = min(s0 + j, n - 1) * stride + base;
#pragma unroll
        for (int k = 0; k < PER4; ++k) e[j][k] = ld4<float>(t + at + min((tid + k * NT) * 4, last));
      }
#pragma unroll
      for (int j = 0; j < G; ++j) {
        if (s0 + j < n) {
#pragma unroll
          for (int k = 0; k < PER4; ++k) {
            d[k].x += e[j][k].x; d[k].y += e[j][k].y; d[k].z += e[j][k].z; d[k].w += e[j][k].w;
          }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < PER4; ++k) {
      if (bias) {
        const float4 e = ld4<TA>(bias + min((tid + k * NT) * 4, last));
        d[k].x += e.x; d[k].y += e.y; d[k].z += e.z; d[k].w += e.w;
      }
      x[k].x += d[k].x; x[k].y += d[k].y; x[k].z += d[k].z; x[k].w += d[k].w;
    }
  };
  // the norm weights are fetched now, not behind the two reductions that their use waits for
  const TA* weights[4] = {wa, wb, ca, cb};
  Raw4<TA> w_raw[4][PER4];
#pragma unroll
  for (int m = 0; m < 4; ++m)
    if (weights[m])
#pragma unroll
      for (int k = 0; k < PER4; ++k) w_raw[m][k] = ld_raw<TA>(weights[m] + min((tid + k * NT) * 4, last));
  constexpr int BACK = CT > 0 ? CT - 1 : 1, TAPS = CT > 0 ? CT : 1;
  [[maybe_unused]] Raw4<TA> before[PER4][BACK], tap[PER4][TAPS];   // the rows before this one, oldest first; 4 channels' taps
  [[maybe_unused]] TA* mine = nullptr;
  if constexpr (CT > 0) {
    mine = conv.state + static_cast<int64_t>(conv.slot[r]) * (CT - 1) * width;
#pragma unroll
    for (int k = 0; k < PER4; ++k) {
      const int i = min((tid + k * NT) * 4, last);
#pragma unroll
      for (int j = 0; j < CT - 1; ++j) before[k][j] = ld_raw<TA>(mine + static_cast<int64_t>(j) * width + i);
#pragma unroll
      for (int j = 0; j < CT; ++j) tap[k][j] = ld_raw<TA>(conv.w + static_cast<int64_t>(i) * CT + 4 * j);
    }
  }
  if constexpr (U > 0) {
    if (t0) add_fetched(e0, n0, bias0, b0);
    if (t1) add_fetched(e1, n1, bias1, b1);
  } else {
    if (t0) add_term(t0, n0, s0, b0);
    if (t1) add_term(t1, n1, s1, b1);
  }
  float sum = 0.f;
#pragma unroll
  for (int k = 0; k < PER4; ++k) {
    const int i = (tid + k * NT) * 4;
    if (i < width) {
      if (!rows && (t0 || t1)) st4<float>(residual + base + i, x[k]);
      sum += (x[k].x + x[k].y) + (x[k].z + x[k].w);
    }
  }
  const float mu = block_sum_once<NT / kWave>(sum, lds[0]) / static_cast<float>(width);
  float sq = 0.f;
#pragma unroll
  for (int k = 0; k < PER4; ++k) {
    const int i = (tid + k * NT) * 4;
    x[k].x -= mu; x[k].y -= mu; x[k].z -= mu; x[k].w -= mu;
    if (i < width) sq += (x[k].x * x[k].x + x[k].y * x[k].y) + (x[k].z * x[k].z + x[k].w * x[k].w);
  }
  const float inv = 1.0f / sqrtf(block_sum_once<NT / kWave>(sq, lds[1]) / static_cast<float>(width) + eps);
  const int64_t o = static_cast<int64_t>(r) * width;
#pragma unroll
  for (int k = 0; k < PER4; ++k) {
    const int i = (tid + k * NT) * 4;
    if (i < width) {
      const float4 w = widen<TA>(w_raw[0][k]), c = ca ? widen<TA>(w_raw[2][k]) : float4{0.f, 0.f, 0.f, 0.f};
      float4 a = float4{fmaf(x[k].x * inv, w.x, c.x), fmaf(x[k].y * inv, w.y, c.y), fmaf(x[k].z * inv, w.z, c.z), fmaf(x[k].w * inv, w.w, c.w)};
      if constexpr (CT > 0) {
        // the convolution reads what the norm alone would have written, and adds in the order of conv_step
        const float now[4] = {to_float(from_float<TA>(a.x)), to_float(from_float<TA>(a.y)), to_float(from_float<TA>(a.z)), to_float(from_float<TA>(a.w))};
        float wt[4][TAPS], acc[4];
#pragma unroll
        for (int j = 0; j < CT; ++j) {
          const float4 taps = widen<TA>(tap[k][j]);
          const float e[4] = {taps.x, taps.y, taps.z, taps.w};
#pragma unroll
          for (int q = 0; q < 4; ++q) wt[(4 * j + q) / TAPS][(4 * j + q) % TAPS] = e[q];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = fmaf(wt[q][TAPS - 1], now[q], now[q]);
#pragma unroll
        for (int j = CT - 2; j >= 0; --j) {
          const float4 in = widen<TA>(before[k][j]);
          const float v[4] = {in.x, in.y, in.z, in.w};
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[q] = fmaf(wt[q][j], v[q], acc[q]);
        }
#pragma unroll
        for (int j = 0; j + 1 < CT - 1; ++j) *reinterpret_cast<Raw4<TA>*>(mine + static_cast<int64_t>(j) * width + i) = before[k][j + 1];
        st4<TA>(mine + static_cast<int64_t>(CT - 2) * width + i, float4{now[0], now[1], now[2], now[3]});
        a = float4{acc[0], acc[1], acc[2], acc[3]};
      }
      st4<TA>(out_a + o + i, a);
      if (out_b) {
        const float4 v = widen<TA>(w_raw[1][k]), e = cb ? widen<TA>(w_raw[3][k]) : float4{0.f, 0.f, 0.f, 0.f};
        st4<TA>(out_b + o + i, float4{fmaf(x[k].x * inv, v.x, e.x), fmaf(x[k].y * inv, v.y, e.y), fmaf(x[k].z * inv, v.z, e.z),
                                      fmaf(x[k].w * inv, v.w, e.w)});
      }
    }
  }
}

// Workgroups as wide as the row where that is more than 2,048 elements: nearly every load of a row is then on its way at once
// and few are of the row's end again.  MI355X, terms of one and two parts (six up to 64 rows), 256 lanes / as here, us:
// 2,560 wide, 8 rows 6.0 / 4.7, 2,048 39.3 / 32.7, 8,192 146.8 / 109.4; 4,096 wide 6.1 / 5.7, 45.9 / 40.7, 172.8 / 152.0; 5,120
// wide 8.2 / 6.2, 2,048 rows 68.7 / 60.8.  Narrower rows need several a compute unit (1,536 wide, 2,048 rows 20.0 / 27.1), and
// so do many rows beyond 5,120: 6,144 wide 8 rows 8.4 / 7.8, 256 9.5 / 9.5, 512 19.6 / 17.7, 1,536 48.4 / 46.8, 2,048 62.2 / 60.7,
// 4,096 139.5 / 158.9; 8,192 wide 8.7 / 7.9, 11.3 / 10.6, 23.6 / 20.1, 62.6 / 55.2, 87.6 / 86.6, 172.7 / 177.5 (elsewhere 2,048 rows 86.2 /
// 89.8).  In bfloat16: a float32 row's sums have one order in every step, so the width alone chooses there.
struct LnShape {
  int threads, per_lane;   // lanes a row, groups of four elements a lane
};
constexpr LnShape ln_shape(int width, int n_rows, bool f32, int taps) {
  if (width <= 2048) return {256, width <= 1024 ? 1 : 2};
  if (width <= 2560) return {640, 1};
  if (width <= 4096) return {1024, 1};
  if (width <= 5120) return {640, 2};
  if (width <= 8192) return f32 || n_rows < 2048 || taps > 0 ? LnShape{1024, 2} : LnShape{256, 8};
  return {256, 16};
}

// How many parts of both terms a lane fetches together: two or eight where the registers hold them (ln_holds), else one term after
// the other; the order of the sums is the same.
// MI355X, terms of 4 and 6 parts / 1 and 2 / 1 and 1, us, term after term with the parts past the last fetched again / as here: 8 rows
// of 2,560 4.9, 4.1, 3.6 / 4.1, 3.4, 3.3, with the convolution 5.6, 4.7, 4.2 / 4.6, 3.9, 3.9; 2,048 rows - 23.9, 19.7 / - 21.5, 18.8
// (126 and 105 MB); 8 rows of 5,120 6.9, 5.3, 4.3 / 5.7, 4.2, 4.1; 2,048 rows - 50.1, 37.0 / - 38.7, 33.2; 512 rows of 8,192 - 20.5, 17.0
// / - 18.9, 16.9, of one term of one part 14.1 / 13.1.  Only rows of 4,096 with two terms of one part, of which there are many, lose: 512
// 8.8 / 8.4, 2,048 28.6 / 29.6, 4,096 51.9 / 52.5, and so they do one term after the other (2,048 29.8).  (Eight parts of eight float32 elements a lane spill: 8 rows of 5,120 7.0 / 9.1.)
constexpr bool ln_holds(int threads, int per_lane, int taps, bool f32, int parts) {
  return parts == 2 ? per_lane <= 2 && !(per_lane == 2 && threads > 640 && taps > 0)
                    : per_lane == 1 || (per_lane == 2 && taps == 0 && (threads <= 256 || (threads <= 640 && !f32)));
}
// Eight at a time pay while the rows wait for one trip to memory; with more rows than the chip has at work at once it is the rows beside
// each other that hide the trips, and the registers of eight parts leave room for fewer.  MI355X, bfloat16, us, one term after the other /
// eight together: 2,560 wide, terms of 6 and 6 parts, 64 rows 4.6 / 4.1, 256 6.7 / 6.0, 384 10.8 / 11.5, 1,024 24.2 / 25.6, one of 3 parts 256
// rows 4.3 / 3.8, 1,024 11.8 / 13.4; 4,096 wide, 6 parts, 256 5.5 / 5.1, 384 10.4 / 11.2, 2,048 41.7 / 48.1; 1,024 wide, 6 and 6, 768 8.2 / 7.7,
// 1,024 11.0 / 11.2, 2,048 19.3 / 21.9; 2,048 wide, 256 5.2 / 4.6, 384 9.1 / 9.3 (8 parts 5.2 / 4.8), 512 11.3 / 12.1.  Workgroups of 640 lanes with
// two groups each (5,120 wide) are level or ahead at all rows: 6 parts, 512 rows 16.9 / 16.4, 2,048 62.8 / 60.7.
constexpr int ln_ahead(int threads, int per_lane, int taps, bool f32, int parts, int n_rows) {
  if (parts <= 2) return ln_holds(threads, per_lane, taps, f32, 2) ? 2 : 0;
  const int rows_most = threads <= 256 ? 768 / per_lane : (per_lane == 1 ? 256 : 1 << 30);
  return parts <= 8 && n_rows <= rows_most && ln_holds(threads, per_lane, taps, f32, 8) ? 8 : 0;
}

template <typename TA>
static int launch_ln_vec(float* residual, const LnTerm& t0, const LnTerm& t1, const void* wa, const void* wb, void* out_a,
                         void* out_b, const int* rows, int n_rows, int width, float eps, const void* ca, const void* cb,
                         const LnConv<TA>& conv, int taps, hipStream_t s) {
#define ARLE_LNV_U(NT, PER4, CT, U)                                                                                 \
  add_layernorm_vec_kernel<TA, NT, PER4, CT, U><<<n_rows, NT, 0, s>>>(                                                  \
      residual, static_cast<const float*>(t0.data), t0.n_stack, t0.stack_stride, static_cast<const TA*>(t0.bias),  \
      static_cast<const float*>(t1.data), t1.n_stack, t1.stack_stride, static_cast<const TA*>(t1.bias),            \
      static_cast<const TA*>(wa), static_cast<const TA*>(wb), static_cast<TA*>(out_a), static_cast<TA*>(out_b), rows, \
      width, eps, static_cast<const TA*>(ca), static_cast<const TA*>(cb), conv)
#define ARLE_LNV_CT(NT, PER4, CT)                                                     \
  do {                                                                                \
    constexpr bool f32 = std::is_same<TA, float>::value;                              \
    constexpr int two = ln_holds(NT, PER4, CT, f32, 2) ? 2 : 0, eight = ln_holds(NT, PER4, CT, f32, 8) ? 8 : 0; \
    const int ahead = ln_ahead(NT, PER4, CT, f32, parts, n_rows);                     \
    if (two && ahead == 2) ARLE_LNV_U(NT, PER4, CT, two);                             \
    else if (eight && ahead == 8) ARLE_LNV_U(NT, PER4, CT, eight);                    \
    else ARLE_LNV_U(NT, PER4, CT, 0);                                                 \
  } while (0)
#define ARLE_LNV(NT, PER4)                                                            \
  do {                                                                                \
    if (taps == 0) ARLE_LNV_CT(NT, PER4, 0); else if (taps == 2) ARLE_LNV_CT(NT, PER4, 2); \
    else if (taps == 3) ARLE_LNV_CT(NT, PER4, 3); else ARLE_LNV_CT(NT, PER4, 4);      \
  } while (0)
  const int parts = max(t0.data ? t0.n_stack : 0, t1.data ? t1.n_stack : 0);
  const LnShape shape = ln_shape(width, n_rows, std::is_same<TA, float>::value, taps);
  const int lanes = shape.threads, each = shape.per_lane;
  if (lanes == 256 && each == 1) {
    ARLE_LNV(256, 1);
  } else if (lanes == 256 && each == 2) {
    ARLE_LNV(256, 2);
  } else if (lanes == 640 && each == 1) {
    ARLE_LNV(640, 1);
  } else if (lanes == 1024 && each == 1) {
    ARLE_LNV(1024, 1);
  } else if (lanes == 640) {
    ARLE_LNV(640, 2);
  } else if (lanes == 1024) {
    ARLE_LNV(1024, 2);
  } else if (each == 8) {
    if constexpr (!std::is_same<TA, float>::value) ARLE_LNV_CT(256, 8, 0);
  } else {
    ARLE_LNV_CT(256, 16, 0);
  }
#undef ARLE_LNV
#undef ARLE_LNV_CT
#undef ARLE_LNV_U
  return launch_status();
}

}  // namespace arle

using namespace arle;

// How many parts of both terms a lane of the vector form fetches together (0: one term after the other); parts: the larger of the two stacks.
extern "C" int arle_layernorm_parts_ahead(int width, int n_rows, int parts, int taps, int dtype) {
  const LnShape shape = ln_shape(width, n_rows, dtype == kF32, taps);
  return ln_ahead(shape.threads, shape.per_lane, taps, dtype == kF32, parts, n_rows);
}

// residual float32 [T, width] contiguous.  term*: null, [T, width] (n_stack 1) or a stack; bias*: null or [width].
// out_a, out_b (out_b and wb may be null): [n_rows, width] contiguous of out_dtype.  width <= 16384.
// norm_bias_a, norm_bias_b: the norms' own biases, [width] of the weights' type, or null.
extern "C" int arle_add_layernorm(float* residual, const void* term0, int n0, long long stride0, int dtype0,
                                  const void* bias0, int bias_dtype0, const void* term1, int n1, long long stride1,
                                  int dtype1, const void* bias1, int bias_dtype1, const void* wa, const void* wb,
                                  int w_dtype, void* out_a, void* out_b, int out_dtype, const int* rows, int n_rows,
                                  int width, float eps, const void* norm_bias_a, const void* norm_bias_b, void* stream) {
  if (n_rows == 0) return 0;
  if (width <= 0 || width > kLnThreads * 64) return static_cast<int>(hipErrorInvalidValue);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const LnTerm t0{term0, n0, stride0, dtype0, bias0, bias_dtype0};
  const LnTerm t1{term1, n1, stride1, dtype1, bias1, bias_dtype1};
  // the usual case: float32 terms, everything else of the output's type, whole groups of four
  const auto fits = [&](const LnTerm& t) { return !t.data || (t.dtype == kF32 && (!t.bias || t.bias_dtype == out_dtype)); };
  if (width % 4 == 0 && fits(t0) && fits(t1) && w_dtype == out_dtype) {
    return out_dtype == kF32 ? launch_ln_vec<float>(residual, t0, t1, wa, wb, out_a, out_b, rows, n_rows, width, eps, norm_bias_a, norm_bias_b, {}, 0, s)
                             : launch_ln_vec<bf16>(residual, t0, t1, wa, wb, out_a, out_b, rows, n_rows, width, eps, norm_bias_a, norm_bias_b, {}, 0, s);
  }
#define ARLE_LN(PER)                                                                                          \
  add_layernorm_kernel<PER><<<n_rows, kLnThreads, 0, s>>>(residual, t0, t1, wa, wb, w_dtype, out_a, out_b, \
                                                          out_dtype, rows, width, eps, norm_bias_a, norm_bias_b)
  if (width <= kLnThreads * 4) {
    ARLE_LN(4);
  } else if (width <= kLnThreads * 16) {
    ARLE_LN(16);
  } else {
    ARLE_LN(64);
  }
#undef ARLE_LN
  return launch_status();
}

// Every row a single one of a request (no slot twice): as arle_add_layernorm, with a convolution of `taps` taps and its own input on
// the first norm's output and the requests' states moved on.  Terms float32, everything else of `dtype` and on the 16-byte grid;
// width a multiple of 4 up to 8,192, taps 2 to 4.  conv_w [width, taps], conv_state [slots, taps - 1, width].
extern "C" int arle_add_layernorm_conv(float* residual, const void* term0, int n0, long long stride0, const void* bias0, const void* term1,
                                       int n1, long long stride1, const void* bias1, const void* wa, const void* wb, void* out_a,
                                       void* out_b, int dtype, int n_rows, int width, float eps, const void* norm_bias_a,
                                       const void* norm_bias_b, const void* conv_w, void* conv_state, const int* slot_of_row, int taps,
                                       void* stream) {
  if (n_rows == 0) return 0;
  const auto at16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (width <= 0 || width > 8192 || width % 4 != 0 || taps < 2 || taps > 4 || (dtype != kF32 && dtype != kBF16) || !at16(conv_w) || !at16(conv_state))
    return static_cast<int>(hipErrorInvalidValue);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const LnTerm t0{term0, n0, stride0, kF32, bias0, dtype}, t1{term1, n1, stride1, kF32, bias1, dtype};
  return dtype == kF32 ? launch_ln_vec<float>(residual, t0, t1, wa, wb, out_a, out_b, nullptr, n_rows, width, eps, norm_bias_a, norm_bias_b,
                                              {static_cast<const float*>(conv_w), static_cast<float*>(conv_state), slot_of_row}, taps, s)
                       : launch_ln_vec<bf16>(residual, t0, t1, wa, wb, out_a, out_b, nullptr, n_rows, width, eps, norm_bias_a, norm_bias_b,
                                             {static_cast<const bf16*>(conv_w), static_cast<bf16*>(conv_state), slot_of_row}, taps, s);
}
