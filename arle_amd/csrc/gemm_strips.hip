// bfloat16 matrix product of one to eight rows whose sums go into the residual:  residual[M,N] += X[M,K] . W[N,K]^T, and
// with it what the root-mean-square norm behind it needs: rows[M,N] = residual * norm weight, rounded, and the sums of squares of
// the residual's rows, a strip of columns at a time.  Dividing a row by its root mean square is one number a row, and the product
// that reads `rows` can do that to its 32-bit sums (RowsArgs::sums in gemm_rows.hip), so no kernel stands between the two.
//
// What that replaces in a decode step: a product that leaves a stack of partial sums and a kernel that adds them into the residual
// and norms its rows, 4.6 us for a few kilobytes (a launch and three trips to memory one behind the other), twice a layer.
// No stack may be left for that, so K is not cut over workgroups; what is cut evenly over the compute units instead is N: one
// workgroup a strip of N / 256 columns (10 of 2,560, 16 of 4,096), whose waves share K and add through LDS, in the order of K and in pairs.
// The bound is the weights from memory.  MI355X, cold weights, us at 1 / 4 / 8 rows, product and norm before -> here:
//   2,560 x 4,096   9.0 / 9.4 / 9.8 ->  6.0 /  6.1 /  7.0      2,560 x 9,728   13.8 / 14.2 / 14.6 ->  9.9 / 10.1 / 11.7
//   4,096 x 4,096  11.6 / 12.1 / 12.6 -> 7.7 / 7.9 /  8.0      4,096 x 12,288  22.5 / 23.1 / 24.4 -> 17.5 / 17.7 / 18.0
//   2,048 x 2,048   6.9 / 7.0 / 7.3 ->  4.4 /  4.5 /  4.8      1,024 x 3,072    6.1 / 6.3 / 6.4 ->  4.7 /  5.0 /  5.3
//
//   * W as strips: [N / c][K / 32][4][c][8], strip t, step s, element (g, i, e) = W[c t + i][32 s + 8 g + e], zeros past N.  A step of
//     a strip is one run of 64 c bytes.  Lanes 16 g + i with i >= c fetch column c - 1 again; their sums are dropped.
//   * W is read once, past the caches (4,096 columns, K 12,288: 19.9 -> 18.2 us; 2,560, K 9,728: 11.6 -> 10.7).
//   * X comes from the L2, all of it to every workgroup, so it counts: 16 rows of 9,728 would take as long as W.  With up to
//     eight rows one load brings two steps, lanes i < 8 the first and lanes i >= 8 the second of row i % 8, whole lines; each
//     is multiplied with both steps' weights, and what met the other step's falls in lanes that are dropped
//     (2,560 x 9,728, 1 row: 12.9 -> 11.6 us).
//   * Eight waves with four pairs of steps ahead each; sixteen waves with two measured within 4 % either way.
//   * Whole sums mean long chains of additions: a wave keeps four sums (even and odd steps of even and odd pairs) and the waves' are added
//     two by two.  The residual is then off by less than with the stack of partial sums (error against 64 bits, stack / one chain a
//     step parity and the waves in a row / here: 2,560 x 9,728 7.7e-8 / 8.9e-8 / 6.9e-8; 2,560 x 4,096 5.6e-8 / 5.7e-8 / 4.9e-8;
//     4,096 x 12,288 16.7e-8 / 9.9e-8 / 7.5e-8), in the same time.
#include "common.h"
#include "lane_sums.h"
#include "scaled_rows.h"

namespace arle {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kStripWaves = 8, kStripAhead = 4;   // waves; pairs of steps that a wave has in flight

struct StripArgs {
  const uint16_t* x;
  int64_t ldx;
  const uint16_t* w;
  float* residual;       // [M, N]
  const void* weight;    // of the norm, [N]
  int weight_f32;
  uint16_t* rows;        // [M, N]
  float* sums;           // [M, kRowSums]
  int M, N, K, c;
};

__global__ __launch_bounds__(kStripWaves* kWave) void gemm_strips_kernel(const StripArgs a) {
  constexpr int PD = kStripAhead;
  constexpr int kPitch = 17;
  __shared__ float parts[kStripWaves * 16 * kPitch];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int c = a.c, M = a.M;
  const int pairs = a.K / 64, per = (pairs + kStripWaves - 1) / kStripWaves;
  const int p0 = min(wave * per, pairs - 1);                      // a wave without pairs fetches one that exists and multiplies nothing
  const int n = max(0, min(per, pairs - wave * per));
  const uint16_t* w = a.w + (static_cast<int64_t>(blockIdx.x) * pairs + p0) * (c * 64) + (g * c + min(i, c - 1)) * 8;
  const uint16_t* x = a.x + static_cast<int64_t>(min(i & 7, M - 1)) * a.ldx + p0 * 64 + (i >> 3) * 32 + 8 * g;
  const int step = c * 32;
  auto load_w = [&](int at) { return __builtin_bit_cast(bf16x8, __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(w + at))); };
  auto load_x = [&](int pair) { return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(x + pair * 64)); };
  bf16x8 wr[PD][2], xr[PD];
  f32x4 even[2] = {}, odd[2] = {};
  const int last = max(n - 1, 0);
#pragma unroll
  for (int u = 0; u < PD; ++u) {
    const int p = min(u, last);
    xr[u] = load_x(p);
    wr[u][0] = load_w(2 * p * step);
    wr[u][1] = load_w(2 * p * step + step);
  }
  // what the output of this thread needs is on its way before the loop
  const int row = tid >> 4, col = static_cast<int>(blockIdx.x) * c + min(tid & 15, c - 1);
  const bool mine = row < M && (tid & 15) < c && col < a.N;
  const int col_in = min(col, a.N - 1);
  const int64_t at = static_cast<int64_t>(min(row, M - 1)) * a.N + col_in;
  const float before = a.residual[at];
  const uint32_t w_raw = a.weight_f32 ? static_cast<const uint32_t*>(a.weight)[col_in]
                                      : static_cast<uint32_t>(static_cast<const uint16_t*>(a.weight)[col_in]) << 16;
  auto multiply = [&](int u) {
    even[u & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wr[u][0], xr[u], even[u & 1], 0, 0, 0);
    odd[u & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wr[u][1], xr[u], odd[u & 1], 0, 0, 0);
  };
  int base = 0;
  for (; base + 2 * PD <= n; base += PD) {
#pragma unroll
    for (int u = 0; u < PD; ++u) {
      multiply(u);
      const int p = base + u + PD;
      xr[u] = load_x(p);
      wr[u][0] = load_w(2 * p * step);
      wr[u][1] = load_w(2 * p * step + step);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (base + PD <= n) {
#pragma unroll
    for (int u = 0; u < PD; ++u) {
      multiply(u);
      const int p = base + u + PD;
      if (p < n) {
        xr[u] = load_x(p);
        wr[u][0] = load_w(2 * p * step);
        wr[u][1] = load_w(2 * p * step + step);
      }
    }
    base += PD;
  }
#pragma unroll
  for (int u = 0; u < PD; ++u)
    if (base + u < n) multiply(u);

  // lane (i, g), register r: column 4 g + r of the strip; row i and the even steps in lanes i < 8, row i - 8 and the odd ones behind
#pragma unroll
  for (int r = 0; r < 4; ++r) parts[(wave * 16 + i) * kPitch + 4 * g + r] = i < 8 ? even[0][r] + even[1][r] : odd[0][r] + odd[1][r];
  __syncthreads();
  if (tid >= kScaledRows * 16) return;
  float sum[kStripWaves];
#pragma unroll
  for (int k = 0; k < kStripWaves; ++k) sum[k] = parts[(k * 16 + row) * kPitch + (tid & 15)] + parts[(k * 16 + 8 + row) * kPitch + (tid & 15)];
#pragma unroll
  for (int half = kStripWaves / 2; half > 0; half /= 2)
#pragma unroll
    for (int k = 0; k < half; ++k) sum[k] = sum[2 * k] + sum[2 * k + 1];
  const float v = sum[0] + before;
  const float square = row_sum16(mine ? v * v : 0.f);
  if (mine) {
    a.residual[at] = v;
    a.rows[at] = f32_to_bf16_bits(v * __uint_as_float(w_raw));
  }
  if ((tid & 15) == 0 && row < M) a.sums[row * kRowSums + blockIdx.x] = square;
}

}  // namespace arle

using namespace arle;

// x [M, K] bfloat16, 1 <= M <= 8, K % 64 == 0, rows of 16-byte aligned pieces; w the strips of [N, K], 1 <= c <= 16 columns each, at most 256 of them.
// residual [M, N] float32, contiguous, is updated; rows [M, N] bfloat16 and sums [M, 256] float32 (the first ceil(N / c) of a row) are written.
extern "C" int arle_gemm_strips(const void* x, long long ldx, const void* w, void* residual, const void* weight, int weight_f32,
                                void* rows, void* sums, int M, int N, int K, int c, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > kScaledRows || K < 64 || K % 64 != 0 || ldx % 8 != 0 || c < 1 || c > 16 || (N + c - 1) / c > kRowSums ||
      static_cast<long long>(c) * K > (1 << 26) || reinterpret_cast<uintptr_t>(x) % 16 != 0 || reinterpret_cast<uintptr_t>(w) % 16 != 0)
    return static_cast<int>(hipErrorInvalidValue);
  const StripArgs a{static_cast<const uint16_t*>(x), ldx, static_cast<const uint16_t*>(w), static_cast<float*>(residual), weight,
                    weight_f32, static_cast<uint16_t*>(rows), static_cast<float*>(sums), M, N, K, c};
  gemm_strips_kernel<<<(N + c - 1) / c, kStripWaves * kWave, 0, static_cast<hipStream_t>(stream)>>>(a);
  return launch_status();
}

extern "C" int arle_gemm_strips_most() { return kRowSums; }
