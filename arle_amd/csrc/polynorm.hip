// PolyNorm activation over the rows of a feed-forward's hidden layer:
//
//   z = u + bias;   N(y) = y / sqrt(mean_j(y_j^2) + eps)   (over the row)
//   out = a N(z) + b N(z^2) + c N(z^3) + e                 (powers element by element)
//
// so a row needs the means of z^2, z^4 and z^6; they, the roots and the sum are 32-bit.  The row stays in
// registers between the reduction and the output.  (a, b, c, e) are read from the checkpoint's tensor on
// the GPU.
#include "common.h"

#include <type_traits>

namespace arle {

constexpr int kPnThreads = 256;
constexpr int kPnWaves = kPnThreads / kWave;

template <int PER>
__global__ __launch_bounds__(kPnThreads) void polynorm_kernel(const void* __restrict__ u, long long u_stride,
                                                              int u_dtype, const void* __restrict__ bias,
                                                              int bias_dtype, const void* __restrict__ coef,
                                                              int coef_dtype, void* __restrict__ out, int out_dtype,
                                                              int width, float eps) {
  __shared__ float lds[kPnWaves];
  const int64_t r = blockIdx.x;
  float z[PER];
  float s2 = 0.f, s4 = 0.f, s6 = 0.f;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = threadIdx.x + k * kPnThreads;
    float v = 0.f;
    if (i < width) {
      v = load_as_float(u, u_dtype, r * u_stride + i);
      if (bias) v += load_as_float(bias, bias_dtype, i);
    }
    z[k] = v;
    const float q = v * v;
    s2 += q;
    s4 += q * q;
    s6 += q * q * q;
  }
  const float n = static_cast<float>(width);
  const float i1 = 1.0f / sqrtf(block_sum<kPnWaves>(s2, lds) / n + eps);
  const float i2 = 1.0f / sqrtf(block_sum<kPnWaves>(s4, lds) / n + eps);
  const float i3 = 1.0f / sqrtf(block_sum<kPnWaves>(s6, lds) / n + eps);
  const float a = load_as_float(coef, coef_dtype, 0) * i1, b = load_as_float(coef, coef_dtype, 1) * i2,
              c = load_as_float(coef, coef_dtype, 2) * i3, e = load_as_float(coef, coef_dtype, 3);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = threadIdx.x + k * kPnThreads;
    if (i < width) {
      const float v = z[k];
      store_from_float(out, out_dtype, r * width + i, fmaf(v, fmaf(v, fmaf(v, c, b), a), e));
    }
  }
}

// One element type T for input, bias, coefficients and output, a width that is a multiple of 4: four elements a lane
// and access, all loads of the row and what its end takes issued together, one barrier for the three sums: a chain of latencies for
// few rows (8 rows of 9,728 in three parts 4.4 us; a part at a time, the coefficients behind the sums and two barriers a sum 4.7),
// the bytes for many (2,048 rows, no parts, 15.0 -> 14.4 us for 80 MB).  PARTS: u is a stack of float32 partial sums instead, added in order and
// rounded to T, as the kernel that adds such stacks does.
template <typename T, int NT, int PER4, bool PARTS>
__global__ __launch_bounds__(NT) void polynorm_vec_kernel(const void* __restrict__ u, long long u_stride, int parts, long long part_stride,
                                                                  const T* __restrict__ bias, const T* __restrict__ coef,
                                                                  T* __restrict__ out, int width, float eps) {
  __shared__ float lds[3][(NT / kWave)];
  const int64_t r = blockIdx.x;
  const int last = width - 4, tid = threadIdx.x;
  // everything that the row's end takes is on its way with the row
  T a1[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) a1[j] = coef[j];
  float4 z[PER4];
  if constexpr (PARTS) {
    const float* at = static_cast<const float*>(u) + r * u_stride;
#pragma unroll
    for (int k = 0; k < PER4; ++k) z[k] = ld4<float>(at + min((tid + k * NT) * 4, last));
    // Parts at a time (a jump that all lanes take together waits for no load); two of seven accesses each, or three in float32, cost
    // many rows more in waves a SIMD than they gain (2,048 rows of 12,288, one part, 24.9 us / 29.9).  Where three are taken, 4,096 wide
    // keeps four waves a SIMD for eight, 9,728 wide four for seven, and many rows are level: 2,048 rows of one, three and six parts, one at a
    // time / three, 10.6 / 10.1, 19.0 / 18.9, 32.8 / 33.2 and 21.0 / 19.8, 42.8 / 41.5, 98.0 / 97.5; 64 rows of three parts 3.8 / 3.4 and 5.0 / 4.3.
    constexpr int G = !std::is_same<T, float>::value && PER4 <= 5 ? 3 : 1;
    for (int s0 = 1; s0 < parts; s0 += G) {
      float4 e[G][PER4];
#pragma unroll
      for (int j = 0; j < G; ++j)
        if (s0 + j < parts)
#pragma unroll
          for (int k = 0; k < PER4; ++k) e[j][k] = ld4<float>(at + (s0 + j) * part_stride + min((tid + k * NT) * 4, last));
#pragma unroll
      for (int j = 0; j < G; ++j)
        if (s0 + j < parts)
#pragma unroll
          for (int k = 0; k < PER4; ++k) z[k] = float4{z[k].x + e[j][k].x, z[k].y + e[j][k].y, z[k].z + e[j][k].z, z[k].w + e[j][k].w};
    }
#pragma unroll
    for (int k = 0; k < PER4; ++k)
      z[k] = float4{to_float(from_float<T>(z[k].x)), to_float(from_float<T>(z[k].y)), to_float(from_float<T>(z[k].z)), to_float(from_float<T>(z[k].w))};
  } else {
#pragma unroll
    for (int k = 0; k < PER4; ++k) z[k] = ld4<T>(static_cast<const T*>(u) + r * u_stride + min((tid + k * NT) * 4, last));
  }
  if (bias) {
#pragma unroll
    for (int k = 0; k < PER4; ++k) {
      const float4 b = ld4<T>(bias + min((tid + k * NT) * 4, last));
      z[k].x += b.x; z[k].y += b.y; z[k].z += b.z; z[k].w += b.w;
    }
  }
  float s2 = 0.f, s4 = 0.f, s6 = 0.f;
#pragma unroll
  for (int k = 0; k < PER4; ++k) {
    if ((tid + k * NT) * 4 < width) {
      const float e[4] = {z[k].x, z[k].y, z[k].z, z[k].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float q = e[j] * e[j];
        s2 += q;
        s4 += q * q;
        s6 += q * q * q;
      }
    }
  }
  const float n = static_cast<float>(width);
  // the three sums meet behind one barrier, each in the order of block_sum
  const float waves[3] = {wave_sum(s2), wave_sum(s4), wave_sum(s6)};
  if (tid % kWave == 0) {
#pragma unroll
    for (int j = 0; j < 3; ++j) lds[j][tid / kWave] = waves[j];
  }
  __syncthreads();
  float inv[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    float total = 0.f;
#pragma unroll
    for (int k = 0; k < NT / kWave; ++k) total += lds[j][k];
    inv[j] = 1.0f / sqrtf(total / n + eps);
  }
  const float a = to_float(a1[0]) * inv[0], b = to_float(a1[1]) * inv[1], c = to_float(a1[2]) * inv[2], e = to_float(a1[3]);
  auto poly = [&](float v) { return fmaf(v, fmaf(v, fmaf(v, c, b), a), e); };
#pragma unroll
  for (int k = 0; k < PER4; ++k) {
    const int i = (tid + k * NT) * 4;
    if (i < width) st4<T>(out + r * width + i, float4{poly(z[k].x), poly(z[k].y), poly(z[k].z), poly(z[k].w)});
  }
}

template <typename T, bool PARTS>
static int launch_pn_vec(const void* u, long long u_stride, int parts, long long part_stride, const void* bias, const void* coef,
                         void* out, int tokens, int width, float eps, hipStream_t s) {
#define ARLE_PNV(NT, PER4)                                                                                            \
  polynorm_vec_kernel<T, NT, PER4, PARTS><<<tokens, NT, 0, s>>>(u, u_stride, parts, part_stride, static_cast<const T*>(bias), \
                                                                static_cast<const T*>(coef), static_cast<T*>(out), width, eps)
  // 512 lanes where a row has more than two accesses for each; MI355X, us, 256 lanes / 512: 9,728 wide 8 rows 5.2 / 4.6, 2,048
  // 19.6 / 18.6; 12,288 wide 5.5 / 5.0, 22.4 / 20.6; 2,048 wide 3.5 / 3.7, 7.1 / 10.0.  Between 4,097 and 8,192 it is the step's rows
  // that decide: 4,100 wide 8 rows 4.4 / 4.1, 256 4.7 / 4.5, 384 5.3 / 5.4, 1,024 7.1 / 7.4, 4,096 18.0 / 21.2; 6,144 wide 256 rows
  // 5.1 / 4.8, 384 5.7 / 5.7, 1,024 8.4 / 8.7; 8,192 wide 8 rows 5.0 / 4.7, 256 5.2 / 5.1, 384 6.0 / 6.3, 768 7.5 / 8.3, 4,096 23.9 /
  // 28.2.  They count in bfloat16 only: a float32 row's sums have one order in every step.
  if (width <= 2048) {
    ARLE_PNV(256, 2);
  } else if (width <= 4096) {
    ARLE_PNV(256, 4);
  } else if (!std::is_same<T, float>::value && width <= 8192 && tokens > 256) {
    if constexpr (!std::is_same<T, float>::value) ARLE_PNV(256, 8);
  } else if (width <= 6144) {
    ARLE_PNV(512, 3);
  } else if (width <= 10240) {
    ARLE_PNV(512, 5);
  } else if (width <= 14336) {
    ARLE_PNV(512, 7);
  } else {
    ARLE_PNV(512, 12);
  }
#undef ARLE_PNV
  return launch_status();
}

}  // namespace arle

using namespace arle;

// u [T, width] rows u_stride apart; bias [width] or null; coef [4]; out [T, width] contiguous.  width <= 24576.
extern "C" int arle_polynorm(const void* u, long long u_stride, int u_dtype, const void* bias, int bias_dtype,
                             const void* coef, int coef_dtype, void* out, int out_dtype, int tokens, int width,
                             float eps, void* stream) {
  if (tokens == 0) return 0;
  if (width <= 0 || width > kPnThreads * 96) return static_cast<int>(hipErrorInvalidValue);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool aligned = reinterpret_cast<uintptr_t>(u) % 16 == 0 && u_stride % 4 == 0;
  if (width % 4 == 0 && aligned && u_dtype == out_dtype && coef_dtype == out_dtype && (!bias || bias_dtype == out_dtype)) {
    return out_dtype == kF32 ? launch_pn_vec<float, false>(u, u_stride, 0, 0, bias, coef, out, tokens, width, eps, s)
                             : launch_pn_vec<bf16, false>(u, u_stride, 0, 0, bias, coef, out, tokens, width, eps, s);
  }
#define ARLE_PN(PER)                                                                                              \
  polynorm_kernel<PER><<<tokens, kPnThreads, 0, s>>>(u, u_stride, u_dtype, bias, bias_dtype, coef, coef_dtype, out, \
                                                     out_dtype, width, eps)
  if (width <= kPnThreads * 8) {
    ARLE_PN(8);
  } else if (width <= kPnThreads * 32) {
    ARLE_PN(32);
  } else {
    ARLE_PN(96);
  }
#undef ARLE_PN
  return launch_status();
}

// The same of a stack: u float32 [parts][T][width] contiguous, added in order and rounded to `dtype`, the type of bias, coef and
// out.  width % 4 == 0, u on the 16-byte grid.
extern "C" int arle_polynorm_parts(const float* u, int parts, const void* bias, const void* coef, void* out, int dtype, int tokens,
                                   int width, float eps, void* stream) {
  if (tokens == 0) return 0;
  if (width <= 0 || width > kPnThreads * 96 || width % 4 != 0 || parts < 1 || reinterpret_cast<uintptr_t>(u) % 16 != 0)
    return static_cast<int>(hipErrorInvalidValue);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const long long part = static_cast<long long>(tokens) * width;
  return dtype == kF32 ? launch_pn_vec<float, true>(u, width, parts, part, bias, coef, out, tokens, width, eps, s)
                       : launch_pn_vec<bf16, true>(u, width, parts, part, bias, coef, out, tokens, width, eps, s);
}
