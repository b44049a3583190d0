// Shared device helpers for the gfx950 kernels: element types, 64-lane wave
// reductions and the launch-status convention of the C entry points.
//
// Every entry point is `extern "C" int arle_<name>(..., void* stream)`; it checks
// nothing about shapes (the Python wrapper does, on the host, before the call),
// launches on the given HIP stream and returns the hipError_t of the launch.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <initializer_list>

#include "once_a_device.h"

namespace arle {

constexpr int kWave = 64;

// bfloat16 is carried as its 16 raw bits.
struct bf16 {
  uint16_t bits;
};

__device__ __forceinline__ float to_float(float v) { return v; }
__device__ __forceinline__ float to_float(bf16 v) {
  return __uint_as_float(static_cast<uint32_t>(v.bits) << 16);
}

// Round to nearest, ties to even (the hardware conversion of gfx950, v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) {
  return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f));
}

// Two floats to two bfloat16 in one register: a in the low half, b in the high half.
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  const f32x2_t v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

template <typename T>
__device__ __forceinline__ T from_float(float v);
template <>
__device__ __forceinline__ float from_float<float>(float v) {
  return v;
}
template <>
__device__ __forceinline__ bf16 from_float<bf16>(float v) {
  bf16 r;
  r.bits = f32_to_bf16_bits(v);
  return r;
}

// Reductions over the lanes of a wave, all of them active, by moves inside the vector unit: a shuffle is a trip through the LDS
// unit, and the six of a wave's sum stand one behind the other (MI355X: a layer norm of 8 rows of 2,560, two such sums, 3.4 us
// with shuffles, 3.2 so; a decode step of one request of the Qwen3-4B shape, with the sums of the attention, 2,436 -> 2,400).
// A value of lane i and the value of lane i ^ 32, or of i ^ 16, in the same order in both lanes:
struct LanePair {
  float lo, hi;
};
__device__ __forceinline__ LanePair across32(float x) {
  const unsigned bits = __float_as_uint(x);
  const auto r = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
  return {__uint_as_float(r[0]), __uint_as_float(r[1])};
}
__device__ __forceinline__ LanePair across16(float x) {
  const unsigned bits = __float_as_uint(x);
  const auto r = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
  return {__uint_as_float(r[0]), __uint_as_float(r[1])};
}
template <int CTRL>
__device__ __forceinline__ float row_move(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// Over groups of LANES neighbouring lanes (a power of two from 16 on): the lanes that are LANES / 2 apart first, then LANES / 4, ..., 1,
// the order and with it the bits of a butterfly of exchanges with lane ^ 32, 16, 8, 4, 2, 1.  (A row of sixteen turned by 8 holds lane
// ^ 8; after that step lanes 8 apart hold the same, so that a turn by 4 brings the value of lane ^ 4.)
template <int LANES, typename Join>
__device__ __forceinline__ float lanes_join(float v, Join join) {
  static_assert(LANES == 16 || LANES == 32 || LANES == 64, "whole rows of sixteen lanes");
  if constexpr (LANES == 64) {
    const LanePair p = across32(v);
    v = join(p.lo, p.hi);
  }
  if constexpr (LANES >= 32) {
    const LanePair p = across16(v);
    v = join(p.lo, p.hi);
  }
  v = join(v, row_move<0x128>(v));   // row_ror:8
  v = join(v, row_move<0x124>(v));   // row_ror:4
  v = join(v, row_move<0x4E>(v));    // quad_perm [2, 3, 0, 1]
  return join(v, row_move<0xB1>(v));   // quad_perm [1, 0, 3, 2]
}
template <int LANES>
__device__ __forceinline__ float lanes_sum(float v) {
  if constexpr (LANES >= 16) {
    return lanes_join<LANES>(v, [](float a, float b) { return a + b; });
  } else {
#pragma unroll
    for (int off = LANES / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
  }
}
__device__ __forceinline__ float wave_sum(float v) { return lanes_sum<kWave>(v); }
__device__ __forceinline__ float wave_max(float v) {
  return lanes_join<kWave>(v, [](float a, float b) { return fmaxf(a, b); });
}

// Sum over a block of `kWaves` waves; every thread gets the result.  The order
// of additions is fixed (butterfly inside a wave, then waves 0..n-1), so a row's
// reduction never depends on what else is in the launch.
template <int kWaves>
__device__ __forceinline__ float block_sum_once(float v, float* lds /* [kWaves], used for nothing else */) {
  v = wave_sum(v);
  const int wave = threadIdx.x / kWave;
  if ((threadIdx.x % kWave) == 0) lds[wave] = v;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int i = 0; i < kWaves; ++i) total += lds[i];
  return total;
}
// The same with words that are free again behind it.
template <int kWaves>
__device__ __forceinline__ float block_sum(float v, float* lds /* [kWaves] */) {
  const float total = block_sum_once<kWaves>(v, lds);
  __syncthreads();
  return total;
}

template <int kWaves>
__device__ __forceinline__ float block_max(float v, float* lds /* [kWaves] */) {
  v = wave_max(v);
  const int wave = threadIdx.x / kWave;
  if ((threadIdx.x % kWave) == 0) lds[wave] = v;
  __syncthreads();
  float total = lds[0];
#pragma unroll
  for (int i = 1; i < kWaves; ++i) total = fmaxf(total, lds[i]);
  __syncthreads();
  return total;
}

// Element access by a run-time type code (kF32 / kBF16 below), for operands whose type follows the checkpoint
// or the engine's mode and whose kernels are bound by memory: the branch is the same in every lane.
__device__ __forceinline__ float load_as_float(const void* p, int code, int64_t i) {
  return code == 0 ? static_cast<const float*>(p)[i] : to_float(static_cast<const bf16*>(p)[i]);
}
__device__ __forceinline__ void store_from_float(void* p, int code, int64_t i, float v) {
  if (code == 0) {
    static_cast<float*>(p)[i] = v;
  } else {
    static_cast<bf16*>(p)[i] = from_float<bf16>(v);
  }
}

// Four consecutive elements as floats, by one 16-byte (float) or 8-byte (bfloat16) access; the address is aligned
// to that size.
template <typename T>
__device__ __forceinline__ float4 ld4(const T* p);
template <>
__device__ __forceinline__ float4 ld4<float>(const float* p) {
  return *reinterpret_cast<const float4*>(p);
}
template <>
__device__ __forceinline__ float4 ld4<bf16>(const bf16* p) {
  const uint2 raw = *reinterpret_cast<const uint2*>(p);
  return float4{__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u), __uint_as_float(raw.y << 16),
                __uint_as_float(raw.y & 0xffff0000u)};
}
template <typename T>
__device__ __forceinline__ void st4(T* p, float4 v);
template <>
__device__ __forceinline__ void st4<float>(float* p, float4 v) {
  *reinterpret_cast<float4*>(p) = v;
}
template <>
__device__ __forceinline__ void st4<bf16>(bf16* p, float4 v) {
  uint2 raw;
  raw.x = pack_bf16x2(v.x, v.y);
  raw.y = pack_bf16x2(v.z, v.w);
  *reinterpret_cast<uint2*>(p) = raw;
}

// The activation of a gated feed-forward's gate, by a code shared with the Python side (the same in every lane).
constexpr int kActSilu = 0;
constexpr int kActGeluTanh = 1;   // 0.5 z (1 + tanh(sqrt(2/pi) (z + 0.044715 z^3)))
constexpr int kActSigmoid = 2;    // 1 / (1 + exp(-z)): a gate that is not multiplied by its own input
__device__ __forceinline__ float gate_act(float z, int act) {
  if (act == kActSigmoid) return 1.0f / (1.0f + expf(-z));
  if (act == kActGeluTanh) return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
  return z / (1.0f + expf(-z));
}

// Dynamic LDS beyond what a launch gets unasked has to be asked for, for every kernel and on every GPU: the attribute is the current
// device's.  Returns a hipError_t, and leaves none behind for the next call to find.
inline int ask_lds(OnceADevice& asked, size_t bytes, std::initializer_list<const void*> kernels) {
  int device = -1;
  hipError_t e = hipGetDevice(&device);
  if (e == hipSuccess && asked.done(device)) return 0;
  for (const void* kernel : kernels)
    if (e == hipSuccess) e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return static_cast<int>(e);
  }
  asked.mark(device);
  return 0;
}

inline int launch_status() { return static_cast<int>(hipGetLastError()); }

// Element type codes shared with the Python side.
constexpr int kF32 = 0;
constexpr int kBF16 = 1;

}  // namespace arle
