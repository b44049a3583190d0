// Loads from memory straight into LDS that the compiler does not count.
#pragma once
#include "common.h"

namespace arle {

// Sixteen bytes a lane from memory straight into LDS: the wave's 64 pieces land one after the other from
// lds_base on, which has to be the same in all lanes.  Written as assembly, and not with the compiler's builtin,
// because of what the builtin does to every later wait: while such a load is in flight the compiler takes LDS
// reads to finish in any order and turns each wait for one of them into a wait for all of them, so that no read
// can stay in flight behind a matrix product.  The loads it does not know of only make its own waits for memory
// stricter than needed; that the data has landed before it is read is the caller's business (s_waitcnt vmcnt(0)
// and a barrier).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 is a reserved register: naming it as clobbered is the point
__device__ __forceinline__ void load_to_lds_16(const void* src, unsigned char* lds_at) {
  const uint32_t base = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)lds_at)));
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(base), "v"(src) : "memory", "m0");
}
// The same with the address as a wave-wide base and a byte offset of the lane.
__device__ __forceinline__ void load_to_lds_16(const void* base_uniform, uint32_t lane_bytes, unsigned char* lds_at) {
  const uint32_t base = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)lds_at)));
  const uint64_t src = reinterpret_cast<uint64_t>(base_uniform);
  // the builtin returns a signed int: widened as it is, a low half with its top bit set would fill the high half
  const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(src))));
  const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(src >> 32)));
  const uint64_t src_s = (static_cast<uint64_t>(hi) << 32) | lo;
  // s_nop 4: a scalar register written by a vector instruction may not be a memory instruction's address for
  // five cycles, and the compiler does not look into this text for that
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(base), "v"(lane_bytes), "s"(src_s)
               : "memory", "m0");
}
#pragma clang diagnostic pop

}  // namespace arle
