// Direct loads from memory to LDS and the waits that order them.
#pragma once
#include "common.h"

namespace dtree {

// Direct load of 16 bytes per lane into LDS (lane l's land at lds + 16 l).
// Offsets past the resource's size read zero without a memory access. Not the
// builtin: the compiler would order every later LDS read behind all such
// loads; the stage waits below do it by count. The load has no register
// result, and the callers wait for it before its LDS is read or released.
// s_nop 4 covers m0 and a resource word that a VALU lane read has just written.
// m0 is named as clobbered, so that a value the compiler puts there is made again
// after the block; its warning about reserved registers means that the block
// does not preserve it, which is what is said here.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ int uni(uint32_t v) { return __builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ void lds_load16(u32x4_t r, unsigned off, unsigned lds_addr) {
  typedef int s32x4_t __attribute__((ext_vector_type(4)));
  const s32x4_t rsrc = s32x4_t{uni(r[0]), uni(r[1]), uni(r[2]), uni(r[3])};
  const int lds = uni(lds_addr);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :: "s"(lds), "v"(off), "s"(rsrc) : "m0", "memory");
}

// The same for a resource and an LDS address that are in scalar registers.
__device__ __forceinline__ void lds_load16_s(uint32_t base_lo, uint32_t base_hi, uint32_t size, unsigned off,
                                             uint32_t lds_addr) {
  typedef uint32_t s32x4_t __attribute__((ext_vector_type(4)));
  const s32x4_t rsrc = s32x4_t{base_lo, base_hi, size, 0x00020000u};
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :: "s"(lds_addr), "v"(off), "s"(rsrc) : "m0", "memory");
}

#pragma clang diagnostic pop

// This wave's loads but the N youngest have landed and its LDS reads are done;
// then the workgroup barrier.
template <int N>
__device__ __forceinline__ void stage_wait() {
  static_assert(N >= 0 && N <= 63, "vmcnt is 6 bits");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory");
}

__device__ __forceinline__ u32x4_t strip_rsrc(const void* p, unsigned bytes) {
  const uint64_t a = (uint64_t)p;
  return u32x4_t{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32) & 0xffff),
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}

}  // namespace dtree
