// Global memory to LDS without registers in between, and the waits that order it (prefill GEMMs, gated delta rule).
#pragma once
#include "../common.h"

namespace aios {

__device__ __forceinline__ void pf_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
template <int N>
__device__ __forceinline__ void pf_vmcnt() {
  static_assert(N >= 0 && N <= 63, "vmcnt immediate");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// LDS-DMA through inline asm: hipcc's waitcnt pass then does not see the DMA, so it no longer puts
// an `s_waitcnt vmcnt(0)` in front of the first ds_read after every issue (it cannot prove the read
// misses the DMA's target slot -- measured: that drain serialised every K-step).  The counted
// pf_vmcnt waits are the only ordering these loads need.  M0 is set and restored inside the
// statement.
__device__ __forceinline__ uint32_t pf_lds_addr(const uint8_t* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)p;
}
__device__ __forceinline__ void pf_glds16(const void* src, uint32_t lds) {
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
               : "=&s"(keep)
               : "v"(src), "s"(lds)
               : "memory");
}
__device__ __forceinline__ void pf_glds4(const void* src, uint32_t lds) {
  uint32_t keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %1, off\n\ts_mov_b32 m0, %0"
               : "=&s"(keep)
               : "v"(src), "s"(lds)
               : "memory");
}

// ... from a uniform base and a 32-bit byte offset per lane: no 64-bit addition per lane and request.  A scalar register
// that the vector unit wrote (v_readlane, where the base comes back from a spilled lane) is an address five wait states
// later at the earliest; the compiler guards its own loads, but not one inside an asm.  The scalar unit waits for it by
// itself, so the base goes through s_mov, in the place of the s_nop that M0 needs (s_nop 2 cost 1 to 2 %).
__device__ __forceinline__ void pf_glds16(const void* base, uint32_t off, uint32_t lds) {
  uint32_t keep;
  uint64_t from;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %4\n\ts_mov_b64 %1, %3\n\tglobal_load_lds_dwordx4 %2, %1\n\ts_mov_b32 m0, %0"
               : "=&s"(keep), "=&s"(from)
               : "v"(off), "s"(base), "s"(lds)
               : "memory");
}
__device__ __forceinline__ void pf_glds4(const void* base, uint32_t off, uint32_t lds) {
  uint32_t keep;
  uint64_t from;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %4\n\ts_mov_b64 %1, %3\n\tglobal_load_lds_dword %2, %1\n\ts_mov_b32 m0, %0"
               : "=&s"(keep), "=&s"(from)
               : "v"(off), "s"(base), "s"(lds)
               : "memory");
}

// ... both uniform operands through v_readfirstlane, for a request inside a branch that not all lanes take (the compiler
// puts uniform values into vector registers there); s_nop: a scalar register written by the vector unit is read as
// an address five cycles later at the earliest
template <int LANES, int BYTES>
__device__ __forceinline__ void pf_glds_part(const void* base, uint32_t off, uint32_t lds) {
  const uint64_t b = (uint64_t)base;
  const uint64_t u = ((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b);
  const uint32_t to = __builtin_amdgcn_readfirstlane(lds);
  if ((threadIdx.x & 63) < LANES) {
    uint32_t keep;
    if constexpr (BYTES == 16)
      asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                   : "=&s"(keep) : "v"(off), "s"(u), "s"(to) : "memory");
    else
      asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 4\n\tglobal_load_lds_dword %1, %2\n\ts_mov_b32 m0, %0"
                   : "=&s"(keep) : "v"(off), "s"(u), "s"(to) : "memory");
  }
}

}  // namespace aios
