// Global memory straight into LDS, 16 bytes a lane, outside the compiler's
// wait-count tracking.
//
// The compiler's LDS-destination load builtin makes it wait for every such
// load in flight (s_waitcnt vmcnt(0)) before the next LDS read it cannot tell
// apart from the load's target, so a tile requested ahead was waited for at
// the first fragment read of the tile before it. Here the load is an asm
// statement: the kernel waits itself (s_waitcnt vmcnt, then a barrier) before
// a stage is read, and the loads stay in flight until then. The statement has
// no register output; its "memory" clobber keeps LDS reads on their side of
// it.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace pjrtx {

typedef unsigned int lds_rsrc __attribute__((ext_vector_type(4)));

// A raw buffer resource over `bytes` at `base` (loads past it read as zero).
// The arguments are the same on every lane.
__device__ __forceinline__ lds_rsrc make_lds_rsrc(const void* base, uint32_t bytes) {
  const uint64_t b = reinterpret_cast<uint64_t>(base);
  return lds_rsrc{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b),
                  (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(b >> 32) & 0xffffu)),
                  (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}

// Byte offset of an LDS address in the workgroup's allocation.
template <typename T>
__device__ __forceinline__ uint32_t lds_offset(T* p) {
  return (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) T*)p);
}

// Lane L's 16 bytes from resource offset voff (its range check covers it)
// plus soff go to LDS bytes lds + 16 L. The write of m0 needs one wait state
// before the load reads it; m0 is the compiler's to reserve and cannot be
// listed as clobbered, and it writes m0 itself right before its own uses (which
// kernels without LDS-load builtins and register-indexed moves do not have).
__device__ __forceinline__ void lds_dma16(const lds_rsrc& r, uint32_t voff, uint32_t soff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(lds), "v"(voff), "s"(r), "s"(soff)
               : "memory");
}

}  // namespace pjrtx
