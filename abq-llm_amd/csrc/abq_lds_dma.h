// Loads from global memory straight into LDS (global_load_lds): lane l of the wave lands at lds_addr + its size * l.  Issued
// from inline assembly because the kernels count their own loads in flight; the only place that writes M0.
//
// A scalar write of M0 needs one wait state before a load that reads it as its LDS address (S_MOV M0 followed by a global
// load with LDS = 1).  The compiler's hazard pass does not look into an assembly string, so the s_nop stands in each of
// them: without it a load may still see the M0 of the one before and land in that one's place.  (M0 cannot be named as
// clobbered: the compiler reserves it and sets it up itself right before each of its own uses; it keeps no value there
// across other instructions.)
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace abq {

// 16 bytes per lane from src (per lane)
__device__ __forceinline__ void lds_dma16(const void *src, unsigned lds_addr)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(src)
                 : "memory");
}

// 16 bytes per lane from base + off: `base` the same in every lane (a scalar register pair), `off` the lane's byte offset
__device__ __forceinline__ void lds_dma16(const void *base, uint32_t off, unsigned lds_addr)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(off),
                 "s"(base)
                 : "memory");
}

// four bytes per lane from base + off
__device__ __forceinline__ void lds_dma4(const void *base, uint32_t off, unsigned lds_addr)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(off),
                 "s"(base)
                 : "memory");
}

} // namespace abq
