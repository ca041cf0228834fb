// Global -> LDS DMA helpers shared by the MFMA GEMMs (gfx950).
//
// The DMA loads are issued from inline asm with the LDS base in M0 and are
// waited for with explicit s_waitcnt counts: the compiler treats LDS DMA as
// aliasing every LDS read and would otherwise wait for all of them (including
// the stage just issued) before each fragment read.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cellm {
namespace ldsdma {

constexpr size_t kMaxLds = 160 * 1024;

__device__ __forceinline__ uint32_t lds_addr(const void* p)
{
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

// 16 bytes per lane, global -> LDS; lane i lands at lds + 16 i (checked on gfx950).  A uniform 64-bit
// base in SGPRs and a per-lane 32-bit byte offset: a loop that only changes the base never rewrites the
// VGPR operand (the compiler's wait pass treats an asm's VGPR operands as pending after it, and
// rewriting them cost a vmcnt(0) drain per iteration).
__device__ __forceinline__ void dma16_s(uint32_t voff, const void* sbase, uint32_t lds)
{
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase),
                 "s"(__builtin_amdgcn_readfirstlane(lds))
                 : "memory", "m0");
}

// 4 bytes per lane; lane i lands at lds + 4 i
__device__ __forceinline__ void dma4_s(uint32_t voff, const void* sbase, uint32_t lds)
{
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(sbase),
                 "s"(__builtin_amdgcn_readfirstlane(lds))
                 : "memory", "m0");
}

// 2 bytes per lane, zero-extended; lane i lands at lds + 4 i
__device__ __forceinline__ void dma2_s(uint32_t voff, const void* sbase, uint32_t lds)
{
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_ushort %0, %1" ::"v"(voff), "s"(sbase),
                 "s"(__builtin_amdgcn_readfirstlane(lds))
                 : "memory", "m0");
}

template <int N>
__device__ __forceinline__ void wait_vmcnt()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

}  // namespace ldsdma
}  // namespace cellm
