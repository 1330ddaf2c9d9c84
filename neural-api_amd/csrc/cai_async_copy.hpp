// Copies from memory straight into LDS (64 lanes x 16, 4 or 2 bytes), in lane order from the uniform byte address lds on; two bytes take a dword
// each.  A lane's source is an address of its own or a 32-bit byte offset from a uniform base.  No registers are written and the compiler does
// not see the load: vmcnt counts it, and the caller waits for it before the barrier that publishes the tile and before the kernel's LDS could go
// to another work-group.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cai {

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"     // (m0 is reserved, and named all the same: the statement changes it)
__device__ __forceinline__ void copy16_to_lds(uint32_t lds, const void* from)
{
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" :: "s"(lds), "v"(from) : "memory", "m0");
}
__device__ __forceinline__ void copy16_to_lds(uint32_t lds, uint32_t voff, const void* base)
{
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(lds), "v"(voff), "s"(base) : "memory", "m0");
}
// of what is read once: not kept in the caches
__device__ __forceinline__ void copy16_to_lds_once(uint32_t lds, uint32_t voff, const void* base)
{
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" :: "s"(lds), "v"(voff), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void copy4_to_lds(uint32_t lds, uint32_t voff, const void* base)
{
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" :: "s"(lds), "v"(voff), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void copy2_to_lds(uint32_t lds, uint32_t voff, const void* base)
{
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_ushort %1, %2" :: "s"(lds), "v"(voff), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop

// until at most N of the wave's copies and loads are on their way
template <int N> __device__ __forceinline__ void wait_copies()
{
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
  asm volatile("" ::: "memory");
}

}  // namespace cai
