/* kt_dma.h - global to LDS copies without registers (buffer_load ... lds), as asm: the compiler would wait for all of
   them before any LDS read, so the kernels that use them count a wave's vector memory instructions by hand
   (s_waitcnt vmcnt(n): loads retire in order). */
#pragma once
#include "kt_common.h"

typedef int kt_dma_v4i __attribute__((ext_vector_type(4)));
#define KT_L3 __attribute__((address_space(3)))

/* a buffer resource as the 4 dwords the asm takes: base, stride 0, num_records bytes, gfx950 default flags */
__device__ __forceinline__ kt_dma_v4i kt_dma_rsrc(const void* p, uint32_t bytes){
  const unsigned long long a = (unsigned long long)p;
  kt_dma_v4i r;
  r.x = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
  r.y = __builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32) & 0xFFFF);
  r.z = (int)bytes;
  r.w = 0x00020000;
  return r;
}
/* lane i's 16 (4) bytes at byte voff + soff of the buffer land at LDS byte address lds + 16 i (4 i); soff and lds
   wave-uniform. voff alone past the buffer lands zeros: soff is not part of the range check */
__device__ __forceinline__ void kt_dma16(kt_dma_v4i rs, uint32_t voff, uint32_t soff, uint32_t lds){
  const uint32_t l = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds);
  const uint32_t o = (uint32_t)__builtin_amdgcn_readfirstlane((int)soff);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(l), "v"(voff), "s"(rs), "s"(o) : "memory", "m0");
}
__device__ __forceinline__ void kt_dma4(kt_dma_v4i rs, uint32_t voff, uint32_t soff, uint32_t lds){
  const uint32_t l = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds);
  const uint32_t o = (uint32_t)__builtin_amdgcn_readfirstlane((int)soff);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
               :: "s"(l), "v"(voff), "s"(rs), "s"(o) : "memory", "m0");
}
__device__ __forceinline__ uint32_t kt_dma_lds(const void* p){
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)(const KT_L3 void*)p);
}
