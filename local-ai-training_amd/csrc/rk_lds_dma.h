// gfx950 LDS-DMA loads (buffer_load ... lds) and the waits that go with them, shared by the
// kernels that stage tiles this way (the persistent int8 GEMM, the attention backward).
#pragma once

#include "rk_common.h"

namespace rk {

typedef __attribute__((address_space(3))) void* lds_void_ptr;

__host__ __device__ constexpr int vmcnt_imm(int n) {
  // s_waitcnt immediate that waits for vmcnt <= n only (expcnt 7, lgkmcnt 15)
  return 0x0F70 | (n & 15) | ((n >> 4) << 14);
}

// The byte address of a __shared__ object in LDS, as the DMA's M0 takes it.
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void_ptr)(void*)p));
}

// One LDS-DMA load: 16 bytes per lane at buffer offset voff + soff into LDS bytes
// lds + 16 lane .. + 15. M0 holds the LDS address (wave-uniform).
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, uint32_t lds, int voff, int soff) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(lds), "v"(voff), "s"(r), "s"(soff) : "memory", "m0");
}

// The same with 4 bytes per lane: LDS bytes lds + 4 lane .. + 3.
__device__ __forceinline__ void dma4(__amdgpu_buffer_rsrc_t r, uint32_t lds, int voff, int soff) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dword %1, %2, %3 offen lds"
               :: "s"(lds), "v"(voff), "s"(r), "s"(soff) : "memory", "m0");
}

// Waits until at most `ahead` of this wavefront's loads are in flight and its LDS counter is
// zero (the LDS write of an LDS-DMA load is tracked there; with vmcnt alone a wavefront on a
// busy CU was measured reading stale bytes), then meets the workgroup's other wavefronts.
template <int AHEAD>
__device__ __forceinline__ void dma_wait_barrier() {
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(AHEAD) & ~0x0F00);
  asm volatile("s_barrier" ::: "memory");
}

}  // namespace rk
