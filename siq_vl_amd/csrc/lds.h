// Direct global->LDS loads, and the waits and barriers that order them, shared
// by the GEMM core and the attention kernels.
#pragma once
#include "common.h"

namespace siq {

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;

// One wave instruction of direct global->LDS loading from a uniform base and
// this lane's byte offset: lane l's 16 bytes land at LDS byte lds + 16 l.
// Written as inline asm so that the compiler's wait insertion does not track
// it: it cannot tell the buffer being read from the one being loaded (both live
// in one LDS array) and would wait for the prefetch before the first transposed
// read of every step.  The caller orders the loads with the LDS reads itself (a
// vmcnt wait, then a barrier).  The LDS address goes in m0 (one wait state after
// its write) and the uniform base in SGPRs, which the compiler may have just
// written from a VALU instruction (v_readfirstlane; an SGPR written by VALU and
// read by VMEM needs five wait states): its hazard checks do not look inside
// the asm, so it starts with s_nop 4.
__device__ __forceinline__ void dma16(const bf16* gbase, uint32_t byte_off, const bf16* lds) {
  const uint32_t la = (uint32_t)(uintptr_t)(lds_void*)lds;
  asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(byte_off), "s"(gbase), "{m0}"(la) : "memory");
}

// One dword per lane from gptr (lane l's 4 bytes land at LDS byte lds + 4 l),
// untracked like dma16.  s_nop 0: m0 needs one wait state after its write; the
// address is a VGPR pair.
__device__ __forceinline__ void dma4_untracked(const void* gptr, const void* lds) {
  const uint32_t la = (uint32_t)(uintptr_t)(lds_void*)lds;
  asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(gptr), "{m0}"(la) : "memory");
}

// Wait for this wave's outstanding global (and direct-to-LDS) loads.
__device__ __forceinline__ void wait_vmem() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// Wait for this wave's outstanding LDS reads (lgkmcnt(0), vmcnt untouched).
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xC07F); }

// Wait until at most N of this wave's global loads are outstanding (loads
// complete in issue order, so everything but the newest N has landed).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | (0x7 << 4) | (0xF << 8) | ((N >> 4) << 14));
}

// A workgroup barrier that waits for no memory: the compiler neither moves
// code across it nor drains the load queue at it.
__device__ __forceinline__ void phase_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}

}  // namespace siq
