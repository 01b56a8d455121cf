// Loads from global memory straight into LDS, and the waits and barriers that go with them: what the
// stage rings of the GEMM kernels (ns_gemm_big.hip, ns_gemm_tile.hip) are built from.
#pragma once
#include "common.h"

// vmcnt(n): wait until at most n vector-memory operations of this wavefront are outstanding
// (they complete in issue order), leaving lgkmcnt/expcnt alone.
template <int N> __device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// One LDS-DMA instruction: lane l of the wavefront copies 16 bytes from g (per lane) to LDS byte
// address lds_base + 16*l (lds_base wavefront-uniform, carried in M0). Written as inline
// assembly so that the stage ring's explicit vmcnt waits are the only ones: the compiler's own
// wait insertion is conservative about LDS-DMA writes that it cannot prove distinct from later
// LDS reads and would drain the ring on every tile.
__device__ __forceinline__ void dma16(const void *g, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_base), "v"(g)
               : "memory", "m0");
}
// The same for bytes that nobody reads again: the first to leave the caches.
__device__ __forceinline__ void dma16_once(const void *g, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(lds_base), "v"(g)
               : "memory", "m0");
}
// The same as the first from a wavefront-uniform address and 32-bit offsets per lane: no 64-bit addition in vector registers. The
// address is copied by a scalar instruction, which is the wait state that the write of M0 needs and makes it safe to
// use at once even where a vector instruction (v_readfirstlane) has just produced it.
__device__ __forceinline__ void dma16(const void *g, uint32_t off, uint32_t lds_base) {
  uint64_t base;
  asm volatile("s_mov_b32 m0, %1\n\ts_mov_b64 %0, %3\n\tglobal_load_lds_dwordx4 %2, %0"
               : "=&s"(base) : "s"(lds_base), "v"(off), "s"(g) : "memory", "m0");
}
__device__ __forceinline__ uint32_t lds_addr(const void *p) {
  return (uint32_t)(uintptr_t)((__attribute__((address_space(3))) const void *)p);
}

// Workgroup barrier that orders LDS traffic only: this wavefront's LDS reads and writes have
// completed (lgkmcnt 0) before it arrives. Unlike __syncthreads() it carries no fence over
// global memory, so LDS-DMA loads of younger stages stay in flight across it; the caller waits
// (wait_vm<N>) for the DMA it needs before calling this.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// The same inside one wavefront: its LDS writes have landed, nothing moves across.
__device__ __forceinline__ void lds_wave_sync() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_wave_barrier();
  asm volatile("" ::: "memory");
}
