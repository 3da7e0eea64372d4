// LDS copies issued from inline asm (gfx950): global_load_lds rows that the
// compiler neither orders against its own LDS reads nor waits on. The caller
// waits for them (wait_copies) before the barrier that publishes the data,
// and never reads a buffer that a copy in flight may still write.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gemma4 {

// LDS byte address of a __shared__ object (for M0).
__device__ __forceinline__ uint32_t lds_address(const void *ptr) {
  return (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const char *)ptr);
}

// One 1 KiB LDS copy (global_load_lds, 16 bytes per lane): LDS bytes
// [lds_addr, +1024) from the per-lane addresses src. The copy is invisible
// to the compiler's memory counters: the caller waits for it (vmcnt) before
// the barrier that publishes the tile.
__device__ __forceinline__ void copy_row_pair(uint64_t src, uint32_t lds_addr) {
  uint32_t m0_saved;
  asm volatile(
      "s_mov_b32 %[m0s], m0\n\t"
      "s_mov_b32 m0, %[lds]\n\t"
      "s_nop 0\n\t"  // SALU write of M0 -> LDS DMA reading it: one wait state (gfx9)
      "global_load_lds_dwordx4 %[src], off\n\t"
      "s_mov_b32 m0, %[m0s]"
      : [m0s] "=&s"(m0_saved)
      : [lds] "s"(lds_addr), [src] "v"(src));
}

// One 4-byte-per-lane LDS copy: LDS bytes [lds_addr, +256) from the
// per-lane addresses src (global_load_lds_dword); waited for like
// copy_row_pair.
__device__ __forceinline__ void copy_dwords(const void *src, uint32_t lds_addr) {
  uint32_t m0_saved;
  asm volatile(
      "s_mov_b32 %[m0s], m0\n\t"
      "s_mov_b32 m0, %[lds]\n\t"
      "s_nop 0\n\t"  // SALU write of M0 -> LDS DMA reading it: one wait state (gfx9)
      "global_load_lds_dword %[src], off\n\t"
      "s_mov_b32 m0, %[m0s]"
      : [m0s] "=&s"(m0_saved)
      : [lds] "s"(lds_addr), [src] "v"(src));
}

// Two 1 KiB copies into consecutive LDS rows: 16 bytes per lane from
// base0 + off0, then base1 + off1. The bases must not come straight from a vector
// instruction (v_readlane: five wait states before a memory instruction reads
// the SGPR, which the compiler does not see for inline asm).
__device__ __forceinline__ void copy_lanes2(uint64_t base0, uint32_t off0, uint64_t base1,
                                            uint32_t off1, uint32_t lds_addr) {
  uint32_t m0_saved;
  asm volatile(
      "s_mov_b32 %[m0s], m0\n\t"
      "s_mov_b32 m0, %[lds]\n\t"
      "s_nop 0\n\t"  // SALU write of M0 -> LDS DMA reading it: one wait state (gfx9)
      "global_load_lds_dwordx4 %[o0], %[b0]\n\t"
      "s_add_u32 m0, m0, 1024\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %[o1], %[b1]\n\t"
      "s_mov_b32 m0, %[m0s]"
      : [m0s] "=&s"(m0_saved)
      : [lds] "s"(lds_addr), [b0] "s"(base0), [b1] "s"(base1), [o0] "v"(off0), [o1] "v"(off1)
      : "memory", "scc");
}

// Waits until at most n vector memory operations of this wave are
// outstanding, the copies included.
template <int n>
__device__ __forceinline__ void wait_vector() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(n) : "memory");
}
// Waits for this wave's LDS reads: a copy issued next may overwrite what
// they read.
__device__ __forceinline__ void wait_lds_reads() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// Workgroup barrier that orders LDS traffic only: the copies in flight stay
// in flight (__syncthreads may wait for them).
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Waits for every vector memory operation of this wave, the copies
// included (s_waitcnt vmcnt(0); a builtin rather than inline asm so the
// compiler's own counter bookkeeping sees it as well).
__device__ __forceinline__ void wait_copies() {
  constexpr int kVmcnt0 = 0x0F70;  // gfx9 encoding: vmcnt 0, expcnt 7, lgkmcnt 15 (no wait)
  __builtin_amdgcn_s_waitcnt(kVmcnt0);
}

}  // namespace gemma4
