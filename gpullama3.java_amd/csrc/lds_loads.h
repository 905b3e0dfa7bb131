// Loads from memory straight into shared memory, and the waits and barriers of kernels whose two groups of waves take turns:
// shared by the tiled products (gemm_mfma.hip) and prefill attention (attention_prefill.hip).
#pragma once
#include "common.h"

typedef int i32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void mf_dma16(unsigned lds, unsigned offset, i32x4 rsrc, unsigned step_offset) {
  // (by hand: behind the builtin the compiler waits for every load in front of every read of shared memory. The
  // instruction has no destination register; its data lands at m0 + 16 * lane. m0 is an operand that the compiler sets, so that it
  // knows what the register holds. A memory instruction may read a scalar register only five wait states after a vector
  // instruction wrote it, and the compiler does not look into this block to keep them: 10 of the 806 loads it placed had
  // readfirstlane of the step's offset three states ahead. A scalar instruction's result may be read at once, so the offset is copied by
  // one; it is also the instruction that has to stand between m0's setting and the load. Five states of waiting instead: 1% of
  // 8,192 tokens of the 8B layers.)
  unsigned s;
  asm volatile("s_mov_b32 %0, %4\n\tbuffer_load_dwordx4 %2, %3, %0 offen lds" : "=&s"(s) : "{m0}"(__builtin_amdgcn_readfirstlane(lds)), "v"(offset), "s"(rsrc), "s"(__builtin_amdgcn_readfirstlane(step_offset))
               : "memory");
}
template <int N>
__device__ __forceinline__ void mf_wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
template <int N>
__device__ __forceinline__ void mf_wait_reads() {
  asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void mf_barrier() {      // no wait of its own, and nothing moves across it
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ i32x4 mf_rsrc(const void* p) {
  const unsigned long a = (unsigned long)p;
  int lo, hi;      // (through scalar instructions, as above)
  asm("s_mov_b32 %0, %1" : "=s"(lo) : "s"(__builtin_amdgcn_readfirstlane((int)a)));
  asm("s_mov_b32 %0, %1" : "=s"(hi) : "s"(__builtin_amdgcn_readfirstlane((int)(a >> 32))));
  return i32x4{lo, hi, 0x7fffffff, 0x00020000};
}
