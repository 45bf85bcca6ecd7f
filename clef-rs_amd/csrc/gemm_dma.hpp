// Device helpers of the f16 GEMMs' LDS rings: global -> LDS DMA from buffer
// resources and the waits for it.
#pragma once
#include <utility>

#include "common.hpp"

namespace clef {

// buffer_load_dwordx4 ... lds written as inline asm: the compiler does not
// see an LDS write it would have to order before every later LDS read (it
// would wait for all DMAs in flight, i.e. for the next stage, before
// computing on the current one).  Completion is awaited explicitly (vmcnt)
// before the barrier that publishes a stage.  The source is a buffer resource
// (SGPR base and size) plus a 32-bit lane byte offset; the LDS destination
// goes in M0 (low 32 bits of the LDS address), lane l writing 16 bytes at
// M0 + 16 l.  The asm carries the one wait state an LDS DMA needs after the
// SALU write of M0.  (1-6% faster than global_load_lds_dwordx4 with 64-bit
// lane addresses on the projection shapes, bit-identical.)
__device__ __forceinline__ void bdma16(__amdgpu_buffer_rsrc_t r, uint32_t off, void* lds_block) {
  const uint32_t m0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds_block));
  asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off), "s"(r), "{m0}"(m0) : "memory");
}
// the same with a wave-uniform byte offset added to every lane's
__device__ __forceinline__ void bdma16(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t uniform_off, void* lds_block) {
  const uint32_t m0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds_block));
  asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, %3 offen lds" ::"v"(off), "s"(r), "{m0}"(m0), "s"(uniform_off)
               : "memory");
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t operand_rsrc(const half_t* base, int64_t rows, int64_t ld) {
  // rows * ld * 2 < 2^32 (checked by gemm_f16_dma_ok)
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(base), 0, static_cast<int>(static_cast<uint32_t>(rows * ld * 2)),
                                           0x00020000);
}

__device__ __forceinline__ void vm_wait_all() { __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8)); }
template <int N>
__device__ __forceinline__ void vm_wait() {  // s_waitcnt vmcnt(N)
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
// vmcnt(n) for an n that is a constant once loops are unrolled
template <int... Ns>
__device__ __forceinline__ void vm_wait_n(int n, std::integer_sequence<int, Ns...>) {
  ((n == Ns ? (vm_wait<Ns>(), 0) : 0), ...);
}
__device__ __forceinline__ void vm_wait_n(int n) { vm_wait_n(n, std::make_integer_sequence<int, 40>{}); }

}  // namespace clef
