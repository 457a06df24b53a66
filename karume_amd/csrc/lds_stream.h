// Loads from memory straight to LDS, and the wait for them.
#pragma once

#include "krm_internal.h"

namespace krm {
namespace {

// 16 bytes a lane from base + offset to LDS at lds + 16 * lane.
__device__ inline void stream_to_lds(uint32_t lds, uint32_t offset, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds),
               "v"(offset), "s"(base)
               : "memory");
}
// The same for a dword or a zero-extended ushort a lane, to LDS at lds + 4 * lane.
__device__ inline void stream_word_to_lds(uint32_t lds, uint32_t offset, const void* base, bool half) {
  if (half)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_ushort %1, %2" ::"s"(lds),
                 "v"(offset), "s"(base)
                 : "memory");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds),
                 "v"(offset), "s"(base)
                 : "memory");
}
template <int N>
__device__ inline void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// Everything streamed has landed, and everything this wave read from LDS has arrived: what is asked for behind it
// may land where it read.  (A read's own wait stands at its first use, which may come later.)
__device__ inline void wait_streamed_and_read() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); }

}  // namespace
}  // namespace krm
