// What a ring of stages in LDS is made of: loads that the memory writes into LDS by itself, the waits for them, and a
// barrier that leaves them in flight.  The kernels that use it: gemm_ring.h (which says how the steps interlock), experts.hip.
#pragma once

#include "common.h"

namespace ls {

typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;

// A buffer descriptor over `bytes` bytes from `p`: loads at offsets from there on return zeros.
__device__ __forceinline__ u32x4_t buffer_of(const void* p, long bytes) {
  const unsigned long a = reinterpret_cast<unsigned long>(p);
  u32x4_t r;
  r[0] = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(a));
  r[1] = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(a >> 32) & 0xffffu);
  r[2] = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(bytes > 0xffffffffL ? 0xffffffffL : bytes));
  r[3] = 0x00020000u;
  return r;
}

// (Naming m0 keeps the compiler from relying on a value of its own there; that it warns of the name is all the diagnostic says.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// Sixteen bytes a lane from buffer + lane_off + off straight into LDS: the wave's 64 pieces land at lds_base + 16 *
// lane.  The instruction itself, because the compiler would wait for the compiler's own form of it in front of every
// later LDS read.  The whole offset goes through the vector register: the buffer's bound counts that one for certain.
__device__ __forceinline__ void buffer_to_lds16(unsigned lane_off, unsigned off, u32x4_t buffer, unsigned lds_base) {
  unsigned at;
  __asm__ volatile("v_add_u32 %0, %2, %1\n\ts_mov_b32 m0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %3, 0 offen lds"
                   : "=&v"(at)
                   : "v"(lane_off), "s"(off), "s"(buffer), "s"(lds_base)
                   : "memory", "m0");
}
#pragma clang diagnostic pop

template <int YOUNGER>  // loads issued after those that are waited for
__device__ __forceinline__ void wait_loads() {
  static_assert(YOUNGER >= 0 && YOUNGER <= 63, "the count of a wait has six bits");
  __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNGER) : "memory");
}

// A barrier behind the waves' own LDS reads and writes; loads into LDS stay in flight (wait_loads waits for those).
__device__ __forceinline__ void ring_barrier() { __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

}  // namespace ls
