// What stages and tiles in LDS are made of: loads that the memory writes into LDS by itself, the waits for them, and a
// barrier that leaves them in flight.  The kernels that use it: gemm_ring.h (which says how the steps interlock), experts.hip,
// attention.hip, sink_attention.hip.
#pragma once

#include "common.h"

namespace ls {

typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;

// The offset of a load that is to read nothing, and the most bytes a descriptor is given: an operand that goes on for 4 GiB and
// more ends there for the hardware too, and neither this offset nor its sixteen bytes come round to the operand's start.
constexpr unsigned kNothing = 0xfffffff0u;

// A buffer descriptor over `bytes` bytes from `p` (kNothing of them at most): loads at offsets from there on return zeros.
__device__ __forceinline__ u32x4_t buffer_of(const void* p, long bytes) {
  const unsigned long a = reinterpret_cast<unsigned long>(p);
  u32x4_t r;
  r[0] = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(a));
  r[1] = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(a >> 32) & 0xffffu);
  r[2] = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(bytes > (long)kNothing ? (long)kNothing : bytes));
  r[3] = 0x00020000u;
  return r;
}

// (Naming m0 keeps the compiler from relying on a value of its own there; that it warns of the name is all the diagnostic says.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// Sixteen bytes a lane from buffer + at straight into LDS: the wave's 64 pieces land at lds_base + 16 *
// lane.  The instruction itself, because the compiler would wait for the compiler's own form of it in front of every
// later LDS read.  The whole offset goes through the vector register: the buffer's bound counts that one for certain.
// The descriptor may come from vector instructions (v_readfirstlane): the s_mov and the s_nop are the five wait states that
// a memory instruction needs behind those (see load_to_lds16_from).
__device__ __forceinline__ void buffer_to_lds16(unsigned at, u32x4_t buffer, unsigned lds_base) {
  __asm__ volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
                   :
                   : "v"(at), "s"(buffer), "s"(lds_base)
                   : "memory", "m0");
}
// One 16-byte piece per lane from global memory straight into LDS: the wave's 64 pieces land at
// `lds_wave_base` + 16 * lane, each lane names its own source.  Written as the instruction itself
// (M0 holds the wave's LDS address): after the compiler's own form of it
// (__builtin_amdgcn_global_load_lds) every later LDS read and every barrier waits for all such
// loads in flight, because they might be reading what the loads write, and the loads of the next
// tile could not overlap the work on this one.  The kernels wait for a tile's loads themselves
// (s_waitcnt vmcnt) before the barrier after which the tile is read.
__device__ __forceinline__ void load_to_lds16(const void* src, __attribute__((address_space(3))) void* lds_wave_base) {
  const unsigned base = __builtin_amdgcn_readfirstlane((unsigned)(unsigned long)lds_wave_base);
  __asm__ volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(base) : "memory", "m0");
}
// The same with the address in two parts: a base that the wave shares, in scalar registers, and a lane's 32-bit offset.
// The base may come from a vector instruction (v_readlane) right in front of this.  A memory instruction may read such a scalar
// register five wait states later at the earliest, the hardware does not check it, and the compiler, which sees to it for loads of
// its own, does not look in here: the s_mov is one of the five, the s_nop four.
__device__ __forceinline__ void load_to_lds16_from(unsigned long long base, unsigned offset, unsigned lds_wave_base) {
  __asm__ volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(offset), "s"(base),
                   "s"(lds_wave_base)
                   : "memory", "m0");
}
#pragma clang diagnostic pop

template <int YOUNGER>  // loads issued after those that are waited for
__device__ __forceinline__ void wait_loads() {
  static_assert(YOUNGER >= 0 && YOUNGER <= 63, "the count of a wait has six bits");
  __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNGER) : "memory");
}

// A barrier behind the waves' own LDS reads and writes; loads into LDS stay in flight (wait_loads waits for those).
// (__syncthreads() would wait for them too, which would end the overlap of the next tile's loads with the work on this one.)
__device__ __forceinline__ void ring_barrier() { __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

}  // namespace ls
