// Rows of an operand in pieces of 16 bytes, for the kernels that take one straight into registers.
#pragma once
#include "common.h"

namespace ls {

// The same piece of 16 bytes for the kernels of few rows.  WHOLE (rows and k on 16 bytes, offsets within a block of rows in 31
// bits): one buffer load whatever the lane, a lane with nothing to load asking past the buffer's end, which reads as zero
// without going to memory.  load_vec (common.h) leaves a choice at every load, and the compiler makes branches of those: a load to a
// block, the element-by-element path between every two (a product of few rows 2,600 lines, now 300), and a wait behind
// branches counted by the way with the fewest loads, so that a ring of loads in flight was waited for whole.  A chunk that starts
// behind the slice is multiplied as zeros rather than jumped over: behind a jump the compiler asks for the next chunk only
// once the last one has come.  Measured (us in a decode step, load_vec / row_piece): slice sums 1 x 1,024 x 3,072 4.1 / 3.5,
// float32 8 x 1,024 x 3,072 6.5 / 5.5, 8 x 4,096 x 1,024 8.4 / 7.0, the head 8 x 151,936 x 1,024 153 / 125.
// `base`, the first of the block's rows, must be the same for the wave; !any: the block does not exist.
constexpr int kNoPiece = 0x7ffffff0;  // past every buffer's end
template <typename T, bool WHOLE>
__device__ __forceinline__ typename Atom<T>::vec_t row_piece(const T* __restrict__ base, int row, int k, int limit, long ld, bool ok,
                                                             bool aligned, bool any = true) {
  if constexpr (WHOLE) {
    const auto from = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, any ? kNoPiece : 0, 0x00020000);
    int offset = (int)ok & (int)(k < limit) ? (row * (int)ld + k) * (int)sizeof(T) : kNoPiece;
    __asm__("" : "+v"(offset));  // (a choice of offsets, not a branch to one of two loads)
    return __builtin_bit_cast(typename Atom<T>::vec_t, __builtin_amdgcn_raw_buffer_load_b128(from, offset, 0, 0));
  } else {
    if (!any) return Atom<T>::zero();  // (load_vec may read at `base` for a lane without a piece)
    return load_vec<T>(base, row, k, limit, ld, ok, aligned);
  }
}

}  // namespace ls
