// The tiled product of gemm.hip: BM x BN outputs a workgroup, both operands through LDS, and a ring of
// stages that the memory writes into LDS by itself (buffer loads with LDS as their target), so that a stage
// takes no register and no instruction of its own on its way; a ring of n stages has n - 1 of them in flight.
// The loop, its layout and its order are ring_product.h's.
//
// What bounds it: a workgroup's stage (128 bytes of K of all its rows, or 256) has to arrive before anyone may
// multiply it, and takes 1 to 2 us from the memory side; a CU's 160 KB of LDS hold two to five stages, so the
// larger the tile, the more multiplications stand behind a byte in flight.  Loads without any product between them bring
// 55 GB/s a CU (256 x 192 outputs) to 75 (128 x 64), 95 where L2 holds everything.  Measured (bfloat16, weights from
// HBM, us): 2,048 x 24,576 x 4,096 326 (1,265 TFLOP/s; 356 in a long run of them), 2,048 x 6,144 x 4,096 83 to 89, 2,048 x 4,096 x 12,288 172 to 177
// (1,195), 1,000 x 4,096 x 4,096 42, 97 x 4,096 x 1,024 6.4; the clock falls to 1.9 GHz under the large ones, and products alone, without a load
// or a fragment read, take 235 us where the first takes 326.  Counters of the first: matrix pipes busy 67 % of the cycles that its CU is, LDS 28 %, no
// bank conflicts.
#pragma once

#include "ring_product.h"

namespace ls {

// NWM x NWN waves.  Rows of X and W are 16-byte aligned and K is whole 16-byte pieces; what a stage reads behind K (and the
// stages behind the last one) comes from beyond the end of the buffer, as zeros.
template <typename T, int EPI, int BM, int BN, int NWM, int NWN, int WS, int XS, int SUB>
__global__ __launch_bounds__(64 * NWM * NWN) void gemm_ring_kernel(const T* __restrict__ X, const T* __restrict__ W,
                                                        void* __restrict__ C, int M, int N, int K, long ldx, long ldc,
                                                        int kslice, int vec_ok, int tiles_m, int tiles_n, int out_cols,
                                                        const float* __restrict__ act) {
  const Factors factors = load_factors<EPI>(act);
  constexpr bool SLICES = EPI == kSliceSums;
  constexpr int NW = NWM * NWN;
  constexpr int BK = SUB * 128 / sizeof(T);   // elements of K a stage
  constexpr int TI = BN / (16 * NWN);         // weight tiles (16 columns) a wave
  constexpr int TJ = BM / (16 * NWM);         // row tiles a wave
  constexpr int LW = BN / (8 * NW) * SUB, LX = BM / (8 * NW) * SUB;  // a wave's loads a stage: eight rows each
  static_assert(BN % (8 * NW) == 0 && BM % (8 * NW) == 0 && TI * 16 * NWN == BN && TJ * 16 * NWM == BM, "tile shape");
  static_assert(EPI != kSwiGLU || TI % 2 == 0 || (TI == 1 && NWN == 2), "gate and up tiles meet in a wave or in a pair of waves");
  typedef RingProduct<T, TI, TJ, 2048, BN, BM, LW, LX, WS, XS, SUB, !SLICES> Product;
  extern __shared__ __attribute__((aligned(1024))) unsigned char ring[];  // WS stages of W, then XS of X

  // Workgroup ids go round the eight XCDs: give each XCD a contiguous run of tiles, numbered in bands of
  // LS_GEMM_GROUP_M row tiles, so that the workgroups that run together on an XCD share operands in its L2.
  const int total_tiles = tiles_m * tiles_n;
  const int xcd = blockIdx.x & 7, per_xcd = total_tiles >> 3, extra = total_tiles & 7;
  const int id = xcd * per_xcd + min(xcd, extra) + (int)(blockIdx.x >> 3);
  const int band = id / (LS_GEMM_GROUP_M * tiles_n);
  const int in_band = id % (LS_GEMM_GROUP_M * tiles_n);
  const int band_rows = min(LS_GEMM_GROUP_M, tiles_m - band * LS_GEMM_GROUP_M);
  const int m_base = (band * LS_GEMM_GROUP_M + in_band % band_rows) * BM;
  const int n_base = (in_band / band_rows) * BN;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = (wave % NWN) * (BN / NWN);
  const int wm = (wave / NWN) * (BM / NWM);
  const int row16 = lane & 15;
  const int g = lane >> 4;

  // Loads: lane l of a wave's load takes row (l / 8) of eight and the piece that belongs into slot l % 8.  Rows past
  // the last read as zeros; their products land in outputs that are not stored.
  const unsigned piece = ((lane & 7) ^ (lane >> 3)) * 16;
  const unsigned w_off = (unsigned)((wave * 8 + (lane >> 3)) * (long)K * sizeof(T)) + piece;
  const unsigned x_off = (unsigned)((wave * 8 + (lane >> 3)) * ldx * sizeof(T)) + piece;
  const unsigned w_step = (unsigned)(NW * 8 * (long)K * sizeof(T)), x_step = (unsigned)(NW * 8 * ldx * sizeof(T));
  const u32x4_t w_buffer = buffer_of(W + (long)n_base * K, (long)(N - n_base) * K * sizeof(T));
  const u32x4_t x_buffer = buffer_of(X + (long)m_base * ldx, ((long)(M - m_base - 1) * ldx + K) * sizeof(T));
  const unsigned lds0 = (unsigned)(unsigned long)(__attribute__((address_space(3))) void*)ring + wave * 1024;

  // the stages of this workgroup: all of K, or (kSliceSums) those of its group of out_cols slices
  const int all_stages = (K + BK - 1) / BK;
  const int first_stage = SLICES ? (int)blockIdx.y * out_cols * (kslice / BK) : 0;
  const int stages = SLICES ? min(all_stages - first_stage, out_cols * (kslice / BK)) : all_stages;
  const int per_slice = kslice / BK;  // a stage never straddles a slice
  // bytes of a row from this lane's piece on that belong to this workgroup
  const int limit = min(K, (first_stage + stages) * BK) * (int)sizeof(T) - (int)piece;

  auto request_w = [&](int st, int buf, int n) LS_INLINED {
    const int i = n / SUB, part = n % SUB, k = ((first_stage + st) * SUB + part) * 128;
    buffer_to_lds16(k < limit ? w_off + k + i * w_step : kNothing, w_buffer,
                    lds0 + buf * Product::W_BYTES + part * BN * 128 + i * NW * 1024);
  };
  auto request_x = [&](int st, int buf, int n) LS_INLINED {
    const int i = n / SUB, part = n % SUB, k = ((first_stage + st) * SUB + part) * 128;
    buffer_to_lds16(k < limit ? x_off + k + i * x_step : kNothing, x_buffer,
                    lds0 + WS * Product::W_BYTES + buf * Product::X_BYTES + part * BM * 128 + i * NW * 1024);
  };
  Product product;
  auto store_slice = [&](int slice) LS_INLINED {  // the sums of one slice to their place among the slice sums
    if constexpr (SLICES) {
      float* sums = reinterpret_cast<float*>(C) + (long)slice * M * N;
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
          const f32x4& acc = product.acc[i][j];
          const float t[4] = {acc[0], acc[1], acc[2], acc[3]};
          epilogue4<T, kStoreF32>(sums, ldc, m_base + wm + j * 16 + row16, n_base + wn + i * 16 + g * 4, M, N, t, vec_ok);
        }
    }
  };
  product.run(ring + wn * 128, ring + WS * Product::W_BYTES + wm * 128, stages, per_slice, request_w, request_x,
              [&](int st) LS_INLINED { store_slice((first_stage + st) / per_slice - 1); });

  if constexpr (SLICES) {
    if (stages > 0) store_slice((first_stage + stages - 1) / per_slice);
  } else if constexpr (EPI == kSwiGLU) {  // weight tiles come in pairs (gate t, up t)
    auto gated = [&](const f32x4& gate, const f32x4& up, int j, int n) LS_INLINED {
      const float gs[4] = {gate[0], gate[1], gate[2], gate[3]}, us[4] = {up[0], up[1], up[2], up[3]};
      epilogue_swiglu4<T>(C, ldc, m_base + wm + j * 16 + row16, n / 2 + g * 4, M, out_cols, gs, us, vec_ok);
    };
    if constexpr (TI == 1) {  // ... of two neighbouring waves: the second one's totals go through LDS, which nobody reads any more
      f32x4* const ups = reinterpret_cast<f32x4*>(ring) + (wave / NWN) * TJ * 64 + lane;
      ring_barrier();
      if (wave % NWN == 1)
#pragma unroll
        for (int j = 0; j < TJ; ++j) ups[j * 64] = product.total[0][j];
      ring_barrier();
      if (wave % NWN == 0)
#pragma unroll
        for (int j = 0; j < TJ; ++j) gated(product.total[0][j], ups[j * 64], j, n_base);
    } else {
#pragma unroll
      for (int i = 0; i < TI; i += 2)
#pragma unroll
        for (int j = 0; j < TJ; ++j) gated(product.total[i][j], product.total[i + 1][j], j, n_base + wn + i * 16);
    }
  } else {
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        const f32x4& total = product.total[i][j];
        const float t[4] = {total[0], total[1], total[2], total[3]};
        const int m = m_base + wm + j * 16 + row16, n = n_base + wn + i * 16 + g * 4;
        if constexpr (EPI == kXielu) epilogue_xielu4<T>(C, ldc, m, n, M, N, t, vec_ok, factors);
        else epilogue4<T, EPI>(C, ldc, m, n, M, N, t, vec_ok);
      }
  }
}

}  // namespace ls
