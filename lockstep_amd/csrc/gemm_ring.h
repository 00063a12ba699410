// The tiled product of gemm.hip: BM x BN outputs a workgroup, both operands through LDS, and a ring of
// stages that the memory writes into LDS by itself (buffer loads with LDS as their target), so that a stage
// takes no register and no instruction of its own on its way; a ring of n stages has n - 1 of them in flight.
//
// What bounds it: a workgroup's stage (128 bytes of K of all its rows) has to arrive before anyone may
// multiply it, and takes 1 to 2 us from the memory side; a CU's 160 KB of LDS hold two to five stages, so the
// larger the tile, the more multiplications stand behind a byte in flight.  Counters (256 x 192 tiles, 2,048 x
// 24,576 x 4,096): of the cycles that a CU is busy the matrix pipe is busy 56 %, LDS 24 %, no bank conflicts; the clock falls
// to 1.9 GHz under this load.  Measured against the register-staged kernel that was here before (bfloat16, weights from
// HBM, us): 2,048 x 24,576 x 4,096 471 -> 341 (1,210 TFLOP/s), 2,048 x 6,144 x 4,096 142 -> 86, 2,048 x 4,096 x
// 12,288 218 -> 164 (1,255), 999 x 4,096 x 4,096 64 -> 38, 97 x 4,096 x 1,024 10.0 -> 7.0; float32 2,000 x
// 1,024 x 2,048 90 -> 71 (118 TFLOP/s).
//
// How a stage is laid out: rows of 128 bytes, W's rows and X's rows in rings of their own (the ring of W may be
// longer: its lines come from HBM, X's mostly from the XCD's L2).  The 16-byte piece q of row r lies in slot q ^
// (r & 7), so that the sixteen rows a fragment read takes together lie in different banks; a lane of a load picks
// its piece accordingly, inside the same 128-byte line.
//
// How the steps interlock (XS and WS stages of X and W in LDS, one barrier a stage):
//   first half of stage st:  multiply its first chunk, read the fragments of the second;
//                            request W's stage st + WS - 1 into the buffer that stage st - 1 left;
//   wait until the own loads of stage st + 1 are there, then the barrier: now stage st + 1 is whole, and
//   everyone's reads of stage st are done (lgkmcnt(0) in front of the barrier);
//   second half:             request X's stage st + XS into the buffer of stage st;
//                            multiply the second chunk, read the first fragments of stage st + 1.
// Loads complete in the order of their issue, so a wait counts the younger ones; where the last stages leave
// fewer in flight it waits for all.  Every load has landed before the kernel's last barrier (the wait in front
// of it is for all), so no workgroup ends with LDS still being written.
//
// A weight fragment is replaced in its register as soon as the products of its tile have been issued, so the
// sums, their totals (the K slices are folded in order) and one set of fragments fit 256 registers at 64 x 96
// outputs a wave.  Requesting a stage's loads one by one between the products was measured and gave nothing
// (2 to 5 % less at the two largest tiles), nor did s_setprio around the products.
#pragma once

#include "common.h"
#include "ring.h"

namespace ls {

// NWM x NWN waves.  Rows of X and W are 16-byte aligned and K is whole 16-byte pieces; columns from K on, which the
// last stage may hold, are cleared in LDS once it has landed.
template <typename T, int EPI, int BM, int BN, int NWM, int NWN, int WS, int XS>
__global__ __launch_bounds__(64 * NWM * NWN) void gemm_ring_kernel(const T* __restrict__ X, const T* __restrict__ W,
                                                        void* __restrict__ C, int M, int N, int K, long ldx, long ldc,
                                                        int kslice, int vec_ok, int tiles_m, int tiles_n, int out_cols,
                                                        const float* __restrict__ act) {
  typedef Atom<T> A;
  typedef typename A::vec_t vec_t;
  const Factors factors = load_factors<EPI>(act);
  constexpr bool SLICES = EPI == kSliceSums;
  constexpr int NW = NWM * NWN;
  constexpr int BK = 128 / sizeof(T);         // elements of K a stage (two chunks)
  constexpr int TI = BN / (16 * NWN);         // weight tiles (16 columns) a wave
  constexpr int TJ = BM / (16 * NWM);         // row tiles a wave
  constexpr int LW = BN / (8 * NW), LX = BM / (8 * NW);  // a wave's loads a stage: eight rows each
  constexpr int W_BYTES = BN * 128, X_BYTES = BM * 128;
  static_assert(BN % (8 * NW) == 0 && BM % (8 * NW) == 0 && TI * 16 * NWN == BN && TJ * 16 * NWM == BM, "tile shape");
  static_assert(WS >= 3 && WS >= XS && XS >= 2, "rings");
  static_assert(EPI != kSwiGLU || TI % 2 == 0, "a wave holds the gate and the up tile of its columns");
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

  auto request_w = [&](int st, int buf) LS_INLINED {
#pragma unroll
    for (int i = 0; i < LW; ++i)
      buffer_to_lds16(w_off, (first_stage + st) * 128 + i * w_step, w_buffer, lds0 + buf * W_BYTES + i * NW * 1024);
  };
  auto request_x = [&](int st, int buf) LS_INLINED {
#pragma unroll
    for (int i = 0; i < LX; ++i)
      buffer_to_lds16(x_off, (first_stage + st) * 128 + i * x_step, x_buffer,
                      lds0 + WS * W_BYTES + buf * X_BYTES + i * NW * 1024);
  };

  f32x4 total[TI][TJ], acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) total[i][j] = acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto store_slice = [&](int slice) LS_INLINED {  // the sums of one slice to their place among the slice sums
    float* sums = reinterpret_cast<float*>(C) + (long)slice * M * N;
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        const float t[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
        epilogue4<T, kStoreF32>(sums, ldc, m_base + wm + j * 16 + row16, n_base + wn + i * 16 + g * 4, M, N, t, vec_ok);
      }
  };

  const bool ragged = K % BK != 0 && first_stage + stages == all_stages;  // uniform: the last stage is this workgroup's
  auto clear_past_k = [&](int wb, int xb) LS_INLINED {
    const int first = (K % BK) / A::VEC;  // the first piece of a row that lies past K
    for (int idx = threadIdx.x; idx < (BN + BM) * 8; idx += 64 * NW) {
      const int row = idx >> 3;
      if (((idx & 7) ^ (row & 7)) < first) continue;
      unsigned char* at = row < BN ? ring + wb * W_BYTES + idx * 16 : ring + WS * W_BYTES + xb * X_BYTES + (idx - BN * 8) * 16;
      *reinterpret_cast<vec_t*>(at) = A::zero();
    }
    ring_barrier();
  };

  // Fragments: a lane's 16 bytes of chunk c of row 16 i + row16; chunk 1 lies four slots (64 bytes) across.
  const unsigned at = row16 * 128 + ((g ^ (row16 & 7)) << 4);
  vec_t a[TI], b[2][TJ];
  auto read_b = [&](vec_t (&dst)[TJ], int buf, int c) LS_INLINED {
    const unsigned char* src = ring + WS * W_BYTES + buf * X_BYTES + wm * 128 + (at ^ (c * 64));
#pragma unroll
    for (int j = 0; j < TJ; ++j) dst[j] = *reinterpret_cast<const vec_t*>(src + j * 2048);
  };
  // the products of the chunk in (a, mine); a and `next` get the fragments of chunk c of the stage in (wb, xb)
  auto multiply = [&](const vec_t (&mine)[TJ], vec_t (&next)[TJ], int wb, int xb, int c) LS_INLINED {
    const unsigned char* src = ring + wb * W_BYTES + wn * 128 + (at ^ (c * 64));
    read_b(next, xb, c);
#pragma unroll
    for (int i = 0; i < TI; ++i) {
#pragma unroll
      for (int j = 0; j < TJ; ++j) A::mma(acc[i][j], a[i], mine[j]);
      a[i] = *reinterpret_cast<const vec_t*>(src + i * 2048);
    }
  };

#pragma unroll
  for (int s = 0; s < WS; ++s) {
    if (s < XS && s < stages) request_x(s, s);
    if (s < WS - 1 && s < stages) request_w(s, s);
  }
  if (stages >= WS) wait_loads<(XS - 1) * LX + (WS - 2) * LW>(); else wait_loads<0>();
  ring_barrier();
  if (ragged && stages == 1) clear_past_k(0, 0);
  read_b(b[0], 0, 0);
#pragma unroll
  for (int i = 0; i < TI; ++i) a[i] = *reinterpret_cast<const vec_t*>(ring + wn * 128 + at + i * 2048);

  int wb = 0, xb = 0, left = per_slice;
  for (int st = 0; st < stages; ++st) {
    if (left == 0) {
      left = per_slice;
      if (SLICES) store_slice((first_stage + st) / per_slice - 1);
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
#pragma unroll
          for (int r = 0; r < 4; ++r) total[i][j][r] = total[i][j][r] + acc[i][j][r];
          acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    --left;
    if (st + WS - 1 < stages) request_w(st + WS - 1, wb == 0 ? WS - 1 : wb - 1);
    multiply(b[0], b[1], wb, xb, 1);
    // in flight behind what stage st + 1 needs: the W just requested and XS - 2 (XS == WS: no newer W than X's)
    // whole stages
    if (st + WS > stages) wait_loads<0>();
    else if (XS < WS) wait_loads<(XS - 2) * (LX + LW) + LW>();
    else wait_loads<(XS - 2) * (LX + LW)>();
    ring_barrier();
    if (st + XS < stages) request_x(st + XS, xb);
    wb = wb + 1 == WS ? 0 : wb + 1;
    xb = xb + 1 == XS ? 0 : xb + 1;
    if (ragged && st + 2 == stages) clear_past_k(wb, xb);  // (nothing is in flight: WS >= 3)
    // (behind the last stage this reads the fragments of a stage that is not there: they are not used)
    multiply(b[1], b[0], wb, xb, 0);
  }

  if constexpr (SLICES) {
    if (stages > 0) store_slice((first_stage + stages - 1) / per_slice);
  } else {
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) total[i][j][r] = total[i][j][r] + acc[i][j][r];
    if constexpr (EPI == kSwiGLU) {  // the wave's weight tiles come in pairs (gate t, up t)
#pragma unroll
      for (int i = 0; i < TI; i += 2)
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
          const float gate[4] = {total[i][j][0], total[i][j][1], total[i][j][2], total[i][j][3]};
          const float up[4] = {total[i + 1][j][0], total[i + 1][j][1], total[i + 1][j][2], total[i + 1][j][3]};
          epilogue_swiglu4<T>(C, ldc, m_base + wm + j * 16 + row16, (n_base + wn + i * 16) / 2 + g * 4, M, out_cols,
                              gate, up, vec_ok);
        }
    } else {
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
          const float t[4] = {total[i][j][0], total[i][j][1], total[i][j][2], total[i][j][3]};
          const int m = m_base + wm + j * 16 + row16, n = n_base + wn + i * 16 + g * 4;
          if constexpr (EPI == kXielu) epilogue_xielu4<T>(C, ldc, m, n, M, N, t, vec_ok, factors);
          else epilogue4<T, EPI>(C, ldc, m, n, M, N, t, vec_ok);
        }
    }
  }
}

}  // namespace ls
