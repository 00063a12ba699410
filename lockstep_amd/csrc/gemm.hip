// C[M,N] = X[M,K] * W[N,K]^T with a fixed summation order per output element.
//
// The order, for every (m, n), whatever M is and whichever kernel runs:
//   K is cut into slices of `kslice` elements (a function of K alone);
//   inside a slice the products are accumulated by a chain of MFMA atoms over
//   ascending 64-byte chunks of K, starting from zero;
//   the slice sums are added in ascending order to a total that starts at +0.
// The skinny kernel (M <= 64, decode) gives each slice to a wave, so the
// weights stream from HBM with many waves in flight; the streaming kernel
// does the same for products with many columns, one workgroup walking many
// column blocks; the slice kernels leave the slice sums to their consumer; the
// ring kernel (gemm_ring.h: prefill, and decode over many columns) walks the
// slices one after the other with both operands staged in LDS, or (slice sums
// of 17 rows and more) a group of them a workgroup; the tiled kernel does the
// same for operands that are not 16-byte aligned.  All produce the same bits for
// a row, so a token's projections do not depend on how many tokens share its step.
//
// The MFMA runs "swapped": W rows are the first operand, X rows the second,
// so a lane ends with four consecutive n of one row m and stores them as one
// vector.

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "row_piece.h"
#include "core_api.h"

namespace ls {

#ifndef LS_GEMM_SLICES_WIDE
#define LS_GEMM_SLICES_WIDE 1       // 0: never the wide slice kernel
#endif
#ifndef LS_GEMM_SLICES_WIDE_WGS
#define LS_GEMM_SLICES_WIDE_WGS 192  // its workgroups (64 columns, up to four slices) must be at least this many
#endif
#ifndef LS_GEMM_SLICES_WIDE_UNR
#define LS_GEMM_SLICES_WIDE_UNR 2   // chunks it loads at a time
#endif
#ifndef LS_GEMM_STREAM
#define LS_GEMM_STREAM 1      // 0: never the streaming kernel
#endif
#ifndef LS_GEMM_GROUP_M
#define LS_GEMM_GROUP_M 4     // row tiles per band of the tile numbering
#endif
static_assert(LS_GEMM_GROUP_M > 0, "a band of the tile numbering has a row of tiles at least");
#ifndef LS_GEMM_READ_AHEAD
#define LS_GEMM_READ_AHEAD 1  // the tiled kernel reads a stage's second chunk of fragments from LDS before it multiplies the first
#endif
#ifndef LS_GEMM_SLICES_TILED
#define LS_GEMM_SLICES_TILED 1      // 0: never the ring kernel for slice sums
#endif
#ifndef LS_GEMM_PD_SMALL
#define LS_GEMM_PD_SMALL 4    // register prefetch depth (stages) of the tiled kernel (measured 1 to 4: 4 is 2 to 10 % ahead of 2)
#endif

enum Epilogue : int {
  kStore = 0,     // C[m][n] = total, in the compute dtype
  kStoreF32 = 1,  // C[m][n] = total, float
  kAddF32 = 2,    // C[m][n] += total, float (residual stream)
  kSwiGLU = 3,    // W holds gate and up rows interleaved in tiles of 16 (gate rows 16t.., then up rows 16t..);
                  // C[m][16t + i] = (g * 1/(1 + exp(-g))) * u in float, stored in the compute dtype
  kSliceSums = 4, // the ring kernel only: C is float [slices][M][N] and gets the sums of the K slices, not their
                  // total; the workgroups with blockIdx.y = y take the slices [y * out_cols, (y + 1) * out_cols)
  kXielu = 5,     // C[m][n] = xielu(total) in the compute dtype, the activation's two factors from act[0], act[1]
};

__host__ __device__ inline int kslice_for(int K) { return 256 * ((K + 4095) / 4096); }

// `old`: for kAddF32 with vector stores, the four values the element's owner
// has already read from C (nullptr: read them here).
template <typename T, int EPI>
__device__ __forceinline__ void epilogue4(void* __restrict__ C, long ldc, int m, int n, int M, int N,
                                          const float total[4], bool vec_ok, const f32x4* old_vals = nullptr) {
  if (m >= M || n >= N) return;
  if (EPI == kStore) {
    T* row = reinterpret_cast<T*>(C) + (long)m * ldc;
    if (vec_ok && n + 3 < N) {
      if (sizeof(T) == 2) {
        bf16x4 v;
        v[0] = (bf16_t)total[0]; v[1] = (bf16_t)total[1]; v[2] = (bf16_t)total[2]; v[3] = (bf16_t)total[3];
        *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16_t*>(C) + (long)m * ldc + n) = v;
      } else {
        *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(C) + (long)m * ldc + n) =
            f32x4{total[0], total[1], total[2], total[3]};
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < N) row[n + r] = from_f32<T>(total[r]);
    }
  } else {
    float* row = reinterpret_cast<float*>(C) + (long)m * ldc;
    if (vec_ok && n + 3 < N) {
      f32x4* p = reinterpret_cast<f32x4*>(row + n);
      f32x4 v = f32x4{total[0], total[1], total[2], total[3]};
      if (EPI == kAddF32) {
        const f32x4 old = old_vals ? *old_vals : *p;
        v = f32x4{old[0] + v[0], old[1] + v[1], old[2] + v[2], old[3] + v[3]};
      }
      *p = v;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < N) row[n + r] = (EPI == kAddF32) ? row[n + r] + total[r] : total[r];
    }
  }
}

// SwiGLU epilogue on the float totals of a gate tile and the matching up tile.
template <typename T>
__device__ __forceinline__ void epilogue_swiglu4(void* __restrict__ C, long ldc, int m, int col, int M, int width,
                                                 const float gate[4], const float up[4], bool vec_ok) {
  if (m >= M || col >= width) return;
  float act[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float sig = 1.0f / (1.0f + expf(-gate[r]));
    act[r] = (gate[r] * sig) * up[r];
  }
  epilogue4<T, kStore>(C, ldc, m, col, M, width, act, vec_ok);
}

// e^z - 1 - z for z <= 0, where the terms cancel near zero: the library's e^z - 1 on the 32-bit path.  In front of a
// rounding to bfloat16 the hardware's exponential: what it loses is 1e-7 at most, beside the z/2 that is added to it.
template <typename T> __device__ __forceinline__ float exp_beyond_linear(float z);
template <> __device__ __forceinline__ float exp_beyond_linear<float>(float z) { return expm1f(z) - z; }
template <> __device__ __forceinline__ float exp_beyond_linear<bf16_t>(float z) { return (__expf(z) - 1.0f) - z; }

// xIELU of a float total:  up z^2 + z/2 above zero,  down (e^z - 1 - z) + z/2 elsewhere.
template <typename T>
__device__ __forceinline__ float xielu(float z, float up, float down) {
  return (z > 0.f ? up * (z * z) : down * exp_beyond_linear<T>(fminf(z, 0.f))) + 0.5f * z;
}

// The activation's two factors, asked for when a kernel starts (they are needed when it ends).
struct Factors {
  float up, down;
};
template <int EPI>
__device__ __forceinline__ Factors load_factors(const float* __restrict__ act) {
  if constexpr (EPI == kXielu) return Factors{act[0], act[1]};
  return Factors{0.f, 0.f};
}

template <typename T>
__device__ __forceinline__ void epilogue_xielu4(void* __restrict__ C, long ldc, int m, int n, int M, int N,
                                                const float total[4], bool vec_ok, const Factors& factors) {
  if (m >= M || n >= N) return;
  float v[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = xielu<T>(total[r], factors.up, factors.down);
  epilogue4<T, kStore>(C, ldc, m, n, M, N, v, vec_ok);
}

// RMSNorm of rows of the float residual stream, as a prologue of the skinny
// kernel (at most 16 rows): the sum of squares of a row is formed exactly as
// rmsnorm_kernel forms it (row_sumsq_part over the first 256 threads, a
// butterfly over the wave, the four wave sums in wave order), so the
// normalised operand has the same bits as the stand-alone kernel's.
template <int NW>
__device__ __forceinline__ void row_scales(const float* __restrict__ H, long ldh, int M, int K, float eps,
                                           float* __restrict__ wave_part /*[16][4]*/, float* __restrict__ scale /*[16]*/) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  if (wave < 4) {
    const bool vec_ok = (ldh & 3) == 0 && (reinterpret_cast<uintptr_t>(H) & 15) == 0;
    // four rows at a time, so that their loads are in flight together
    for (int m0 = 0; m0 < M; m0 += 4) {
      float part[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        part[j] = row_sumsq_part(H + (long)min(m0 + j, M - 1) * ldh, K, threadIdx.x, vec_ok);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float total = wave_sum(part[j]);
        if (lane == 0 && m0 + j < M) wave_part[(m0 + j) * 4 + wave] = total;
      }
    }
  }
  __syncthreads();
  if (threadIdx.x < 16) {
    const float* p = wave_part + threadIdx.x * 4;
    const float total = ((p[0] + p[1]) + p[2]) + p[3];
    scale[threadIdx.x] = 1.0f / sqrtf(total / (float)K + eps);
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------
// Skinny kernel: one workgroup per 16 output columns, NW waves, wave w takes
// slices w, w + NW, ...; slice sums meet in LDS and are folded in ascending
// order by the thread that owns the output element.
// ---------------------------------------------------------------------------
template <typename T, int MT, int NW, int EPI, bool NORM, bool WHOLE>
__global__ __launch_bounds__(NW * 64) void gemm_skinny_kernel(const void* __restrict__ Xv, const T* __restrict__ W,
                                                               void* __restrict__ C, int M, int N, int K, long ldx,
                                                               long ldc, int kslice, int aligned, int vec_ok,
                                                               const float* __restrict__ norm_w, float eps,
                                                               int out_cols, const float* __restrict__ act) {
  typedef Atom<T> A;
  typedef typename A::vec_t vec_t;
  constexpr int NT = (EPI == kSwiGLU) ? 2 : 1;  // weight tiles per workgroup
  const Factors factors = load_factors<EPI>(act);
  extern __shared__ float part[];                // [nslices][NT][MT][256] (+ 80 floats with NORM)

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * 16 * NT;
  const int row16 = lane & 15;
  const int g = lane >> 4;
  const int nslices = (K + kslice - 1) / kslice;

  const T* X = reinterpret_cast<const T*>(Xv);
  const float* H = reinterpret_cast<const float*>(Xv);
  // UNR chunks at a time: all their loads are issued before the first MFMA
  // needs one, so a wave keeps several kilobytes in flight.
  // as many chunks as the registers of a wave allow (512 / (NW / 4) a lane), so that a slice of 256 elements is one round
  constexpr int UNR = ((NT + MT) * 8 * 4 + NT * MT * 4 + 32 <= 2048 / NW && !NORM) ? 8 : 4;
  auto load_w = [&](int k0, int k_end, vec_t (&w)[NT][UNR]) LS_INLINED {
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      const int k = k0 + u * A::KCHUNK + g * A::VEC;
      const bool in = k0 + u * A::KCHUNK < k_end;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int n = n0 + t * 16 + row16;
        w[t][u] = row_piece<T, WHOLE>(W + (long)n0 * K, t * 16 + row16, k, K, K, (n < N) & in, aligned);
      }
    }
  };
  float my_scale = 0.f;
  vec_t w_first[NT][UNR];  // with NORM: the wave's first weights are in flight while the rows are reduced
  if (NORM) {
    if (wave < nslices) load_w(wave * kslice, min(K, (wave + 1) * kslice), w_first);
    float* wave_part = part + nslices * NT * MT * 256;
    float* scale = wave_part + 64;
    row_scales<NW>(H, ldx, M, K, eps, wave_part, scale);
    my_scale = row16 < M ? scale[row16] : 0.f;
  }
  const bool norm_vec = NORM && aligned && ldx % 4 == 0 && reinterpret_cast<uintptr_t>(norm_w) % 16 == 0;

  // kAddF32: the owner of an output element reads its old value now, not after the products
  f32x4 old_vals = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool preload = EPI == kAddF32 && vec_ok && (int)threadIdx.x < MT * 64 &&
                       (int)(threadIdx.x >> 6) * 16 + row16 < M && n0 + g * 4 + 3 < N;
  if (preload)
    old_vals = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(C) +
                                               (long)((threadIdx.x >> 6) * 16 + row16) * ldc + n0 + g * 4);

  for (int s = wave; s < nslices; s += NW) {
    f32x4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int k_begin = s * kslice;
    const int k_end = min(K, k_begin + kslice);
    for (int k0 = k_begin; k0 < k_end; k0 += UNR * A::KCHUNK) {
      vec_t w[NT][UNR], x[MT][UNR];
      if (NORM && s == wave && k0 == k_begin) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int u = 0; u < UNR; ++u) w[t][u] = w_first[t][u];
      } else {
        load_w(k0, k_end, w);
      }
#pragma unroll
      for (int u = 0; u < UNR; ++u) {
        const int k = k0 + u * A::KCHUNK + g * A::VEC;
        const bool in = k0 + u * A::KCHUNK < k_end;
        if (NORM) {
          // normalise on the fly: (x * scale) * weight, rounded to the compute dtype
          vec_t v = A::zero();
          const bool valid = row16 < M && in && k < K;
          if (norm_vec) {  // uniform: rows and k are 16-byte aligned and K is a multiple of VEC
            const float* src = H + (valid ? (long)row16 * ldx + k : 0);
            const float* wsrc = norm_w + (valid ? k : 0);
#pragma unroll
            for (int q4 = 0; q4 < A::VEC / 4; ++q4) {
              const f32x4 xs = *reinterpret_cast<const f32x4*>(src + 4 * q4);
              const f32x4 ws = *reinterpret_cast<const f32x4*>(wsrc + 4 * q4);
#pragma unroll
              for (int e = 0; e < 4; ++e) v[4 * q4 + e] = from_f32<T>((xs[e] * my_scale) * ws[e]);
            }
            if (!valid) v = A::zero();
          } else if (valid) {
            const float* src = H + (long)row16 * ldx + k;
#pragma unroll
            for (int e = 0; e < A::VEC; ++e)
              if (k + e < K) v[e] = from_f32<T>((src[e] * my_scale) * norm_w[k + e]);
          }
          x[0][u] = v;
        } else {
#pragma unroll
          for (int j = 0; j < MT; ++j)
            x[j][u] = row_piece<T, WHOLE>(X, j * 16 + row16, k, K, ldx, (j * 16 + row16 < M) & in, aligned);
        }
      }
      if constexpr (WHOLE) __builtin_amdgcn_sched_barrier(0);  // (the scheduler would move the loads down to their products, two in flight at a time)
#pragma unroll
      for (int u = 0; u < UNR; ++u) {
        if (!WHOLE && k0 + u * A::KCHUNK >= k_end) break;  // uniform: a chunk is visited iff it starts inside the slice
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int j = 0; j < MT; ++j) A::mma(acc[t][j], w[t][u], x[j][u]);
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < MT; ++j)
        *reinterpret_cast<f32x4*>(&part[(((s * NT + t) * MT + j) * 64 + lane) * 4]) = acc[t][j];
  }
  __syncthreads();

  for (int idx = threadIdx.x; idx < MT * 64; idx += NW * 64) {
    const int j = idx >> 6;
    const int l = idx & 63;
    float total[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int r = 0; r < 4; ++r) total[t][r] = 0.f;
      for (int s = 0; s < nslices; ++s) {
        f32x4 p = *reinterpret_cast<const f32x4*>(&part[(((s * NT + t) * MT + j) * 64 + l) * 4]);
#pragma unroll
        for (int r = 0; r < 4; ++r) total[t][r] = total[t][r] + p[r];
      }
    }
    const int m = j * 16 + (l & 15);
    if (EPI == kSwiGLU)
      epilogue_swiglu4<T>(C, ldc, m, blockIdx.x * 16 + (l >> 4) * 4, M, out_cols, total[0], total[NT - 1], vec_ok);
    else if constexpr (EPI == kXielu)
      epilogue_xielu4<T>(C, ldc, m, n0 + (l >> 4) * 4, M, N, total[0], vec_ok, factors);
    else
      epilogue4<T, EPI>(C, ldc, m, n0 + (l >> 4) * 4, M, N, total[0], vec_ok,
                        (preload && idx == (int)threadIdx.x) ? &old_vals : nullptr);
  }
}

// ---------------------------------------------------------------------------
// Streaming kernel (at most 32 rows, many output columns): the skinny kernel's
// arithmetic with another walk.  A workgroup has one wave per K slice and
// takes the column blocks b = blockIdx.x, blockIdx.x + gridDim.x, ...  A wave
// keeps its slice of X in registers for the whole walk, so the rows of X are
// read once per workgroup instead of once per 16 columns (with 8 rows that is
// half as much again as the weights themselves), and the weights of its next
// unit (UC chunks of a tile) are always in flight while it multiplies the
// current one, also across column blocks and across the two barriers of the
// fold.  Slice sums meet in LDS and are folded in ascending order, as in the
// skinny kernel.
// ---------------------------------------------------------------------------
template <typename T, int MT, int EPI, int XC, bool WHOLE>
__global__ __launch_bounds__(1024) void gemm_stream_kernel(const T* __restrict__ X, const T* __restrict__ W,
                                                           void* __restrict__ C, int M, int N, int K, long ldx,
                                                           long ldc, int kslice, int aligned, int vec_ok,
                                                           int out_cols, int blocks, int row_groups, int block_cols,
                                                           const float* __restrict__ act) {
  typedef Atom<T> A;
  typedef typename A::vec_t vec_t;
  constexpr int NT = (EPI == kSwiGLU) ? 2 : 1;  // weight tiles per column block
  const int cols = NT == 2 ? 16 : block_cols;   // of a block: 16 or 12
  const Factors factors = load_factors<EPI>(act);
  constexpr int UC = 4;                          // chunks per unit
  constexpr int UQ = XC / UC;                    // units per tile
  constexpr int UNITS = NT * UQ;                 // units per column block
  constexpr int RING = (MT * XC <= 8) ? 4 : 2;   // unit buffers in registers: one in use, the others in flight
  constexpr int AHEAD = RING - 1;
  static_assert(XC % UC == 0, "a tile is a whole number of units");
  extern __shared__ float part[];  // [2][waves][NT][MT][256]

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = blockDim.x >> 6;  // = number of K slices
  const int row16 = lane & 15;
  const int g = lane >> 4;
  const int k_begin = wave * kslice;
  const int k_end = min(K, k_begin + kslice);
  // With more than 16 * MT rows the rows are cut into groups of 16 * MT, each with workgroups of its own
  // that walk the same column blocks.  Workgroup ids go round the XCDs, so the ids 8i .. 8i + 7 of one group
  // and the next eight ids of the other group sit pairwise on the same XCD and walk in step: what one of
  // them has fetched, the other finds in that XCD's L2.
  const int id = blockIdx.x;
  const int row_group = row_groups > 1 ? (id >> 3) % row_groups : 0;
  const int walker = row_groups > 1 ? (id / (8 * row_groups)) * 8 + (id & 7) : id;
  const int walkers = gridDim.x / row_groups;
  const int m_base = row_group * MT * 16;

  auto fetch = [&](int b, int t, int q, vec_t (&dst)[UC]) LS_INLINED {
    const int n = (b * NT + t) * cols + row16;
#pragma unroll
    for (int c = 0; c < UC; ++c) {
      const int kc = k_begin + (q * UC + c) * A::KCHUNK;
      dst[c] = row_piece<T, WHOLE>(W + (long)(b * NT + t) * cols * K, row16, kc + g * A::VEC, K, K, (row16 < cols) & (n < N) & (kc < k_end),
                                   aligned, b < blocks);
    }
  };

  // Units are numbered through the walk: unit u of the workgroup is unit u % UNITS of its block u / UNITS
  // and lives in buffer u % RING.
  vec_t xs[MT][XC];
#pragma unroll
  for (int j = 0; j < MT; ++j)
#pragma unroll
    for (int c = 0; c < XC; ++c) {
      const int kc = k_begin + c * A::KCHUNK;
      xs[j][c] = row_piece<T, WHOLE>(X, m_base + j * 16 + row16, kc + g * A::VEC, K, ldx,
                                     m_base + j * 16 + row16 < M && kc < k_end, aligned);
    }
  if constexpr (WHOLE) __builtin_amdgcn_sched_barrier(0);
  vec_t wbuf[RING][UC];
  int b = walker;
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) {
    const int bu = b + (u / UNITS) * walkers;
    fetch(bu, (u % UNITS) / UQ, (u % UNITS) % UQ, wbuf[u % RING]);
    if constexpr (WHOLE) __builtin_amdgcn_sched_barrier(0);  // (in the order in which they are waited for)
  }
  // (X has come before the walk begins: inside it the first product's wait for X would be one for every unit in flight)
  if constexpr (WHOLE) {
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int c = 0; c < XC; ++c) __asm__ volatile("" ::"v"(__builtin_bit_cast(f32x4, xs[j][c])));
  }

  // One column block; `par` is the buffer that holds the block's first unit (static, so that the
  // register buffers are addressed statically).
  static_assert(UNITS % RING == 0 || (2 * UNITS) % RING == 0, "the buffer of a block's first unit has period two");
  auto block_step = [&](auto par, int it) LS_INLINED {
    constexpr int P = decltype(par)::value;
    float* mine = part + (it & 1) * (nw * NT * MT * 256);
    f32x4 acc[MT];  // of the tile in work; a finished tile's sums go to LDS at once
#pragma unroll
    for (int idx = 0; idx < UNITS; ++idx) {
      const int t = idx / UQ;
      const int q = idx % UQ;
      if (q == 0) {
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      const int far_block = b + ((idx + AHEAD) / UNITS) * walkers;  // the block of the unit AHEAD units on
      fetch(far_block, ((idx + AHEAD) % UNITS) / UQ, ((idx + AHEAD) % UNITS) % UQ, wbuf[(P + idx + AHEAD) % RING]);
      if constexpr (WHOLE) __builtin_amdgcn_sched_barrier(0);  // (the scheduler would move the loads down to their products, two in flight at a time)
#pragma unroll
      for (int c = 0; c < UC; ++c) {
        if (!WHOLE && k_begin + (q * UC + c) * A::KCHUNK >= k_end) break;  // uniform: a chunk is visited iff it starts inside the slice
#pragma unroll
        for (int j = 0; j < MT; ++j) A::mma(acc[j], wbuf[(P + idx) % RING][c], xs[j][q * UC + c]);
      }
      if (q == UQ - 1) {
#pragma unroll
        for (int j = 0; j < MT; ++j)
          *reinterpret_cast<f32x4*>(&mine[(((wave * NT + t) * MT + j) * 64 + lane) * 4]) = acc[j];
      }
    }
    // One barrier a block: the next block's sums go to the other half of `part`, and the half
    // written now is written again only after the next barrier, which the folding wave reaches
    // after its fold.
    __syncthreads();
    // row tile j of this block is folded by wave (it * MT + j) % nw, so the duty goes round
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      if ((it * MT + j) % nw != wave) continue;  // uniform for the wave
      float total[NT][4];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int r = 0; r < 4; ++r) total[t][r] = 0.f;
        for (int s = 0; s < nw; ++s) {
          const f32x4 p = *reinterpret_cast<const f32x4*>(&mine[(((s * NT + t) * MT + j) * 64 + lane) * 4]);
#pragma unroll
          for (int r = 0; r < 4; ++r) total[t][r] = total[t][r] + p[r];
        }
      }
      const int m = m_base + j * 16 + row16;
      if (EPI == kSwiGLU)
        epilogue_swiglu4<T>(C, ldc, m, b * 16 + g * 4, M, out_cols, total[0], total[NT - 1], vec_ok);
      else if (g * 4 >= cols)
        continue;  // (the next block's columns)
      else if constexpr (EPI == kXielu)
        epilogue_xielu4<T>(C, ldc, m, b * cols + g * 4, M, N, total[0], vec_ok, factors);
      else
        epilogue4<T, EPI>(C, ldc, m, b * cols + g * 4, M, N, total[0], vec_ok);
    }
  };

  // the first buffer of a block advances by UNITS % RING from block to block
  int it = 0;
  if constexpr (UNITS % RING != 0) {  // UNITS = 2, RING = 4: every other block starts in buffer 2
    for (; b + walkers < blocks;) {   // (no way out between the two, which the loop's waits would be counted by)
      block_step(std::integral_constant<int, 0>{}, it++);
      b += walkers;
      block_step(std::integral_constant<int, UNITS % RING>{}, it++);
      b += walkers;
    }
    if (b < blocks) block_step(std::integral_constant<int, 0>{}, it);
  } else {
    for (; b < blocks; b += walkers) block_step(std::integral_constant<int, 0>{}, it++);
  }
}

// Whether row_piece's 31-bit offsets reach up to 64 aligned rows of both operands.
static bool pieces_reach(long ldx, long K, long size) { return 65 * std::max(ldx, K) * size <= kNoPiece; }

// Dynamic LDS beyond 64 KB has to be granted per kernel (once).
template <typename T, int MT, int EPI, int XC, bool WHOLE>
static bool stream_lds_ready(size_t bytes) {
  if (bytes <= 64 * 1024) return true;
  if (bytes > 128 * 1024) return false;
  static int state = 0;  // 0 unknown, 1 granted, -1 refused
  if (state == 0) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_stream_kernel<T, MT, EPI, XC, WHOLE>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024);
    if (e != hipSuccess) (void)hipGetLastError();
    state = e == hipSuccess ? 1 : -1;
  }
  return state == 1;
}

// ---------------------------------------------------------------------------
// Slice kernel (at most 64 rows): the skinny kernel's slice sums, left
// unfolded.  A workgroup takes 16 output columns and a few consecutive K
// slices, one per wave, and writes each slice's sums to P [slices][M][N]
// (float); whoever consumes P adds the slices in ascending order, which is
// the order every other kernel uses.  Cutting K over workgroups puts a
// product with few output columns on all CUs (a CU alone streams its weights
// slowly), at the price of the fold, which the consumer (add_rmsnorm_kernel)
// does on the way.
// ---------------------------------------------------------------------------
template <typename T, int MT, bool WHOLE>
__global__ __launch_bounds__(256) void gemm_slices_kernel(const T* __restrict__ X, const T* __restrict__ W,
                                                          float* __restrict__ P, int M, int N, int K, long ldx,
                                                          int kslice, int aligned, int slices_per_group) {
  typedef Atom<T> A;
  typedef typename A::vec_t vec_t;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * 16;
  const int row16 = lane & 15;
  const int g = lane >> 4;
  const int nslices = (K + kslice - 1) / kslice;
  const int s = blockIdx.y * slices_per_group + wave;
  if (wave >= slices_per_group || s >= nslices) return;

  f32x4 acc[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int k_begin = s * kslice;
  const int k_end = min(K, k_begin + kslice);
  constexpr int UNR = 8;  // a slice of 256 elements in one round of loads
  for (int k0 = k_begin; k0 < k_end; k0 += UNR * A::KCHUNK) {
    vec_t w[UNR], x[MT][UNR];
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      const int k = k0 + u * A::KCHUNK + g * A::VEC;
      const bool in = k0 + u * A::KCHUNK < k_end;
      w[u] = row_piece<T, WHOLE>(W + (long)n0 * K, row16, k, K, K, (n0 + row16 < N) & in, aligned);
#pragma unroll
      for (int j = 0; j < MT; ++j)
        x[j][u] = row_piece<T, WHOLE>(X, j * 16 + row16, k, K, ldx, (j * 16 + row16 < M) & in, aligned);
    }
    if constexpr (WHOLE) __builtin_amdgcn_sched_barrier(0);  // (the scheduler would move the loads down to their products, two in flight at a time)
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      if (!WHOLE && k0 + u * A::KCHUNK >= k_end) break;  // uniform: a chunk is visited iff it starts inside the slice
#pragma unroll
      for (int j = 0; j < MT; ++j) A::mma(acc[j], w[u], x[j][u]);
    }
  }
  // lane: rows j * 16 + row16 of X, columns n0 + 4g .. n0 + 4g + 3
  const int n = n0 + g * 4;
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int m = j * 16 + row16;
    if (m >= M || n >= N) continue;
    float* dst = P + ((long)s * M + m) * N + n;
    if (n + 3 < N && (N & 3) == 0) {
      *reinterpret_cast<f32x4*>(dst) = acc[j];
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < N) dst[r] = acc[j][r];
    }
  }
}

// The slice kernel for an operand that is still the per-split sums of an attention launch (decoded tokens,
// at most 16 rows): X [m][k] is the output of token m, head k / head_dim, column k % head_dim, which the fold
// over the token's `splits` partial results (acc, m, l), ascending from the empty state, skipping empty ones,
// then acc / l rounded to T, would give.  A workgroup takes one K slice and 64 output columns: its four waves
// fold the slice's elements into LDS together first (every group of 64 columns repeats that, which costs
// little while rows times splits are few), then each wave multiplies its 16 columns from there.  The launch
// that would fold them into an output, and the round trip of that output, are saved.  Partial row of (token
// m, head h, split s): (m * heads + h) * splits + s, as the attention kernels lay single decoded tokens out.
// The fold is the attention library's fold_split operation by operation, and the chain of a slice is
// gemm_slices_kernel's: the same bits as fold, then product.
// UNITS, SPLITS: a thread's groups of four elements whose sums are requested together, and the most splits
// each has (instances for few and for more of either; splits <= SPLITS and the host's choice of UNITS
// change nothing in the arithmetic).  REVERSED: a wrong variant for the tests' control library (descending fold).
template <typename T, bool REVERSED, int UNITS, int SPLITS>
__global__ __launch_bounds__(256) void gemm_slices_folded_kernel(const float* __restrict__ part_acc,
                                                                 const float* __restrict__ part_ml, int splits,
                                                                 int head_dim, const T* __restrict__ W,
                                                                 float* __restrict__ P, int M, int N, int K, int kslice) {
  typedef Atom<T> A;
  typedef typename A::vec_t vec_t;
  extern __shared__ __attribute__((aligned(16))) unsigned char folded_lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * 64 + wave * 16;
  const int row16 = lane & 15;
  const int g = lane >> 4;
  const int s = blockIdx.y;
  const int k_begin = s * kslice;
  const int k_end = min(K, k_begin + kslice);
  const int row_stride = kslice + 16 / (int)sizeof(T);  // elements; the pad spreads the rows over the banks
  T* xs = reinterpret_cast<T*>(folded_lds);             // [M][row_stride]
  const int heads = K / head_dim;

  // The weights of the slice's first round are requested before the sums: both are on their way together, and
  // the fold runs while the weights arrive.
  constexpr int UNR = 8;  // a slice of 256 elements in one round of loads
  vec_t w_first[UNR];
#pragma unroll
  for (int u = 0; u < UNR; ++u) {
    const int k = k_begin + u * A::KCHUNK + g * A::VEC;
    w_first[u] = row_piece<T, true>(W + (long)n0 * K, row16, k, K, K, n0 + row16 < N && k_begin + u * A::KCHUNK < k_end, true);
  }
  __builtin_amdgcn_sched_barrier(0);  // (the scheduler would move these loads down to their use, behind the fold)

  // A unit is four neighbouring elements of one row; thread t takes the units t, t + 256, ...  A unit's
  // splits are folded one after the other; the sums of UNITS units are requested together.
  const int quads = kslice / 4;
  const int units = M * quads;
  for (int u0 = threadIdx.x; u0 < units; u0 += 256 * UNITS) {
    f32x4 acc[UNITS][SPLITS];
    float2 ml[UNITS][SPLITS];
#pragma unroll
    for (int j = 0; j < UNITS; ++j) {
      const int unit = min(u0 + 256 * j, units - 1);                 // (clamped: loaded, not used)
      const int m = unit / quads;
      const int k = min(k_begin + 4 * (unit - m * quads), K - 4);
      const int head = k / head_dim;
      const long pr0 = ((long)m * heads + head) * splits;
      const float* from = part_acc + (k - head * head_dim);
#pragma unroll
      for (int sp = 0; sp < SPLITS; ++sp) {
        const int at = min(sp, splits - 1);
        const long pr = pr0 + (REVERSED ? splits - 1 - at : at);
        acc[j][sp] = *reinterpret_cast<const f32x4*>(from + pr * head_dim);
        ml[j][sp] = *reinterpret_cast<const float2*>(part_ml + pr * 2);
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // every request is made before the first sum is used
#pragma unroll
    for (int j = 0; j < UNITS; ++j) {
      f32x4 run_acc = f32x4{0.f, 0.f, 0.f, 0.f};
      float run_m = kNegSentinel, run_l = 0.f;
#pragma unroll
      for (int sp = 0; sp < SPLITS; ++sp) {
        if (sp < splits && ml[j][sp].y > 0.f) {  // fold_split on these four columns
          const float m_new = fmaxf(run_m, ml[j][sp].x);
          const float fa = softmax_exp<T>(run_m - m_new);
          const float fb = softmax_exp<T>(ml[j][sp].x - m_new);
#pragma unroll
          for (int e = 0; e < 4; ++e) run_acc[e] = run_acc[e] * fa + acc[j][sp][e] * fb;
          run_l = run_l * fa + ml[j][sp].y * fb;
          run_m = m_new;
        }
      }
      const int unit = u0 + 256 * j;
      const int m = unit / quads;
      const int k = k_begin + 4 * (unit - m * quads);
      if (unit < units && k < k_end) {  // the unit is folded: acc / l, rounded as the attention output is
        T* dst = xs + (long)m * row_stride + (k - k_begin);
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[e] = from_f32<T>(run_l > 0.f ? run_acc[e] / run_l : 0.f);
      }
    }
  }
  __syncthreads();
  if (n0 >= N) return;

  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = k_begin; k0 < k_end; k0 += UNR * A::KCHUNK) {
    vec_t w[UNR], x[UNR];
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      const int k = k0 + u * A::KCHUNK + g * A::VEC;
      const bool in = k0 + u * A::KCHUNK < k_end;
      w[u] = k0 == k_begin ? w_first[u] : row_piece<T, true>(W + (long)n0 * K, row16, k, K, K, n0 + row16 < N && in, true);
      x[u] = (row16 < M && in && k < k_end) ? *reinterpret_cast<const vec_t*>(xs + (long)row16 * row_stride + (k - k_begin))
                                            : A::zero();
    }
#pragma unroll
    for (int u = 0; u < UNR; ++u) A::mma(acc, w[u], x[u]);  // (beyond the slice zeros, as row_piece has it)
  }
  const int n = n0 + g * 4;
  if (row16 < M && n < N) {
    float* dst = P + ((long)s * M + row16) * N + n;
    if (n + 3 < N && (N & 3) == 0) {
      *reinterpret_cast<f32x4*>(dst) = acc;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < N) dst[r] = acc[r];
    }
  }
}

// The slice kernel for many rows and many columns: a wave takes one K slice of NTL column tiles (16 * NTL
// columns) and all the rows, so a chunk of X that it has loaded meets NTL chunks of weights and a chunk of
// weights MT chunks of X: at 64 rows and 64 columns the rows of X are read once for every byte of weights,
// where the kernel above reads them four times over.  The chain of a slice is the same (ascending chunks,
// from zero), so are the bits.  UNR chunks are loaded at a time, then multiplied; the CU's other waves
// cover the wait.
template <typename T, int MT, int NTL, int UNR>
__global__ __launch_bounds__(256) void gemm_slices_wide_kernel(const T* __restrict__ X, const T* __restrict__ W,
                                                               float* __restrict__ P, int M, int N, int K, long ldx,
                                                               int kslice, int aligned, int slices_per_group) {
  typedef Atom<T> A;
  typedef typename A::vec_t vec_t;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int n0 = blockIdx.x * 16 * NTL;
  const int s = blockIdx.y * slices_per_group + wave;
  if (wave >= slices_per_group || s >= (K + kslice - 1) / kslice) return;
  const int row16 = lane & 15;
  const int g = lane >> 4;

  f32x4 acc[NTL][MT];
#pragma unroll
  for (int i = 0; i < NTL; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int k_begin = s * kslice;
  const int k_end = min(K, k_begin + kslice);
  for (int k0 = k_begin; k0 < k_end; k0 += UNR * A::KCHUNK) {
    vec_t w[UNR][NTL], x[UNR][MT];
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      const int k = k0 + u * A::KCHUNK + g * A::VEC;
      const bool in = k0 + u * A::KCHUNK < k_end;
#pragma unroll
      for (int i = 0; i < NTL; ++i) {
        const int n = n0 + i * 16 + row16;
        w[u][i] = load_vec<T>(W, n, k, K, K, n < N && in, aligned);
      }
#pragma unroll
      for (int j = 0; j < MT; ++j)
        x[u][j] = load_vec<T>(X, j * 16 + row16, k, K, ldx, j * 16 + row16 < M && in, aligned);
    }
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      if (k0 + u * A::KCHUNK >= k_end) break;  // uniform: a chunk is visited iff it starts inside the slice
#pragma unroll
      for (int i = 0; i < NTL; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) A::mma(acc[i][j], w[u][i], x[u][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < NTL; ++i) {
    const int n = n0 + i * 16 + g * 4;
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      const int m = j * 16 + row16;
      if (m >= M || n >= N) continue;
      float* dst = P + ((long)s * M + m) * N + n;
      if (n + 3 < N && (N & 3) == 0) {
        *reinterpret_cast<f32x4*>(dst) = acc[i][j];
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < N) dst[r] = acc[i][j][r];
      }
    }
  }
}

// The slice kernel as a walk (products with many K slices and enough column
// blocks that workgroups can take several): wave = slice, its rows of X stay
// in registers, the weights of the next units are in flight across column
// blocks as in the streaming kernel.  The waves share nothing, so there is no
// barrier.
template <typename T, int MT, int XC, bool WHOLE>
__global__ __launch_bounds__(256) void gemm_slices_stream_kernel(const T* __restrict__ X, const T* __restrict__ W,
                                                                 float* __restrict__ P, int M, int N, int K, long ldx,
                                                                 int kslice, int aligned, int slices_per_group,
                                                                 int blocks) {
  typedef Atom<T> A;
  typedef typename A::vec_t vec_t;
  constexpr int UC = 4;                          // chunks per unit
  constexpr int UNITS = XC / UC;                 // units per column block
  constexpr int RING = (MT * XC <= 24) ? 4 : 2;  // unit buffers in registers
  constexpr int AHEAD = RING - 1;
  static_assert(XC % UC == 0 && (UNITS % RING == 0 || (2 * UNITS) % RING == 0), "units and ring");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row16 = lane & 15;
  const int g = lane >> 4;
  const int nslices = (K + kslice - 1) / kslice;
  const int s = blockIdx.y * slices_per_group + wave;
  if (wave >= slices_per_group || s >= nslices) return;
  const int k_begin = s * kslice;
  const int k_end = min(K, k_begin + kslice);
  const int walkers = gridDim.x;
  const int m_base = blockIdx.z * MT * 16;  // more than 16 * MT rows: groups of rows, each with workgroups of its own

  auto fetch = [&](int b, int q, vec_t (&dst)[UC]) LS_INLINED {
    const int n = b * 16 + row16;
#pragma unroll
    for (int c = 0; c < UC; ++c) {
      const int kc = k_begin + (q * UC + c) * A::KCHUNK;
      dst[c] = row_piece<T, WHOLE>(W + (long)b * 16 * K, row16, kc + g * A::VEC, K, K, (n < N) & (kc < k_end), aligned, b < blocks);
    }
  };
  vec_t xs[MT][XC];
#pragma unroll
  for (int j = 0; j < MT; ++j)
#pragma unroll
    for (int c = 0; c < XC; ++c) {
      const int kc = k_begin + c * A::KCHUNK;
      xs[j][c] = row_piece<T, WHOLE>(X + (long)m_base * ldx, j * 16 + row16, kc + g * A::VEC, K, ldx,
                                     m_base + j * 16 + row16 < M && kc < k_end, aligned);
    }
  if constexpr (WHOLE) __builtin_amdgcn_sched_barrier(0);
  vec_t wbuf[RING][UC];
  int b = blockIdx.x;
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) {
    const int bu = b + (u / UNITS) * walkers;
    fetch(bu, u % UNITS, wbuf[u % RING]);
    if constexpr (WHOLE) __builtin_amdgcn_sched_barrier(0);  // (in the order in which they are waited for)
  }
  // (X has come before the walk begins: inside it the first product's wait for X would be one for every unit in flight)
  if constexpr (WHOLE) {
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int c = 0; c < XC; ++c) __asm__ volatile("" ::"v"(__builtin_bit_cast(f32x4, xs[j][c])));
  }

  auto block_step = [&](auto par) LS_INLINED {
    constexpr int P0 = decltype(par)::value;
    f32x4 acc[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int idx = 0; idx < UNITS; ++idx) {
      const int far_block = b + ((idx + AHEAD) / UNITS) * walkers;
      fetch(far_block, (idx + AHEAD) % UNITS, wbuf[(P0 + idx + AHEAD) % RING]);
      if constexpr (WHOLE) __builtin_amdgcn_sched_barrier(0);  // (the scheduler would move the loads down to their products, two in flight at a time)
#pragma unroll
      for (int c = 0; c < UC; ++c) {
        if (!WHOLE && k_begin + (idx * UC + c) * A::KCHUNK >= k_end) break;  // uniform: a chunk is visited iff it starts inside the slice
#pragma unroll
        for (int j = 0; j < MT; ++j) A::mma(acc[j], wbuf[(P0 + idx) % RING][c], xs[j][idx * UC + c]);
      }
    }
    const int n = b * 16 + g * 4;
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      const int m = m_base + j * 16 + row16;
      if (m >= M || n >= N) continue;
      float* dst = P + ((long)s * M + m) * N + n;
      if (n + 3 < N && (N & 3) == 0) {
        *reinterpret_cast<f32x4*>(dst) = acc[j];
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < N) dst[r] = acc[j][r];
      }
    }
  };
  if constexpr (UNITS % RING != 0) {
    while (b + walkers < blocks) {
      block_step(std::integral_constant<int, 0>{});
      b += walkers;
      block_step(std::integral_constant<int, UNITS % RING>{});
      b += walkers;
    }
    if (b < blocks) block_step(std::integral_constant<int, 0>{});
  } else {
    for (; b < blocks; b += walkers) block_step(std::integral_constant<int, 0>{});
  }
}

}  // namespace ls
#include "gemm_ring.h"
namespace ls {

// ---------------------------------------------------------------------------
// Tiled kernel: 64 x 64 outputs per workgroup by four waves, for operands that
// the ring kernel does not take (rows that are not 16-byte aligned, K that is
// not whole 16-byte pieces): it loads them element by element.  Both go through
// registers into LDS in stages of 128 bytes of K per row, double buffered.
// ---------------------------------------------------------------------------
constexpr int kRowBytes = 128;               // bytes of K per row per stage (two chunks)
constexpr int kRowStride = kRowBytes + 16;   // padded LDS row

template <typename T, int EPI>
__global__ __launch_bounds__(256) void gemm_tiled_kernel(const T* __restrict__ X, const T* __restrict__ W,
                                                         void* __restrict__ C, int M, int N, int K, long ldx,
                                                         long ldc, int kslice, int vec_ok, int tiles_m, int tiles_n,
                                                         int out_cols, const float* __restrict__ act) {
  typedef Atom<T> A;
  typedef typename A::vec_t vec_t;
  const Factors factors = load_factors<EPI>(act);
  constexpr int BM = 64, BN = 64, NWM = 2, NWN = 2, PD = LS_GEMM_PD_SMALL;
  constexpr int BK = kRowBytes / sizeof(T);  // elements of K per stage
  constexpr int TI = BN / (16 * NWN);        // weight tiles (16 columns) per wave
  constexpr int TJ = BM / (16 * NWM);        // row tiles per wave
  constexpr int PASS = 8 * NWM * NWN;        // rows per staging pass: 8 threads a row
  constexpr int WP = BN / PASS;              // staging passes over the weight tile
  constexpr int XP = BM / PASS;
  static_assert(BN % PASS == 0 && BM % PASS == 0 && TI * 16 * NWN == BN && TJ * 16 * NWM == BM, "tile shape");
  constexpr int STAGE_BYTES = (BM + BN) * kRowStride;
  __shared__ __attribute__((aligned(16))) unsigned char lds[2 * STAGE_BYTES];

  // XCD-aware numbering: workgroup ids go round the eight XCDs; give each XCD a contiguous run of tiles
  int id = blockIdx.x;
  const int total_tiles = tiles_m * tiles_n;
  if (total_tiles % 8 == 0) id = (id % 8) * (total_tiles / 8) + id / 8;
  // ... and inside bands of LS_GEMM_GROUP_M row tiles, so that the workgroups that run together on an XCD
  // form a block of tiles with few distinct operand tiles (those stay in the XCD's L2)
  const int band = id / (LS_GEMM_GROUP_M * tiles_n);
  const int in_band = id % (LS_GEMM_GROUP_M * tiles_n);
  const int band_rows = min(LS_GEMM_GROUP_M, tiles_m - band * LS_GEMM_GROUP_M);
  const int tile_m = band * LS_GEMM_GROUP_M + in_band % band_rows;
  const int tile_n = in_band / band_rows;
  const int m_base = tile_m * BM;
  const int n_base = tile_n * BN;

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wn = (wave % NWN) * (BN / NWN);
  const int wm = (wave / NWN) * (BM / NWM);
  const int row16 = lane & 15;
  const int g = lane >> 4;
  const int st_row = threadIdx.x >> 3;             // staging: 8 threads per row, PASS rows per pass
  const int st_col = (threadIdx.x & 7) * A::VEC;

  f32x4 total[TI][TJ];
  f32x4 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

  // PD stages of global loads are in flight in registers (slot = stage % PD)
  vec_t wv[PD][WP], xv[PD][XP];
  auto fetch = [&](int slot, int k0) LS_INLINED {
#pragma unroll
    for (int p = 0; p < WP; ++p) {
      const int r = st_row + PASS * p;
      wv[slot][p] = load_vec<T>(W, n_base + r, k0 + st_col, K, K, n_base + r < N, false);
    }
#pragma unroll
    for (int p = 0; p < XP; ++p) {
      const int r = st_row + PASS * p;
      xv[slot][p] = load_vec<T>(X, m_base + r, k0 + st_col, K, ldx, m_base + r < M, false);
    }
  };
  auto stash = [&](int slot, int buf) LS_INLINED {
    unsigned char* w_lds = lds + buf * STAGE_BYTES;
    unsigned char* x_lds = w_lds + BN * kRowStride;
#pragma unroll
    for (int p = 0; p < WP; ++p)
      *reinterpret_cast<vec_t*>(&w_lds[(st_row + PASS * p) * kRowStride + st_col * sizeof(T)]) = wv[slot][p];
#pragma unroll
    for (int p = 0; p < XP; ++p)
      *reinterpret_cast<vec_t*>(&x_lds[(st_row + PASS * p) * kRowStride + st_col * sizeof(T)]) = xv[slot][p];
  };

  const int stages = (K + BK - 1) / BK;
  auto k_of = [&](int st) LS_INLINED { return st * BK; };
  // stage s lives in register slot s % PD until it is written to LDS buffer s % 2
  fetch(0, k_of(0));
  stash(0, 0);
#pragma unroll
  for (int u = 1; u <= PD; ++u)
    if (u < stages) fetch(u % PD, k_of(u));
  for (int base = 0; base < stages; base += PD) {
#pragma unroll
    for (int u = 0; u < PD; ++u) {  // unrolled so that the register slots are static
      const int st = base + u;
      if (st >= stages) break;
      const int k0 = k_of(st);
      if (st > 0 && k0 % kslice == 0) {  // a stage never straddles a slice: kslice is a multiple of BK
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int j = 0; j < TJ; ++j) {
#pragma unroll
            for (int r = 0; r < 4; ++r) total[i][j][r] = total[i][j][r] + acc[i][j][r];
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
      }
      __syncthreads();  // stage st is in its buffer; the other buffer has been read by every wave
      if (st + 1 < stages) {
        stash((u + 1) % PD, (st + 1) & 1);
        if (st + 1 + PD < stages) fetch((u + 1) % PD, k_of(st + 1 + PD));
      }
      const unsigned char* w_lds = lds + (st & 1) * STAGE_BYTES;
      const unsigned char* x_lds = w_lds + BN * kRowStride;
      // the fragments of the second chunk are read while the first is multiplied
      vec_t a[2][TI], b[2][TJ];
      auto fragments = [&](int c) LS_INLINED {
#pragma unroll
        for (int i = 0; i < TI; ++i)
          a[c][i] = *reinterpret_cast<const vec_t*>(&w_lds[(wn + i * 16 + row16) * kRowStride + c * 64 + g * 16]);
#pragma unroll
        for (int j = 0; j < TJ; ++j)
          b[c][j] = *reinterpret_cast<const vec_t*>(&x_lds[(wm + j * 16 + row16) * kRowStride + c * 64 + g * 16]);
      };
      fragments(0);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        // The skinny kernel visits a chunk iff it starts below K; do the same.
        if (k0 + c * A::KCHUNK >= K) break;
        if (c == 0 && LS_GEMM_READ_AHEAD) fragments(1);
        if (c == 1 && !LS_GEMM_READ_AHEAD) fragments(1);
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int j = 0; j < TJ; ++j) A::mma(acc[i][j], a[c][i], b[c][j]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) total[i][j][r] = total[i][j][r] + acc[i][j][r];

  if (EPI == kSwiGLU) {
    // the wave's weight tiles come in pairs (gate t, up t)
#pragma unroll
    for (int i = 0; i < TI; i += 2)
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        float gate[4] = {total[i][j][0], total[i][j][1], total[i][j][2], total[i][j][3]};
        float up[4] = {total[i + 1][j][0], total[i + 1][j][1], total[i + 1][j][2], total[i + 1][j][3]};
        epilogue_swiglu4<T>(C, ldc, m_base + wm + j * 16 + row16, (n_base + wn + i * 16) / 2 + g * 4, M, out_cols,
                            gate, up, vec_ok);
      }
    return;
  }
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      float t[4] = {total[i][j][0], total[i][j][1], total[i][j][2], total[i][j][3]};
      if constexpr (EPI == kXielu)
        epilogue_xielu4<T>(C, ldc, m_base + wm + j * 16 + row16, n_base + wn + i * 16 + g * 4, M, N, t, vec_ok, factors);
      else
        epilogue4<T, EPI>(C, ldc, m_base + wm + j * 16 + row16, n_base + wn + i * 16 + g * 4, M, N, t, vec_ok);
    }
}

// The ring kernel's tiles: rows, columns, workgroups of it that a CU holds, and the microseconds a stage takes with one
// workgroup on every CU and with as many as it holds (bfloat16, K = 4,096, weights from HBM).  The larger the tile, the
// fewer operand bytes a product loads; the smaller, the more CUs have one, and the fuller the last round.
enum RingTile { kRing256x192, kRing256x128, kRing192x192, kRing128x192, kRing192x128, kRing128x128, kRing128x64, kRing64x128,
                kRing64x64, kRingTiles, kRing32x64 = kRingTiles, kRing32x32 };
struct RingShape {
  int rows, cols, a_cu;
  float one, full;
};
constexpr RingShape kRingShapes[kRingTiles] = {
    {256, 192, 1, 1.33f, 1.33f}, {256, 128, 1, 0.94f, 0.94f}, {192, 192, 1, 1.00f, 1.00f}, {128, 192, 1, 0.76f, 0.76f},
    {192, 128, 1, 0.73f, 0.73f}, {128, 128, 1, 0.58f, 0.58f}, {128, 64, 1, 0.43f, 0.43f},  {64, 128, 2, 0.52f, 0.74f},
    {64, 64, 2, 0.33f, 0.52f}};

// What `tiles` workgroups cost that a CU holds a_cu of: each round `start` and, for each of a workgroup's stages, stage[n - 1] where the fullest CU
// has n of them.  (Microseconds; a cost, to compare tiles by, and not a time.)
static float rounds_cost(long tiles, int a_cu, int stages, float start, const float* stage) {
  const long cus = compute_units(), rest = tiles % (cus * a_cu);
  float cost = (float)(tiles / (cus * a_cu)) * (start + stage[a_cu - 1] * stages);
  if (rest) cost += start + stage[(rest + cus - 1) / cus - 1] * stages;
  return cost;
}
constexpr float kStages32x32[4] = {0.218f, 0.365f, 0.515f, 0.68f}, kStages64x64[3] = {0.59f, 1.15f, 1.7f};  // float32

// The ring kernel's tile of a product that it runs.
// float32 has four times the matrix work a byte: 32 x 32 tiles, four a CU, or 64 x 64, three a CU, whichever the costs above (fitted to 1,900
// products each) give less (us, 32 x 32 / 64 x 64: 64 x 4,096 x 1,024 10.0 / 22.3, 24 x 51,200 x 2,048 90 / 137, 128 x 10,240 x 4,096 107 / 143, 200
// x 4,096 x 8,344 181 / 164, SwiGLU 64 x 16,384 x 2,048 49.6 / 45.7, 256 x 4,096 x 408 13.9 / 11.7, 2,000 x 1,024 x 1,024 41.4 / 38.1).  64 x 32
// tiles beside these two gained 0.4 %.
// bfloat16: 32 x 32 (stages of 256 bytes, so that a barrier and an LDS latency stand every 128 elements of K) and then 32 x 64 where those tiles are
// one round: a wider one would leave CUs idle, and every workgroup loads 32 rows of both operands or 96 a stage in place of 128.  Up to 32 rows 32 x
// 32 also for three rounds of at least 2,048 of K, 32 x 64 for one and a half to two of at most 512.  Weights from HBM, us, 64 x 64 / these:
//   one round of 32 x 32    SwiGLU 8 x 6,144 x 1,024 7.1 / 5.7, 64 x 4,096 x 1,024 7.9 / 5.4, 64 x 4,096 x 4,096 21.3 / 12.4, 97 x 1,024 x 2,048 9.6 /
//                           6.5, 200 x 1,024 x 4,096 17.0 / 11.4
//   one round of 32 x 64    8 x 10,240 x 5,120 23.1 / 22.3, SwiGLU 1 x 14,336 x 1,024 8.0 / 7.5, 64 x 6,144 x 4,096 22.3 / 18.0, 97 x 4,096
//                           x 1,024 7.6 / 6.5; 32 x 32 tiles, two a CU, 6.9 for the last
//   up to 32 rows           SwiGLU 8 x 24,576 x 4,096 40.2 / 35.6 in 32 x 32, 32 x 24,544 x 512 in 32 x 64; four rounds ask for 128 rows of weights a
//                           multiple of 4 KB apart together (8 x 32,768 x 4,096 51.9 / 64.9)
// Others the tile whose rounds of workgroups take least by the table above.  (Every tile forced in turn over 65 to 2,048 rows and nine
// shapes of weights: within 2 % of the best one at 130 of 135 sizes, 5 % at the rest.)  One rule stands in front of it: up to 64 rows whose rows of weights lie a multiple of 4 KB apart
// take 64 x 64 tiles (128 such rows asked for together meet in few memory channels: 16 x 32,768 x 4,096 62.6 -> 55.1 us; other K 0.9 to 1.05 times as long).
template <typename T>
static int ring_tile(int M, int N, int K) {
  const long cus = compute_units();
  auto tiles = [&](int rows, int cols) { return (long)((M + rows - 1) / rows) * ((N + cols - 1) / cols); };
  if (sizeof(T) == 4) {
    const int stages = (K + 31) / 32;
    return rounds_cost(tiles(32, 32), 4, stages, 0.9f, kStages32x32) <= rounds_cost(tiles(64, 64), 3, stages, 1.2f, kStages64x64) ? kRing32x32
                                                                                                                                : kRing64x64;
  }
  if (tiles(32, 32) <= cus) return kRing32x32;
  if (tiles(32, 64) <= cus) return kRing32x64;
  if (M <= 32 && K >= 2048 && tiles(32, 32) <= 3 * cus) return kRing32x32;
  if (M <= 32 && K <= 512 && 2 * tiles(32, 64) >= 3 * cus && tiles(32, 64) <= 2 * cus) return kRing32x64;
  if (M <= 64 && K % 2048 == 0) return kRing64x64;
  int best = 0;
  float least = 0.f;
  for (int t = 0; t < kRingTiles; ++t) {
    const RingShape& s = kRingShapes[t];
    const long all = tiles(s.rows, s.cols), rest = all % (cus * s.a_cu);
    const float time = (float)(all / (cus * s.a_cu)) * s.full + (rest == 0 ? 0.f : rest <= cus ? s.one : s.full);
    if (t == 0 || time < least) {
      least = time;
      best = t;
    }
  }
  return best;
}

// Whether the ring kernel runs a product of aligned operands: more than 32 rows, or where its tiles beat the kernels of a wave a slice, which read
// the rows of X once for 16 columns.  Its stages cost the same at any number of rows, so the line is lower the more columns there are, and for
// SwiGLU, where a wave of the other kernels holds two weight tiles.  Measured on both sides, us, those kernels / the ring kernel in its best tile:
//   plain, 16 rows and less  8 x 4,096 x 256 2.7 / 3.0, 1 x 12,288 x 256 3.6 / 4.1, 7 x 20,000 x 1,024 10.0 / 10.8, 8 x 6,144 x 4,096 13.8 / 11.5, 16 x 6,144 x 4,096 14.7 /
//                            11.8, 16 x 12,288 x 2,048 15.0 / 12.6, 8 x 151,936 x 1,024 58.9 / 55.3, 7 x 65,536 x 64 6.3 / 4.4, 12 x 12,288 x 392 4.3 / 5.2
//   plain, 17 to 32 rows     17 x 1,536 x 1,024 4.5 / 4.4; rows of weights that are no whole lines of 128 bytes: 31 x 1,536 x 1,272 4.6 / 5.1, 20 x 204 x 1,624 4.7 /
//                            5.6, 24 x 371 x 472 2.9 / 3.7, 20 x 6,144 x 144 2.8 / 3.2, 20 x 768 x 4,384 11.0 / 11.9, 32 x 12,288 x 520 6.7 / 6.4
//   SwiGLU                   6 x 6,144 x 512 4.3 / 4.8, 8 x 2,048 x 1,024 5.3 / 4.9, 16 x 12,288 x 512 6.0 / 5.3, 8 x 1,280 x 912 4.2 / 4.8, 16 x 512 x 408 3.2 / 3.8,
//                            8 x 512 x 2,032 5.9 / 6.8
// float32 multiplies longer than it loads, and a tile's one chain of products is the longer way where few columns leave it alone on its CU: 8 x 2,048
// x 1,024 6.2 / 9.7, 8 x 6,144 x 4,096 25.9 / 30.7, 24 x 2,048 x 1,024 8.1 / 9.7, 24 x 2,048 x 256 4.9 / 4.2, 32 x 4,096 x 4,096 27.6 / 29.8, 16 x
// 8,192 x 2,048 19.2 / 17.4, 32 x 6,144 x 1,024 14.5 / 10.2, SwiGLU 8 x 6,144 x 1,024 10.0 / 11.0, 3 x 1,024 x 256 5.6 / 4.5, 16 x 12,288 x 1,024
// 17.5 / 15.2, 3 x 32,768 x 1,024 29.7 / 33.9.
template <typename T, int EPI>
static bool ring_takes(int M, int N, int K) {
  constexpr bool GATED = EPI == kSwiGLU;
  if (M > 32 || (GATED && M > 16)) return true;
  const bool one_round = (N + 15) / 16 <= compute_units();  // of the other kernels' blocks
  if (sizeof(T) == 4) {
    if (GATED) return N <= 8192 ? K <= 512 : M > 8 || N < 30000;
    if (M <= 16) return M > 8 && !one_round && K >= 256;
    return !one_round || K <= 384;
  }
  const bool lines = K % 64 == 0;  // rows of weights are whole lines
  if (N >= 32768 && M <= 16 && (K <= 128 || M > 8 || (M == 8 && K >= 320))) return true;
  if (GATED) return K >= (!lines && N <= 8192 ? 2600 : M <= 8 ? 640 : 320);
  if (M > 16) return lines || (one_round ? M > 24 && K >= 4096 : K > 256 || N >= 20000);
  if (one_round) return false;
  if (M > 8) return K >= (lines ? 384 : 640);
  const int tile = ring_tile<T>(M, N, K);
  return K >= 640 && (tile == kRing32x32 || tile == kRing32x64);
}

// Whether the ring kernel's 32-bit byte offsets inside a tile reach every operand: the rows of the largest tile, and what
// the last stage reads behind the last row.  (Rows further apart go to the other kernels, which form 64-bit addresses.)
static bool ring_reaches(long ldx, long K, long size) { return (256 * std::max(ldx, K) + 128) * size <= (long)kNothing; }

// Dynamic LDS beyond 64 KB has to be granted per kernel (once).
template <typename T, int EPI, int BM, int BN, int NWM, int NWN, int WS, int XS, int SUB>
static bool ring_lds_ready(int bytes) {
  static const bool granted = [bytes] {
    if (bytes <= 64 * 1024) return true;
    const bool ok = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_ring_kernel<T, EPI, BM, BN, NWM, NWN, WS, XS, SUB>),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess;
    if (!ok) (void)hipGetLastError();
    return ok;
  }();
  return granted;
}

constexpr int kNotLaunched = 1;  // the LDS was refused: the caller has another kernel
constexpr int kMutantNoRing = 16;  // bit of the controls' mask (common.h): that refusal, as a test wants it

// groups: workgroups along K (kSliceSums: out_cols slices each); otherwise 1.
template <typename T, int EPI, int BM, int BN, int NWM, int NWN, int WS, int XS, int SUB = 1>
static int launch_ring_tile(const T* X, const T* W, void* C, int M, int N, int K, long ldx, long ldc, int kslice, int vec_ok,
                            int out_cols, int groups, const float* act, hipStream_t stream) {
  constexpr int kBytes = (WS * BN + XS * BM) * SUB * 128;
  if (LS_MUTANT_HOST(kMutantNoRing) || !ring_lds_ready<T, EPI, BM, BN, NWM, NWN, WS, XS, SUB>(kBytes)) return kNotLaunched;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  hipLaunchKernelGGL((gemm_ring_kernel<T, EPI, BM, BN, NWM, NWN, WS, XS, SUB>), dim3(tiles_m * tiles_n, groups),
                     dim3(64 * NWM * NWN), kBytes, stream, X, W, C, M, N, K, ldx, ldc, kslice, vec_ok, tiles_m, tiles_n,
                     out_cols, act);
  return check_launch("gemm");
}

template <typename T, int EPI>
static int launch_ring(int tile, const T* X, const T* W, void* C, int M, int N, int K, long ldx, long ldc, int kslice,
                       int vec_ok, int out_cols, int groups, const float* act, hipStream_t stream) {
#define LS_RING(...) \
  return launch_ring_tile<T, EPI, __VA_ARGS__>(X, W, C, M, N, K, ldx, ldc, kslice, vec_ok, out_cols, groups, act, stream)
  if constexpr (sizeof(T) == 4) {
    if constexpr (EPI != kSliceSums)
      if (tile == kRing32x32) LS_RING(32, 32, 2, 2, 5, 5);
    LS_RING(64, 64, 2, 2, 3, 3);
  } else if constexpr (EPI == kSliceSums) {
    if (tile == kRing32x64) LS_RING(32, 64, 2, 2, 5, 5);
    LS_RING(64, 64, 4, 2, 5, 5);
  } else {
    switch (tile) {
      case kRing256x192: LS_RING(256, 192, 4, 2, 3, 2);
      case kRing256x128: LS_RING(256, 128, 4, 2, 3, 3);
      case kRing192x192: LS_RING(192, 192, 4, 2, 3, 3);
      case kRing128x192: LS_RING(128, 192, 4, 2, 3, 3);
      case kRing192x128: LS_RING(192, 128, 4, 2, 4, 4);
      case kRing128x128: LS_RING(128, 128, 4, 2, 4, 4);
      case kRing128x64: LS_RING(128, 64, 4, 2, 5, 5);
      case kRing64x128: LS_RING(64, 128, 2, 4, 3, 3);
      case kRing32x64: LS_RING(32, 64, 2, 2, 5, 5);
      case kRing32x32: LS_RING(32, 32, 2, 2, 5, 5, 2);
      default: LS_RING(64, 64, 4, 2, 5, 5);
    }
  }
#undef LS_RING
}

// Columns of the streaming kernel's blocks: 12 where the walks have no more rounds with those than with 16, else 16 (a round costs its
// barrier, its fold and a fragment's instructions whatever its columns).  Weights from HBM, blocks of 16 / 12, us.  The same rounds, two or three:
// 8 rows 4,608 x 4,096 16.0 / 14.4, 5,120 x 4,096 16.2 / 14.6, 6,144 x 4,096 16.7 / 15.2, 9,216 x 4,096 22.8 / 21.0, 1 row 6,144 x 4,096 15.3 / 13.9,
// 6,144 x 5,120 23.5 / 22.7, 9,216 x 2,048 14.3 / 12.6, 16 rows 6,144 x 4,096 18.3 / 16.9, 40 rows 3,072 x 4,096 19.8 / 18.2, float32 1 row
// 5,120 x 4,096 31.9 / 30.9.  A round more: 1 row 7,168 x 4,096 15.8 / 18.5, 10,240 21.8 / 24.0, 18,432 34.5 / 36.3, 151,936 232 / 272, 40 rows 5,056
// 24.5 / 27.8.  Blocks of 8 never won (1 row 6,144 16.8, 14,336 36.0 for 28.0).  SwiGLU keeps its pairs of 16.
static int stream_columns(int N, int walkers) {
  auto rounds = [&](int cols) { return ((N + cols - 1) / cols + walkers - 1) / walkers; };
  return rounds(12) <= rounds(16) ? 12 : 16;
}

template <typename T, int EPI>
int launch_gemm(const void* X, const void* W, void* C, int M, int N, int K, long ldx, long ldc, const float* norm_w,
                float eps, int out_cols, hipStream_t stream, const float* act = nullptr) {
  int kslice = kslice_for(K);
  if (LS_MUTANT_HOST(kMutantKsliceByRows) && M > 16 && M <= 64) kslice *= 2;  // the mutant: K blocking that depends on the rows of the launch
  const int nslices = (K + kslice - 1) / kslice;
  constexpr int VEC = Atom<T>::VEC;
  constexpr int NT = (EPI == kSwiGLU) ? 2 : 1;
  const int aligned = (K % VEC == 0) && (norm_w || ldx % VEC == 0) && (reinterpret_cast<uintptr_t>(X) % 16 == 0) &&
                      (reinterpret_cast<uintptr_t>(W) % 16 == 0);
  const size_t out_size = (EPI == kStore || EPI == kSwiGLU || EPI == kXielu) ? sizeof(T) : sizeof(float);
  const int vec_ok = (ldc % 4 == 0) && (reinterpret_cast<uintptr_t>(C) % (4 * out_size) == 0);
  const bool whole = aligned && pieces_reach(ldx, K, sizeof(T));
  const T* w = reinterpret_cast<const T*>(W);
  if (norm_w && M > 16) return fail("gemm: the fused norm prologue takes at most 16 rows, got %d", M);
  const int mt_rows = (M + 15) / 16;
  const int col_blocks = (N + 16 * NT - 1) / (16 * NT);
  bool ring = aligned && ring_reaches(ldx, K, sizeof(T));
  if (!norm_w && ring && ring_takes<T, EPI>(M, N, K)) {
    const int rc = launch_ring<T, EPI>(ring_tile<T>(M, N, K), reinterpret_cast<const T*>(X), w, C, M, N, K, ldx, ldc, kslice, vec_ok,
                                       out_cols, 1, act, stream);
    if (rc != kNotLaunched) return rc;
    ring = false;
  }
  // What the ring kernel cannot take goes to the tiled kernel from 33 rows on (SwiGLU from 17) where its tiles give every CU a
  // workgroup, and from 17 on over the most columns (operands off 16 bytes, the kernels of a wave a slice / tiles, us: 17 x
  // 32,800 x 1,024 151 / 87, 64 x 32,800 x 1,024 336 / 111).
  const bool tiles = !ring && ((N + 63) / 64 >= compute_units() && (M > 32 || (M > 16 && EPI == kSwiGLU)));
  const int xc = kslice / Atom<T>::KCHUNK;  // chunks per slice
  // The streaming kernel where a workgroup would get more than one column block: a CU holds 16 waves
  // of it (one per K slice), so 16 / nslices workgroups.
  const int stream_wgs = compute_units() * (16 / nslices > 0 ? 16 / nslices : 1);
  // up to 32 rows one group of rows; up to 64 two groups of 32 that share the weights through L2
  const int row_groups = mt_rows <= 2 ? 1 : 2;
  const int group_tiles = mt_rows <= 2 ? mt_rows : 2;
  const size_t stream_lds = 2 * (size_t)nslices * NT * group_tiles * 256 * sizeof(float);  // two sets of slice sums
  // (with fewer than eight slices the skinny kernel's small workgroups, several a CU, do as well or better)
  if (!norm_w && mt_rows <= 4 && !tiles && xc % 4 == 0 && xc * group_tiles <= 16 && nslices >= 8 && nslices <= 16 &&
      col_blocks * row_groups > stream_wgs && stream_lds <= 128 * 1024 && LS_GEMM_STREAM) {
    int walkers = stream_wgs / row_groups;
    const int cols = NT == 2 ? 16 : stream_columns(N, walkers);
    const int blocks = NT == 2 ? col_blocks : (N + cols - 1) / cols;
    const int rounds = (blocks + walkers - 1) / walkers;
    walkers = (blocks + rounds - 1) / rounds;
    if (row_groups > 1) walkers = (walkers + 7) / 8 * 8;  // whole rounds of the XCDs, see the kernel
    dim3 grid(walkers * row_groups);
    bool launched = true;
#define LS_STREAM_AS(MT_, XC_, WHOLE_)                                                                             \
  if (stream_lds_ready<T, MT_, EPI, XC_, WHOLE_>(stream_lds))                                                      \
    hipLaunchKernelGGL((gemm_stream_kernel<T, MT_, EPI, XC_, WHOLE_>), grid, dim3(nslices * 64), stream_lds, stream, \
                       reinterpret_cast<const T*>(X), w, C, M, N, K, ldx, ldc, kslice, aligned, vec_ok, out_cols,  \
                       blocks, row_groups, cols, act);                                                             \
  else                                                                                                             \
    launched = false
#define LS_STREAM(MT_, XC_) \
  if (whole) { LS_STREAM_AS(MT_, XC_, true); } else { LS_STREAM_AS(MT_, XC_, false); }
    if (group_tiles == 1 && xc == 8) {
      LS_STREAM(1, 8)
    } else if (group_tiles == 1 && xc == 16) {
      LS_STREAM(1, 16)
    } else if (group_tiles == 2 && xc == 8) {
      LS_STREAM(2, 8)
    } else {
      launched = false;
    }
#undef LS_STREAM
#undef LS_STREAM_AS
    if (launched) return check_launch("gemm");
  }
  if (M <= 64 && !tiles && (ring || M <= 16 || N < 32768)) {
    const int mt = (M + 15) / 16;
    // 16 waves leave 128 registers a lane: only for one or two row tiles
    const int nw = (nslices > 8 && mt * NT <= 2) ? 16 : (nslices > 4 ? 8 : 4);
    dim3 grid((N + 16 * NT - 1) / (16 * NT));
    const size_t lds = ((size_t)nslices * NT * mt * 256 + (norm_w ? 80 : 0)) * sizeof(float);
#define LS_SKINNY_AS(MT_, NW_, NORM_, WHOLE_)                                                                    \
  hipLaunchKernelGGL((gemm_skinny_kernel<T, MT_, NW_, EPI, NORM_, WHOLE_>), grid, dim3(NW_ * 64), lds, stream, X, w, C, \
                     M, N, K, ldx, ldc, kslice, aligned, vec_ok, norm_w, eps, out_cols, act)
#define LS_SKINNY(MT_, NW_) \
  if (whole) LS_SKINNY_AS(MT_, NW_, false, true); else LS_SKINNY_AS(MT_, NW_, false, false)
    if (norm_w) {
      if constexpr (EPI == kXielu) return fail("gemm: the xIELU epilogue has no norm prologue");
      else if (nw >= 8) LS_SKINNY_AS(1, 8, true, false);
      else LS_SKINNY_AS(1, 4, true, false);
    } else if (nw == 16) {
      if (mt == 1) { LS_SKINNY(1, 16); } else { LS_SKINNY(2, 16); }
    } else if (nw == 8) {
      if (mt == 1) { LS_SKINNY(1, 8); } else if (mt == 2) { LS_SKINNY(2, 8); }
      else if (mt == 3) { LS_SKINNY(3, 8); } else { LS_SKINNY(4, 8); }
    } else {
      if (mt == 1) { LS_SKINNY(1, 4); } else if (mt == 2) { LS_SKINNY(2, 4); }
      else if (mt == 3) { LS_SKINNY(3, 4); } else { LS_SKINNY(4, 4); }
    }
#undef LS_SKINNY
#undef LS_SKINNY_AS
  } else {
    const int tiles_m = (M + 63) / 64, tiles_n = (N + 63) / 64;
    hipLaunchKernelGGL((gemm_tiled_kernel<T, EPI>), dim3(tiles_m * tiles_n), dim3(256), 0, stream,
                       reinterpret_cast<const T*>(X), w, C, M, N, K, ldx, ldc, kslice, vec_ok, tiles_m, tiles_n, out_cols, act);
  }
  return check_launch("gemm");
}

}  // namespace ls

// dtype: 0 float32, 1 bfloat16.  epilogue: 0 store in dtype, 1 store float,
// 2 add to float, 3 SwiGLU of interleaved gate/up tiles (N = rows of W, the
// output has out_cols <= N/2 columns; rows of W beyond them are padding).  X [M,K] with ldx elements per row, W [N,K]
// contiguous, C with ldc elements per row.  With norm_w (float [K]) X is the
// float residual stream and is RMS-normalised on the fly (M <= 16).
extern "C" int ls_gemm(int dtype, int epilogue, const void* X, const void* W, void* C, int M, int N, int K, long ldx,
                       long ldc, const float* norm_w, float eps, int out_cols, void* stream) {
  using namespace ls;
  LS_REQUIRE(M > 0 && N > 0 && K > 0, "gemm: sizes must be positive, got M=%d N=%d K=%d", M, N, K);
  if (epilogue != kSwiGLU) out_cols = N;
  LS_REQUIRE(out_cols > 0 && (epilogue != kSwiGLU || (out_cols <= N / 2 && out_cols > N / 2 - 16)),
             "gemm: %d output columns do not fit %d interleaved weight rows", out_cols, N);
  LS_REQUIRE(ldx >= K && ldc >= out_cols, "gemm: row strides ldx=%ld ldc=%ld are shorter than K=%d / %d columns", ldx,
             ldc, K, out_cols);
  LS_REQUIRE(epilogue != kSwiGLU || N % 32 == 0, "gemm: the SwiGLU epilogue needs interleaved tiles, N=%d", N);
  LS_REQUIRE(X && W && C, "gemm: null operand");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
#define LS_GEMM_CASE(T_)                                                                              \
  switch (epilogue) {                                                                                 \
    case kStore: return launch_gemm<T_, kStore>(X, W, C, M, N, K, ldx, ldc, norm_w, eps, out_cols, s);          \
    case kStoreF32: return launch_gemm<T_, kStoreF32>(X, W, C, M, N, K, ldx, ldc, norm_w, eps, out_cols, s);    \
    case kAddF32: return launch_gemm<T_, kAddF32>(X, W, C, M, N, K, ldx, ldc, norm_w, eps, out_cols, s);        \
    case kSwiGLU: return launch_gemm<T_, kSwiGLU>(X, W, C, M, N, K, ldx, ldc, norm_w, eps, out_cols, s);        \
    default: return fail("gemm: unknown epilogue %d", epilogue);                                      \
  }
  if (dtype == kF32) { LS_GEMM_CASE(float) }
  if (dtype == kBF16) { LS_GEMM_CASE(bf16_t) }
#undef LS_GEMM_CASE
  return fail("gemm: unknown dtype %d", dtype);
}

// C [M][N] (dtype) = xielu(X @ W^T), elementwise: act[0] z^2 + z/2 for z > 0, act[1] (e^z - 1 - z) + z/2 elsewhere;
// act: two floats on the device.  Operands as for ls_gemm.
extern "C" int ls_gemm_xielu(int dtype, const void* X, const void* W, void* C, int M, int N, int K, long ldx, long ldc,
                             const float* act, void* stream) {
  using namespace ls;
  LS_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_xielu: sizes must be positive, got M=%d N=%d K=%d", M, N, K);
  LS_REQUIRE(ldx >= K && ldc >= N, "gemm_xielu: row strides ldx=%ld ldc=%ld are shorter than K=%d / N=%d", ldx, ldc, K, N);
  LS_REQUIRE(X && W && C && act, "gemm_xielu: null operand");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (dtype == kF32) return launch_gemm<float, kXielu>(X, W, C, M, N, K, ldx, ldc, nullptr, 0.f, N, s, act);
  if (dtype == kBF16) return launch_gemm<bf16_t, kXielu>(X, W, C, M, N, K, ldx, ldc, nullptr, 0.f, N, s, act);
  return fail("gemm_xielu: unknown dtype %d", dtype);
}

extern "C" int ls_gemm_kslice(int K) { return ls::kslice_for(K); }

// The tile (enum RingTile) in which ls_gemm has the ring kernel compute a product of aligned operands; -1: another kernel does.
extern "C" int ls_gemm_ring_tile(int dtype, int epilogue, int M, int N, int K) {
  using namespace ls;
#define LS_TAKES(T_) (epilogue == kSwiGLU ? ring_takes<T_, kSwiGLU>(M, N, K) : ring_takes<T_, kStore>(M, N, K))
  if (dtype == kF32) return LS_TAKES(float) ? ring_tile<float>(M, N, K) : -1;
  return LS_TAKES(bf16_t) ? ring_tile<bf16_t>(M, N, K) : -1;
#undef LS_TAKES
}

// Columns of a block of the streaming kernel for N columns and that many walkers (workgroups of a group of rows).
extern "C" int ls_gemm_stream_columns(int N, int walkers) { return ls::stream_columns(N, walkers); }

// Number of K slices of a product over K (the first dimension of the partial sums of ls_gemm_slices).
extern "C" int ls_gemm_slices_count(int K) {
  const int kslice = ls::kslice_for(K);
  return (K + kslice - 1) / kslice;
}

// Rows that ls_gemm_slices takes for a product over K: 64 always; 256 where the kernel that keeps
// its rows of X in registers has an instance for the slice length (more rows are further groups of
// workgroups that walk the same weights).
extern "C" int ls_gemm_slices_max_rows(int dtype, int K) {
  const int xc = ls::kslice_for(K) / (dtype == ls::kF32 ? 16 : 32);
  return (LS_GEMM_STREAM && (xc == 8 || xc == 16)) ? 256 : 64;
}

namespace ls {

// The ring kernel's tile for slice sums and the slices a workgroup takes; per 0: another kernel.
struct SlicesPlan {
  int tile, per;
};
// The products a CU (in 256) from which slice sums of bfloat16 come from tiles: what a wave a slice does instead grows with the rows that every
// block of 16 columns reads again, a tile's time hardly.  Measured over 10,655 sizes (us, a wave a slice / tiles): fewer products for rows of weights
// that are whole lines of 128 bytes (17 x 1,408 x 3,072 6.9 / 5.1, 16 x 1,792 x 3,328 6.2 / 5.5, 8 x 4,096 x 2,560 6.5 / 7.6, 32 x 1,280 x 1,280 3.6 / 4.0, 256 x 512 x 512
// 3.3 / 3.9; no whole lines 10 x 6,784 x 1,128 6.0 / 7.9, 48 x 5,120 x 1,576 16.3 / 8.6); under eight rows, which cost little to read again, many more (6 x
// 6,656 x 2,304 8.2 / 10.2), but for long slices (4 x 4,096 x 12,288 24.0 / 21.8) and rows of weights a multiple of 4 KB apart, sixteen of which
// meet in few memory channels (4 x 4,096 x 4,096 9.7 / 8.3).  One row never (5,120 x 8,192 19.8 / 20.4).
static long slices_line(int M, int K) {
  if (K > 4096) return M < 8 ? 50 : 72;  // slices of more than 256
  if (M < 8) return K % 2048 == 0 ? 56 : 180;
  return K % 64 == 0 ? (M <= 16 ? 80 : 64) : (M <= 16 ? 100 : 88);
}
// The cheapest of the tiles and of one, two or four slices a workgroup by rounds_cost.  (us)
// float32, from 33 rows on: 64 x 64 tiles, from nine workgroups for sixteen CUs on (48 x 1,024 x 2,048, eight, 7.1 by a wave a slice / 8.6), eight or
// sixteen stages a workgroup (33 x 4,096 x 4,096 24.9 / 22.1, 160 x 10,240 x 768 31.7 / 36.4, 200 x 5,120 x 1,024 27.4 / 30.4); slices of sixteen
// stages by themselves (56 x 8,192 x 8,192 83, two of them 98).
// bfloat16, from 4 rows on: 32 x 64 or 64 x 64 tiles, two a CU, beyond slices_line.  Sixteen stages a workgroup at most, eight with more than 64
// rows, and beyond 32 rows slices of eight and more by themselves (128 x 5,120 x 5,120 with one, two and four 27.6, 29.5, 30.7; 64 x 10,240 x 5,120 31.3, 33.6, 34.9).
// Up to 32 rows also two longer slices, where that is one nearly full round of one or of two a CU (one slice a workgroup / two: 8 x 1,280 x 14,472
// 13.8 / 12.5, 6 x 1,472 x 9,576 10.9 / 9.9, 8 x 4,096 x 12,288 23.1 / 22.1), unless both the rows of weights and the workgroups' first columns lie a
// multiple of 4 KB apart, so that all ask the same memory channels at once (18 x 2,240 x 14,336 14.2 / 17.0).
static SlicesPlan slices_plan(int dtype, int M, int N, int K) {
  const int kslice = kslice_for(K), nslices = (K + kslice - 1) / kslice;
  const long cus = compute_units();
  const bool f32 = dtype == kF32;
  SlicesPlan best{kRing64x64, 0};
  if (f32 ? M < 33 : M < 4 || (long)((N + 15) / 16) * std::max(K, 256) * M <= slices_line(M, K) * 256 * cus) return best;
  constexpr float k32x64[2] = {0.18f, 0.39f}, k64x64[2] = {0.33f, 0.52f};
  const int most = f32 || M > 64 || (M > 32 && kslice > 256) ? 512 : 1024;  // elements of K a workgroup
  float least = 0.f;
  for (int rows = f32 ? 64 : 32; rows <= 64; rows += 32)
    for (int per = 1; per == 1 || (per <= 4 && per <= nslices); per *= 2) {
      const long all = (long)((M + rows - 1) / rows) * ((N + 63) / 64) * ((nslices + per - 1) / per);
      const int stages = std::min(per, nslices) * (kslice / (f32 ? 32 : 64));
      const bool one_round = per == 2 && M <= 32 && ((16 * all > 9 * cus && all <= cus) || (16 * all > 30 * cus && all <= 2 * cus));
      if (per > 1 && per * kslice > most && !(one_round && (K % 2048 || per * kslice % 2048))) continue;
      if (f32 && 16 * all < 9 * cus) continue;
      const float cost = f32 ? rounds_cost(all, 3, stages, 1.2f, kStages64x64) : rounds_cost(all, 2, stages, 1.5f, rows == 32 ? k32x64 : k64x64);
      if (best.per == 0 || cost < least) {
        least = cost;
        best = {rows == 32 ? kRing32x64 : kRing64x64, per};
      }
    }
  return best;
}

}  // namespace ls

// How ls_gemm_slices computes the sums of aligned operands: rows of the ring kernel's tile times 16 plus slices a workgroup; 0: another kernel.
extern "C" int ls_gemm_slices_plan(int dtype, int M, int N, int K) {
  using namespace ls;
  const SlicesPlan plan = N % 4 == 0 ? slices_plan(dtype, M, N, K) : SlicesPlan{kRing64x64, 0};
  return plan.per == 0 ? 0 : (plan.tile == kRing32x64 ? 32 : 64) * 16 + plan.per;
}

// Slice sums of X [M,K] @ W [N,K]^T for M <= ls_gemm_slices_max_rows: P [slices][M][N] float, P[s] = the
// sum over K slice s.  The product is P[0] + P[1] + ... added in this order, starting from +0.
extern "C" int ls_gemm_slices(int dtype, const void* X, const void* W, float* P, int M, int N, int K, long ldx,
                              void* stream) {
  using namespace ls;
  LS_REQUIRE(M > 0 && M <= ls_gemm_slices_max_rows(dtype, K) && N > 0 && K > 0,
             "gemm_slices: takes 1 to %d rows with K=%d, got M=%d N=%d", ls_gemm_slices_max_rows(dtype, K), K, M, N);
  LS_REQUIRE(ldx >= K && X && W && P, "gemm_slices: bad operands");
  LS_REQUIRE(reinterpret_cast<uintptr_t>(P) % 16 == 0, "gemm_slices: the partial sums must be 16-byte aligned");
  const int kslice = kslice_for(K);
  const int nslices = (K + kslice - 1) / kslice;
  const int col_blocks = (N + 15) / 16;
  // enough groups of slices to fill the GPU, at most four slices (waves) a workgroup
  int groups = (compute_units() + col_blocks - 1) / col_blocks;
  if (groups > nslices) groups = nslices;
  if (groups < (nslices + 3) / 4) groups = (nslices + 3) / 4;
  const int per_group = (nslices + groups - 1) / groups;
  groups = (nslices + per_group - 1) / per_group;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  dim3 grid(col_blocks, groups);
  const int vec = dtype == kF32 ? 4 : 8;
  const int aligned = (K % vec == 0) && (ldx % vec == 0) && (reinterpret_cast<uintptr_t>(X) % 16 == 0) &&
                      (reinterpret_cast<uintptr_t>(W) % 16 == 0);
  const bool whole = aligned && pieces_reach(ldx, K, dtype == kF32 ? 4 : 2);
  const int mt = (M + 15) / 16;
  // With more than 16 rows, where the rows of X outweigh the weights of a column block, and at least four
  // workgroups a CU, workgroups walk two or more column blocks each with X in registers (the walk keeps
  // two workgroups a CU).  Up to 16 rows the walk measured no faster: fewer waves, less in flight.
  const int xc = kslice / (dtype == kF32 ? 16 : 32);  // 64-byte chunks per slice
  // row tiles a workgroup holds in registers (xs: 4 * xc registers a tile); more rows go to further groups
  // (24 chunks a slice with two tiles need 268 registers: one wave a SIMD, measured slower than the plain kernel)
  const int group_tiles = xc <= 8 ? std::min(mt, 4) : (xc <= 16 ? std::min(mt, 2) : 0);
  const int row_groups = group_tiles > 0 ? (mt + group_tiles - 1) / group_tiles : 0;
  int rounds =
      (int)std::min<long>(4, (long)col_blocks * groups * std::max(row_groups, 1) / (2L * compute_units()));
  if (mt > 4 && rounds < 1) rounds = 1;  // more than 64 rows: this kernel only, if with one column block a workgroup
  // The ring kernel, with four stages of both operands in flight, where slices_plan finds its tiles the better ones.
  if (LS_GEMM_SLICES_TILED && aligned && ring_reaches(ldx, K, dtype == kF32 ? 4 : 2) && N % 4 == 0 && (dtype == kF32 || dtype == kBF16)) {
    const SlicesPlan plan = slices_plan(dtype, M, N, K);
    if (plan.per > 0) {
      const int groups_y = (nslices + plan.per - 1) / plan.per;
      const int rc = dtype == kF32 ? launch_ring<float, kSliceSums>(plan.tile, (const float*)X, (const float*)W, P, M, N, K, ldx, N,
                                                                    kslice, 1, plan.per, groups_y, nullptr, s)
                                   : launch_ring<bf16_t, kSliceSums>(plan.tile, (const bf16_t*)X, (const bf16_t*)W, P, M, N, K, ldx,
                                                                     N, kslice, 1, plan.per, groups_y, nullptr, s);
      if (rc != kNotLaunched) return rc;
    }
  }
  // More than 16 rows and enough columns that workgroups of 64 columns fill the GPU: the wide kernel.
  {
    const int wide_blocks = (N + 63) / 64;
    const int wide_per_group = std::min(4, nslices);
    const int wide_groups = (nslices + wide_per_group - 1) / wide_per_group;
    if (mt >= 2 && mt <= 4 && (long)wide_blocks * wide_groups >= LS_GEMM_SLICES_WIDE_WGS && xc % LS_GEMM_SLICES_WIDE_UNR == 0 &&
        LS_GEMM_SLICES_WIDE) {
      dim3 wide_grid(wide_blocks, wide_groups);
#define LS_WIDE(T_, MT_)                                                                                          \
  hipLaunchKernelGGL((gemm_slices_wide_kernel<T_, MT_, 4, LS_GEMM_SLICES_WIDE_UNR>), wide_grid,                 \
                     dim3(64 * wide_per_group), 0, s, (const T_*)X, (const T_*)W, P, M, N, K, ldx, kslice, aligned, \
                     wide_per_group)
#define LS_WIDE_MT(T_)                                       \
  if (mt == 2) LS_WIDE(T_, 2); else if (mt == 3) LS_WIDE(T_, 3); else LS_WIDE(T_, 4)
      if (dtype == kF32) { LS_WIDE_MT(float); } else if (dtype == kBF16) { LS_WIDE_MT(bf16_t); } else return fail("gemm_slices: unknown dtype %d", dtype);
#undef LS_WIDE_MT
#undef LS_WIDE
      return check_launch("gemm_slices");
    }
  }
  if ((rounds >= 2 || mt > 4) && mt >= 2 && group_tiles > 0 && xc % 4 == 0 && LS_GEMM_STREAM) {
    int walkers = (col_blocks + rounds - 1) / rounds;
    if (row_groups > 1) walkers = (walkers + 7) / 8 * 8;  // the groups' workgroups of a walk sit on the same XCD
    dim3 walk_grid(walkers, groups, row_groups);
    bool launched = true;
#define LS_WALK_AS(T_, MT_, XC_, WHOLE_)                                                                           \
  hipLaunchKernelGGL((gemm_slices_stream_kernel<T_, MT_, XC_, WHOLE_>), walk_grid, dim3(64 * per_group), 0, s, (const T_*)X, \
                     (const T_*)W, P, M, N, K, ldx, kslice, aligned, per_group, col_blocks)
#define LS_WALK(T_, MT_, XC_) \
  { if (whole) LS_WALK_AS(T_, MT_, XC_, true); else LS_WALK_AS(T_, MT_, XC_, false); }
#define LS_WALK_T(T_)                                                          \
  if (group_tiles == 2 && xc == 8) LS_WALK(T_, 2, 8)                           \
  else if (group_tiles == 3 && xc == 8) LS_WALK(T_, 3, 8)                      \
  else if (group_tiles == 4 && xc == 8) LS_WALK(T_, 4, 8)                      \
  else if (group_tiles == 2 && xc == 16) LS_WALK(T_, 2, 16)                    \
  else launched = false
    if (dtype == kF32) { LS_WALK_T(float); } else if (dtype == kBF16) { LS_WALK_T(bf16_t); } else launched = false;
#undef LS_WALK_T
#undef LS_WALK
#undef LS_WALK_AS
    if (launched) return check_launch("gemm_slices");
  }
  LS_REQUIRE(mt <= 4, "gemm_slices: no kernel for %d rows with K=%d", M, K);
#define LS_SLICES_AS(T_, MT_, WHOLE_)                                                                            \
  hipLaunchKernelGGL((gemm_slices_kernel<T_, MT_, WHOLE_>), grid, dim3(64 * per_group), 0, s, (const T_*)X,       \
                     (const T_*)W, P, M, N, K, ldx, kslice, aligned, per_group)
#define LS_SLICES(T_, MT_) \
  { if (whole) LS_SLICES_AS(T_, MT_, true); else LS_SLICES_AS(T_, MT_, false); }
#define LS_SLICES_MT(T_)                                              \
  if (mt == 1) LS_SLICES(T_, 1) else if (mt == 2) LS_SLICES(T_, 2)   \
  else if (mt == 3) LS_SLICES(T_, 3) else LS_SLICES(T_, 4)
  if (dtype == kF32) {
    LS_SLICES_MT(float);
  } else if (dtype == kBF16) {
    LS_SLICES_MT(bf16_t);
  } else {
    return fail("gemm_slices: unknown dtype %d", dtype);
  }
#undef LS_SLICES_MT
#undef LS_SLICES
#undef LS_SLICES_AS
  return check_launch("gemm_slices");
}

// Whether ls_gemm_slices_folded takes this product: at most 16 rows, whole heads of a size that is a
// multiple of four, K a multiple of the load width, at most 32 splits, the folded rows of a slice within
// 64 KB of LDS -- and not so many rows over large weights (eight over 64 MB) that a fold of its own and the ring kernel's
// slice sums are ahead.
extern "C" int ls_gemm_slices_folded_ok(int dtype, int M, int N, int K, int head_dim, int splits) {
  using namespace ls;
  if (dtype != kF32 && dtype != kBF16) return 0;
  if (M < 1 || M > 16 || N < 1 || K < 1 || head_dim < 4 || head_dim % 4 || K % head_dim) return 0;
  if (splits < 1 || splits > 32 || K % (dtype == kF32 ? 4 : 8)) return 0;
  const long weight_bytes = (long)N * K * (dtype == kF32 ? 4 : 2);
  const int ring_better_from = dtype == kF32 ? 33 : (weight_bytes >= (64L << 20) ? 8 : 17);
  if (LS_GEMM_SLICES_TILED && M >= ring_better_from && N % 4 == 0) return 0;
  const size_t element = dtype == kF32 ? 4 : 2;
  return (size_t)M * (kslice_for(K) + 16 / element) * element <= 64 * 1024;
}

// ls_gemm_slices for an operand that is still `splits` per-split sums a (token, head) of an attention
// launch over single decoded tokens (see gemm_slices_folded_kernel): part_acc [(M * heads) * splits][head_dim],
// part_ml [(M * heads) * splits][2], heads = K / head_dim.  P as ls_gemm_slices leaves it, bit for bit what
// it leaves for the folded and rounded operand.
extern "C" int ls_gemm_slices_folded(int dtype, const float* part_acc, const float* part_ml, int splits, int head_dim,
                                     const void* W, float* P, int M, int N, int K, void* stream) {
  using namespace ls;
  LS_REQUIRE(ls_gemm_slices_folded_ok(dtype, M, N, K, head_dim, splits),
             "gemm_slices_folded: not for M=%d N=%d K=%d head_dim=%d splits=%d (see ls_gemm_slices_folded_ok)", M, N, K,
             head_dim, splits);
  LS_REQUIRE(part_acc && part_ml && W && P, "gemm_slices_folded: null operand");
  LS_REQUIRE(reinterpret_cast<uintptr_t>(P) % 16 == 0 && reinterpret_cast<uintptr_t>(W) % 16 == 0 &&
                 reinterpret_cast<uintptr_t>(part_acc) % 16 == 0 && reinterpret_cast<uintptr_t>(part_ml) % 8 == 0,
             "gemm_slices_folded: operands must be 16-byte aligned");
  const int kslice = kslice_for(K);
  const int nslices = (K + kslice - 1) / kslice;
  const size_t element = dtype == kF32 ? 4 : 2;
  const size_t lds = (size_t)M * (kslice + 16 / element) * element;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  dim3 grid((N + 63) / 64, nslices);
#define LS_FOLDED_N(T_, REV_, UNITS_, SPLITS_)                                                                       \
  hipLaunchKernelGGL((gemm_slices_folded_kernel<T_, REV_, UNITS_, SPLITS_>), grid, dim3(256), lds, s, part_acc, part_ml, \
                     splits, head_dim, (const T_*)W, P, M, N, K, kslice)
  // units of a thread whose sums are in flight together: all of them up to four
  const int mine = (M * (kslice / 4) + 255) / 256;
#define LS_FOLDED_S(T_, REV_, SPLITS_)                       \
  if (mine <= 1) LS_FOLDED_N(T_, REV_, 1, SPLITS_);          \
  else if (mine <= 2) LS_FOLDED_N(T_, REV_, 2, SPLITS_);     \
  else LS_FOLDED_N(T_, REV_, 4, SPLITS_)
#define LS_FOLDED(T_, REV_)                                  \
  if (splits <= 4) { LS_FOLDED_S(T_, REV_, 4); }             \
  else if (splits <= 8) { LS_FOLDED_S(T_, REV_, 8); }        \
  else LS_FOLDED_N(T_, REV_, 1, 32)
#ifdef LS_MUTANTS
  if (LS_MUTANT_HOST(kMutantReversedFoldInProduct)) {
    if (dtype == kF32) { LS_FOLDED(float, true); } else { LS_FOLDED(bf16_t, true); }
    return check_launch("gemm_slices_folded");
  }
#endif
  if (dtype == kF32) { LS_FOLDED(float, false); } else { LS_FOLDED(bf16_t, false); }
#undef LS_FOLDED_S
#undef LS_FOLDED_N
#undef LS_FOLDED
  return check_launch("gemm_slices_folded");
}
