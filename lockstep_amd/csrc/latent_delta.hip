// More kernels of the mixers library: a residual stream of several copies that every sublayer reads
// as one weighted sum and writes back through a small mixing matrix (with the norm of the next reader
// fused in), the passes around attention over a cached latent (norms of the latents, rotation of the
// shared key part, queries brought into the latent's space by a product a head), and the gated delta
// rule with its short convolutions.
//
// Everything here is computed in float whatever the compute dtype T is: T is the type of what a
// matrix product reads next (and of the cache).  Per-row reductions have an order fixed by the row's
// sizes alone; the recurrence walks a request's tokens in order, so nothing depends on how the
// request was cut into steps or on what else is in the batch.

#include "common.h"
#include "ring.h"
#include "row_piece.h"
#include "mixers_api.h"

namespace ls {

struct SeqMeta {  // one per sequence of the step (all int32), as the step's upload lays it out
  int q_off;      // first packed row
  int q_len;      // rows in this step
  int q_start;    // absolute position of the first row
  int kv_len;     // q_start + q_len
  int table_row;  // row of the block table, and the request's state slot
  int reserved[3];
};

__device__ __forceinline__ float sigmoid_f(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float silu_f(float x) { return x * sigmoid_f(x); }
__device__ __forceinline__ float softplus_f(float x) { return x > 20.0f ? x : log1pf(expf(x)); }

// The four wave sums of a workgroup of 256 threads added in wave order; every thread gets the total.
__device__ __forceinline__ float block_sum4(float v, float* scratch) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) scratch[w] = v;
  __syncthreads();
  return ((scratch[0] + scratch[1]) + scratch[2]) + scratch[3];
}

// ---------------------------------------------------------------------------
// A residual stream of n copies X [rows][n][W] (float).  One launch does, for a row, either or both of
//   write:  y = P[0][row] + P[1][row] + ... (slices ascending, from +0: the sublayer's output, left as slice sums);
//           X'_t = sum_s mix[s][t] X_s + gain[t] y      for all t at once from the old copies
//   read:   u = sum_t take[t] X'_t   (take == null: the plain sum of the copies)
//           out = (u - m) / sqrt(mean((u - m)^2) + eps) * weight + bias     (T; m the row's mean if `centred`, else 0; bias
//           may be null)
// Thread t of 256 owns the elements 1024 c + 4 t + {0..3}, c ascending; the sum of squares adds them in that order, then
// a butterfly over the wave and the wave sums in wave order.  `row` = rows[r] when a row list is given.
// ---------------------------------------------------------------------------
constexpr int kMaxStreams = 8;
constexpr int kStreamChunks = 12;  // a row of up to 1024 * kStreamChunks elements keeps what it read in LDS

__device__ __forceinline__ f32x4 load4(const float* __restrict__ p, int e, int W, bool vec_ok) {
  if (vec_ok) return *reinterpret_cast<const f32x4*>(p + e);
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (e + i < W) v[i] = p[e + i];
  return v;
}

// (N, the number of copies, is a template parameter: every copy's load stands in straight-line code, so all of a
// thread's loads are on their way before the first is used.)  What bounds it at few rows is the chain of answers from memory, so a
// thread's first run of four elements, the slices' sums, the mixing factors and the weights are asked for together, in front of the
// first barrier, and what a run was read as stays in registers: requests of one token through four copies of 1,024 (28 layers,
// all kernels) 2,633 -> 2,574 us a step.  At many rows it is memory, and how many rows a CU has in flight: ONE, rows of up to
// 1,024 elements, one run a thread, without the registers of further runs (2,048 rows, one slice, four copies of 1,024 elements 16.3 ->
// 14.6 us, eight of 512 22.6 -> 18.6); and where seven or eight copies of longer rows are in registers, their first run is not
// asked for in front of the barrier, and the registers are held to what three rows a CU need (seven of 2,048 43.4 -> 41.4, eight
// 49.2 -> 48.3).  WHOLE, rows of whole vectors of four, is an instance of its own: with the test at every load the compiler put each
// into a block with the element-by-element loads behind it (eight rows of four copies of 1,024, 5.6 -> 5.1 us in a decode step).
constexpr bool streams_ahead(int copies, bool one) { return one || copies <= 6; }
constexpr int streams_rows_a_cu(int copies, bool one) { return streams_ahead(copies, one) ? 1 : 3; }
template <typename T, int N, bool ONE, bool WHOLE>
__global__ __launch_bounds__(256, streams_rows_a_cu(N, ONE)) void streams_step_kernel(float* __restrict__ X, long ldx, int W,
                                                           const float* __restrict__ P, int slices, long p_stride,
                                                           const float* __restrict__ mix, const float* __restrict__ gain,
                                                           const float* __restrict__ take, const float* __restrict__ weight,
                                                           const float* __restrict__ bias, int centred, float eps,
                                                           T* __restrict__ out, long ld_out, const int* __restrict__ rows) {
  __shared__ float mix_s[N * N], gain_s[N], take_s[N], scratch[4], sums_s[4];
  const int r_out = blockIdx.x;
  const long row = rows ? rows[r_out] : r_out;
  float* x = X + row * ldx;
  constexpr bool vec_ok = WHOLE;   // rows of whole vectors of four: a copy's elements and a slice's move as 16 bytes
  extern __shared__ float u_s[];   // what the row's read gave, until the row's sum of squares is known (a thread's own elements)
  const int e_first = 4 * (int)threadIdx.x;
  constexpr int BATCH = 8;         // slice sums requested together
  f32x4 copy[N], got[BATCH], w_first = {0.f, 0.f, 0.f, 0.f}, b_first = w_first;
  const float* p = P ? P + row * W : nullptr;
  auto load_run = [&](int e) LS_INLINED {
#pragma unroll
    for (int s = 0; s < N; ++s) copy[s] = load4(x + (long)s * W, e, W, vec_ok);
  };
  auto load_sums = [&](int e, int s0) LS_INLINED {
#pragma unroll
    for (int u = 0; u < BATCH; ++u) got[u] = load4(p + (long)min(s0 + u, slices - 1) * p_stride, e, W, vec_ok);   // (clamped: no branch between the loads)
  };
  const int i_mix = min((int)threadIdx.x, N * N - 1), i_copy = min((int)threadIdx.x, N - 1);
  constexpr bool AHEAD = streams_ahead(N, ONE);
  const float my_mix = P ? mix[i_mix] : 0.f, my_gain = P ? gain[i_copy] : 0.f, my_take = take ? take[i_copy] : 1.0f;
  if (AHEAD && e_first < W) {
    load_run(e_first);
    if (P) load_sums(e_first, 0);
    if (out) {
      w_first = load4(weight, e_first, W, vec_ok);
      if (bias) b_first = load4(bias, e_first, W, vec_ok);
    }
  }
  if (threadIdx.x < N * N) mix_s[threadIdx.x] = my_mix;
  if (threadIdx.x < N) {
    gain_s[threadIdx.x] = my_gain;
    take_s[threadIdx.x] = my_take;
  }
  ring_barrier();                  // (the factors are there; loads from memory stay on their way)
  float part = 0.f;
  f32x4 u_first = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int e = e_first; e < W; e += ONE ? W : 1024) {
    if (!AHEAD || (!ONE && e != e_first)) load_run(e);
    if (P) {
      f32x4 y = {0.f, 0.f, 0.f, 0.f};
      for (int s0 = 0; s0 < slices; s0 += BATCH) {
        if (!AHEAD || s0 > 0 || (!ONE && e != e_first)) load_sums(e, s0);
#pragma unroll
        for (int u = 0; u < BATCH; ++u)
          if (s0 + u < slices) y = y + got[u];
      }
      f32x4 fresh[N];
#pragma unroll
      for (int t = 0; t < N; ++t) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s2 = 0; s2 < N; ++s2) v = v + mix_s[s2 * N + t] * copy[s2];
        fresh[t] = v + gain_s[t] * y;
      }
#pragma unroll
      for (int t = 0; t < N; ++t) {
        copy[t] = fresh[t];
        if (vec_ok) {
          *reinterpret_cast<f32x4*>(x + (long)t * W + e) = fresh[t];
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (e + i < W) x[(long)t * W + e + i] = fresh[t][i];
        }
      }
    }
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < N; ++t) sum = sum + take_s[t] * copy[t];
    if (ONE || (AHEAD && e == e_first)) u_first = sum;
    else if (out) *reinterpret_cast<f32x4*>(u_s + e) = sum;
#pragma unroll
    for (int i = 0; i < 4; ++i) part = part + (centred ? sum[i] : sum[i] * sum[i]);   // (elements beyond W are zeros)
  }
  if (!out) return;
  // (what a thread reads of u_s it wrote itself; the barriers of the sums are for LDS alone)
  auto row_sum = [&](float v, float* sums) LS_INLINED -> float {
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) sums[threadIdx.x >> 6] = v;
    ring_barrier();
    return ((sums[0] + sums[1]) + sums[2]) + sums[3];
  };
  float mean = 0.f;
  if (centred) {   // (the same for the whole launch)
    mean = row_sum(part, sums_s) / (float)W;
    part = 0.f;
#pragma unroll 1
    for (int e = e_first; e < W; e += ONE ? W : 1024) {
      const f32x4 u = ONE || (AHEAD && e == e_first) ? u_first : *reinterpret_cast<const f32x4*>(u_s + e);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float d = e + i < W ? u[i] - mean : 0.f;
        part = part + d * d;
      }
    }
  }
  const float scale = 1.0f / sqrtf(row_sum(part, scratch) / (float)W + eps);
  const bool vec_out = vec_ok && ld_out % 4 == 0 && reinterpret_cast<uintptr_t>(out) % (4 * sizeof(T)) == 0;
#pragma unroll 1
  for (int e0 = e_first; e0 < W; e0 += ONE ? W : 1024) {
    f32x4 u = u_first, w = w_first, b = b_first;
    if (!AHEAD || (!ONE && e0 != e_first)) {
      u = *reinterpret_cast<const f32x4*>(u_s + e0);
      w = load4(weight, e0, W, vec_ok);
      if (bias) b = load4(bias, e0, W, vec_ok);
    }
    typedef __attribute__((ext_vector_type(4))) T t4;
    t4 o;
    T* dst = out + (long)r_out * ld_out + e0;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = from_f32<T>(((u[i] - mean) * scale) * w[i] + b[i]);
    if (vec_out) {
      *reinterpret_cast<t4*>(dst) = o;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (e0 + i < W) dst[i] = o[i];
    }
  }
}

// ---------------------------------------------------------------------------
// Post pass of the down projections of attention over a latent: raw [T][ld] float = a (QR) | c (CR) | r (RD), the
// last two absent for a layer that reads another layer's latent (has_kv == 0).
//   a -> a / sqrt(mean(a^2) + eps) * a_weight            -> a_out [T][QR] (T); as it is where a_weight is null (queries
//                                                           that do not pass a latent)
//   c -> c / sqrt(mean(c^2) + eps) * c_weight            -> key pages [page][0][slot][0 .. CR) and value pages
//                                                           [page][0][0 .. CR)[slot]: the latent is key and value
//   r -> rotated in neighbouring pairs (2i, 2i + 1) on its first `rot` dimensions at the token's position
//                                                        -> key pages [page][0][slot][CR .. CR + RD), zeros up to Dp
// One workgroup a token; the sums of squares as in streams_step_kernel.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void latent_post_kernel(
    const float* __restrict__ raw, long ld, int QR, int CR, int RD, int Dp, int has_kv, const float* __restrict__ a_weight,
    const float* __restrict__ c_weight, float eps, const float* __restrict__ cos_table, const float* __restrict__ sin_table,
    int rot, const int* __restrict__ tok_seq, const int* __restrict__ tok_pos, const SeqMeta* __restrict__ seqs,
    const int* __restrict__ table, int table_stride, T* __restrict__ a_out, long lda, T* __restrict__ k_pages,
    T* __restrict__ v_pages, int page_size) {
  __shared__ float scratch[4];
  const int t = blockIdx.x;
  const float* row = raw + (long)t * ld;
  if (a_weight) {
    const float part = row_sumsq_part(row, QR, threadIdx.x, false);
    const float scale = 1.0f / sqrtf(block_sum4(part, scratch) / (float)QR + eps);
    for (int e = threadIdx.x; e < QR; e += 256) a_out[(long)t * lda + e] = from_f32<T>((row[e] * scale) * a_weight[e]);
  } else {
    for (int e = threadIdx.x; e < QR; e += 256) a_out[(long)t * lda + e] = from_f32<T>(row[e]);
  }
  if (!has_kv) return;
  const int pos = tok_pos[t];
  const int page = table[(long)seqs[tok_seq[t]].table_row * table_stride + pos / page_size];
  const int slot = pos % page_size;
  const float part = row_sumsq_part(row + QR, CR, threadIdx.x, false);
  const float scale = 1.0f / sqrtf(block_sum4(part, scratch) / (float)CR + eps);
  if (page < 0) return;
  T* key = k_pages + ((long)page * page_size + slot) * Dp;
  T* value = v_pages + (long)page * CR * page_size + slot;
  for (int e = threadIdx.x; e < CR; e += 256) {
    const T c = from_f32<T>((row[QR + e] * scale) * c_weight[e]);
    key[e] = c;
    value[(long)e * page_size] = c;
  }
  const float* r = row + QR + CR;
  const int half = rot >> 1;
  for (int i = threadIdx.x; i < Dp - CR; i += 256) {
    float v = 0.f;
    if (i < RD) {
      v = r[i];
      if (i < rot) {
        const float other = r[i ^ 1], c = cos_table[(long)pos * half + (i >> 1)], s = sin_table[(long)pos * half + (i >> 1)];
        v = (i & 1) ? v * c + other * s : v * c - other * s;
      }
    }
    key[CR + i] = from_f32<T>(v);
  }
}

// ---------------------------------------------------------------------------
// Post pass of the up projection of the queries: qf [T][ld] float holds, head by head, D plain dimensions and RD
// rotated ones.  The plain ones go to plain_out [T][H*D] (T), the operand of the product that brings them into the
// latent's space; the rotated ones are rotated (neighbouring pairs, first `rot` dimensions) and written where the
// attention kernel reads them, behind the CR latent dimensions of a query head of Dp elements (zeros up to Dp).
// A thread takes V neighbouring elements: four where every part of a head and every row is whole vectors, else one.  A
// token is a column of the grid, so that an element's head and place are one 32-bit division.  What bounds it is memory: 2,048
// tokens, 16 heads of 128 + 64 dimensions in bfloat16 (37 MB) 25.2 -> 10.4 us by vectors, 16.3 where they are not aligned; 97 tokens
// 3.4 -> 2.8, eight 2.8 -> 2.7.
// ---------------------------------------------------------------------------
template <typename T, int V>
__global__ __launch_bounds__(256) void latent_query_kernel(const float* __restrict__ qf, long ld, int H, int D,
                                                           int RD, int CR, int Dp, const float* __restrict__ cos_table,
                                                           const float* __restrict__ sin_table, int rot,
                                                           const int* __restrict__ tok_pos, T* __restrict__ plain_out,
                                                           long ldp, T* __restrict__ q_out, long ldq) {
  typedef __attribute__((ext_vector_type(V))) float fv;
  typedef __attribute__((ext_vector_type(V))) T tv;
  const int tail = Dp - CR, each = D + tail, t = blockIdx.x;
  const int idx = ((int)blockIdx.y * 256 + (int)threadIdx.x) * V;
  if (idx >= H * each) return;
  const int head = idx / each, i = idx - head * each, j = i - D;
  const float* src = qf + (long)t * ld + (long)head * (D + RD);
  fv v;
#pragma unroll
  for (int k = 0; k < V; ++k) v[k] = 0.f;
  if (i < D + RD) v = *reinterpret_cast<const fv*>(src + i);
  if (j >= 0 && j < min(rot, RD)) {
    const int half = rot >> 1;
    const long pos = tok_pos[t];
    fv r = v;
#pragma unroll
    for (int k = 0; k < V; ++k)
      if (j + k < rot) {
        const float other = V == 1 ? src[D + (j ^ 1)] : v[k ^ (V > 1)], c = cos_table[pos * half + ((j + k) >> 1)],
                    w = sin_table[pos * half + ((j + k) >> 1)];
        r[k] = ((j + k) & 1) ? v[k] * c + other * w : v[k] * c - other * w;
      }
    v = r;
  }
  tv o;
#pragma unroll
  for (int k = 0; k < V; ++k) o[k] = from_f32<T>(v[k]);
  T* dst = i < D ? plain_out + (long)t * ldp + head * D + i : q_out + (long)t * ldq + (long)head * Dp + CR + j;
  *reinterpret_cast<tv*>(dst) = o;
}

// ---------------------------------------------------------------------------
// A product a head: out[t][head * o_stride + n] = sum_k w[head][n][k] x[t][head * x_stride + k], w [H][N][K].
// A workgroup: 16 * RT rows of one head, four waves with 16 columns each.  The 16x16 MFMA atom with the weight rows
// as first operand; a row's contraction is one chain over ascending K from zero.  WHOLE (row_piece.h): rows that buffer loads
// read (eight rows, sixteen heads of 128 x 128 3.5 -> 3.2 us in a decode step).
// ---------------------------------------------------------------------------
template <typename T, int RT, bool WHOLE>
__global__ __launch_bounds__(256) void heads_product_kernel(const T* __restrict__ x, long ldx, int x_stride,
                                                            const T* __restrict__ w, int N, int K, int n_rows,
                                                            T* __restrict__ out, long ldo, int o_stride, int x_aligned,
                                                            int out_vec) {
  constexpr int VEC = Atom<T>::VEC, KC = Atom<T>::KCHUNK;
  const int head = blockIdx.y;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, quad = lane >> 4;
  const int col0 = (blockIdx.z * 4 + wv) * 16;
  if (col0 >= N) return;
  const bool w_ok = col0 + l16 < N;
  const T* w_base = w + ((long)head * N + col0) * K;
  const int row0 = blockIdx.x * 16 * RT;
  const T* x_base = x + (long)row0 * ldx + (long)head * x_stride;
  bool x_ok[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) x_ok[r] = row0 + 16 * r + l16 < n_rows;
  f32x4 acc[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool w_aligned = K % VEC == 0;
  constexpr int U = 4;
  for (int k0 = 0; k0 < K; k0 += U * KC) {
    typename Atom<T>::vec_t a[U], b[U][RT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * KC + VEC * quad;
      a[u] = row_piece<T, WHOLE>(w_base, l16, k, K, K, w_ok, w_aligned);
#pragma unroll
      for (int r = 0; r < RT; ++r) b[u][r] = row_piece<T, WHOLE>(x_base, 16 * r + l16, k, K, ldx, x_ok[r], x_aligned != 0);
    }
    if constexpr (WHOLE) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int r = 0; r < RT; ++r) Atom<T>::mma(acc[r], a[u], b[u][r]);
  }
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    if (!x_ok[r]) continue;
    T* dst = out + (long)(row0 + 16 * r + l16) * ldo + (long)head * o_stride;
    if (out_vec && col0 + 4 * quad + 3 < N) {   // a lane's four columns in one store
      typedef T out4 __attribute__((ext_vector_type(4)));
      out4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = from_f32<T>(acc[r][i]);
      *reinterpret_cast<out4*>(dst + col0 + 4 * quad) = v;
      continue;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = col0 + 4 * quad + i;
      if (c < N) dst[c] = from_f32<T>(acc[r][i]);
    }
  }
}

// ---------------------------------------------------------------------------
// The gated delta rule.  raw [T][ld] float holds the projections q (G heads of D) | k (G of D) | v (H of DV) |
// b (H) | a (H) | whatever follows.  Per request a state of floats: S [H][D][DV], then the last M - 1 inputs of the
// short convolutions [M - 1][C], C = 2 G D + H DV channels, oldest first, zeros before the start.
//
// (1) delta_prep: a wave a (token, unit).  Units: the G query heads, the G key heads, the H value heads, and one for
//     the gates.  A channel's convolution y = sum_m taps[c][m] in(p - (M - 1) + m) (m ascending) takes the inputs of
//     this step from raw and those before it from the state; then silu; queries and keys become unit vectors
//     x / sqrt(sum x^2 + unit_eps) (lane i adds the squares of the elements i, i + 64, ... ascending, then a
//     butterfly), the query also times D^(-1/2).  Gates of head h: beta = sigmoid(b_h),
//     decay = exp(-exp(A_log_h) softplus(a_h + dt_bias_h)).
//     qk [T][2 G][dp] (queries, then keys; zeros beyond D), vv [T][H * DV], gates [T][H][2].
// (2) delta_rule: a wave a (request, head, 64 / L columns of the state); L neighbouring lanes share a column, lane
//     part p of them keeps the rows p * R + {0 .. R-1}.  Per token, in order:
//       kS = decay * sum_r S[r] k[r];  u = beta (v - kS);  S[r] = decay S[r] + k[r] u;  o = sum_r S[r] q[r]
//     (the sums: a lane's rows in four interleaved chains of fused multiply-adds, then the lanes of a column by moves inside their row of sixteen; the
//     decay multiplies the sum of the old state with the key, which is the decayed state's sum up to rounding).
//     A token's operands are requested eight (four) tokens before it is worked on.
//     The request's waves also make the last M - 1 inputs of every channel, which (1) has read, the state of the next step
//     (a launch of its own for that took 5 us of a decode step's 29 a layer).
// ---------------------------------------------------------------------------
// MM: the taps of the convolution where they are one aligned vector (4; all of an element's loads are then on their way
// together: 2,048 tokens, 4,096 channels 51.7 -> 31.3 us, eight tokens 8.4 -> 5.6), or 0: any number, in a loop.
template <int MM>
__global__ __launch_bounds__(256) void delta_prep_kernel(
    const float* __restrict__ raw, long ld, int n_tokens, int G, int H, int D, int DV, int dp, int M,
    const float* __restrict__ taps, const float* __restrict__ a_log, const float* __restrict__ dt_bias, float unit_eps,
    const int* __restrict__ tok_seq, const int* __restrict__ tok_pos, const SeqMeta* __restrict__ seqs,
    const float* __restrict__ state, long state_stride, long conv_at, float* __restrict__ qk, float* __restrict__ vv,
    float* __restrict__ gates, const float* __restrict__ chan, long ldc, float* __restrict__ decays) {
  // (with a decay a key channel, chan [T][ldc] holds its H * D logits and dt_bias has as many entries: a unit a head
  // then forms the head's beta and its row of decays, decays [T][H][dp], ones beyond D)
  const int units = 2 * G + H + (chan ? H : 1);
  const long id = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (id >= (long)n_tokens * units) return;
  const int t = (int)(id / units), unit = (int)(id % units), lane = threadIdx.x & 63;
  const float* row = raw + (long)t * ld;
  const int C = 2 * G * D + H * DV;
  if (chan && unit >= 2 * G + H) {
    const int h = unit - (2 * G + H);
    if (lane < 2) gates[((long)t * H + h) * 2 + lane] = lane == 0 ? sigmoid_f(row[C + h]) : 1.0f;
    const float rate = expf(a_log[h]);
    for (int r = lane; r < dp; r += 64)
      decays[((long)t * H + h) * dp + r] =
          r < D ? expf(-rate * softplus_f(chan[(long)t * ldc + h * D + r] + dt_bias[h * D + r])) : 1.0f;
    return;
  }
  if (unit == units - 1) {
    for (int h = lane; h < H; h += 64) {
      gates[((long)t * H + h) * 2] = sigmoid_f(row[C + h]);
      gates[((long)t * H + h) * 2 + 1] = expf(-expf(a_log[h]) * softplus_f(row[C + H + h] + dt_bias[h]));
    }
    return;
  }
  const SeqMeta m = seqs[tok_seq[t]];
  const int pos = tok_pos[t];
  const float* old = state + (long)m.table_row * state_stride + conv_at;
  const bool is_v = unit >= 2 * G;
  const int size = is_v ? DV : D;
  const int c0 = is_v ? 2 * G * D + (unit - 2 * G) * DV : unit * D;
  // channel c at this token: convolution over the last M inputs, then silu.  An input's address is chosen (this
  // step's rows, or the state), then loaded: no branch stands between the loads of the taps.
  auto channel = [&](int c) LS_INLINED {
    auto input = [&](int a) LS_INLINED {
      const int p = pos - (M - 1) + a;
      return p >= m.q_start ? raw + (long)(m.q_off + p - m.q_start) * ld + c : old + (long)(p - m.q_start + M - 1) * C + c;
    };
    float y = 0.f;
    if constexpr (MM > 0) {
      typedef __attribute__((ext_vector_type(MM > 0 ? MM : 1))) float taps_t;
      const taps_t w = *reinterpret_cast<const taps_t*>(taps + (long)c * MM);
      float x[MM > 0 ? MM : 1];
#pragma unroll
      for (int a = 0; a < MM; ++a) x[a] = *input(a);
#pragma unroll
      for (int a = 0; a < MM; ++a) y = y + w[a] * x[a];
    } else {
      for (int a = 0; a < M; ++a) y = y + taps[(long)c * M + a] * *input(a);
    }
    return silu_f(y);
  };
  if (is_v) {
    for (int i0 = 0; i0 < size; i0 += 128) {   // (two elements of a lane at a time, their loads together)
      float* dst = vv + (long)t * H * DV + (c0 - 2 * G * D) + i0 + lane;
      if (i0 + 64 < size) {
        const float y0 = channel(c0 + i0 + lane), y1 = channel(c0 + min(i0 + 64 + lane, size - 1));
        dst[0] = y0;
        if (i0 + 64 + lane < size) dst[64] = y1;
      } else if (i0 + lane < size) {           // (the same for the wave but for this test: no second element to compute)
        dst[0] = channel(c0 + i0 + lane);
      }
    }
    return;
  }
  // a head of up to 256 elements: a lane keeps its up to four in registers between the sum and the scaling
  float mine[4];
  float part = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = lane + 64 * j;
    mine[j] = 0.f;
    if (64 * j < size) {   // (the same for the wave; the loads of a lane's elements stand together)
      const float y = channel(c0 + min(i, size - 1));
      mine[j] = i < size ? y : 0.f;
    }
    part = part + mine[j] * mine[j];
  }
  float scale = 1.0f / sqrtf(wave_sum(part) + unit_eps);
  if (unit < G) scale = scale * (1.0f / sqrtf((float)D));
  float* dst = qk + ((long)t * 2 * G + unit) * dp;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = lane + 64 * j;
    if (i < dp) dst[i] = mine[j] * scale;
  }
}

// Sum over the L (4, 8 or 16) neighbouring lanes that share a column, by data-parallel moves inside a row of sixteen
// lanes (no LDS): pairs, pairs of pairs, then the mirror image of the half row and of the row.  After every step
// the lanes that were added hold the same value, so all L lanes end with the same bits.
template <int L>
__device__ __forceinline__ float lanes_sum(float v) {
  v = v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));  // lanes 1 0 3 2
  v = v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true));  // lanes 2 3 0 1
  if constexpr (L >= 8) v = v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xF, 0xF, true));  // 7 - i
  if constexpr (L >= 16) v = v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xF, 0xF, true));  // 15 - i
  return v;
}

// The last M - 1 inputs of the channels c, c + step, ...: place a holds the input at position kv_len - (M - 1) + a, one of this
// step's, or one the state already holds further on.  SETTLE: every load is used on every path.  One that might still be on its way to
// its register when the recurrence reuses that was waited for in each of the recurrence's blocks, with all but seven of the loads that are
// ahead there (2,048 tokens 301 / 290 us).  With a decay a channel the compiler finds other registers, and the wait itself costs (16 heads
// over 8 of 128 x 128 352 / 338 without it, 4 over 2 of 96 x 80 313 / 302).
template <bool SETTLE>
__device__ __forceinline__ void keep_inputs(const float* __restrict__ raw, long ld, int C, int M, const SeqMeta& m, float* __restrict__ kept,
                                            int c, int step) {
  for (; c < C; c += step) {
    auto input = [&](int a) LS_INLINED -> const float* {
      const int p = m.kv_len - (M - 1) + a;
      return p >= m.q_start ? raw + (long)(m.q_off + p - m.q_start) * ld + c : kept + (long)(p - m.q_start + M - 1) * C + c;
    };
    constexpr int kAtOnce = 3;
    for (int a0 = 0; a0 < M - 1; a0 += kAtOnce) {  // (read before the ascending walk overwrites it)
      float v[kAtOnce];
#pragma unroll
      for (int u = 0; u < kAtOnce; ++u) v[u] = *input(min(a0 + u, M - 2));
#pragma unroll
      for (int u = 0; u < kAtOnce; ++u)
        if (a0 + u < M - 1) kept[(long)(a0 + u) * C + c] = v[u];
      if constexpr (SETTLE)
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) __asm__ volatile("" ::"v"(v[u]));
    }
  }
}

// R rows a lane, L lanes a column (R * L rows, the head size rounded up), 64 / L columns a wave.  CH: the decay is a
// number a row of the state (decays [T][H][dp]) instead of one a head: S[r] <- g[r] S[r] first, then the rule as stated.
//
// What bounds a long request is the instructions of one wave (a head of 128 x 128 is 32 waves, sixteen heads half of the
// card's SIMDs), so a token carries its arithmetic and little else: operands come by buffer loads whose lane offsets
// never change and whose scalar offset is the token's place in its block of DEPTH; a block moves the bases once; lanes
// and columns past the state have an offset past the buffer's end, which reads as zero and is not written, in place of
// branches; only the blocks whose requests would leave the request hold them at its last token.  beta and the decay come
// by one vector load at the same address in every lane (as scalar loads, which return in any order, a wait for one would
// be a wait for all, also for those of the tokens ahead).
// DEPTH: the tokens whose operands are on their way.  2,048 tokens (16 heads over 8, 128 x 128): 258 us under the profiler (271 with a wait
// for all of them in every block, see keep_inputs and the order of the first requests), 281 with a decay
// a channel; with lane pointers, a conditional step of each, and a branch a token it took 490.  Where the longest request brings a token or two,
// two are enough and leave room for twice the waves: eight requests decoding 28 -> 13 us.  Where most requests decode beside
// a longer one, the longest's chain counts as much as the room: four (63 requests of one token and one of 64, two / four / eight
// ahead, convolution included: 64 x 64 48 / 39 / 38 us, 128 x 128 114 / 113 / 130, 192 x 128 143 / 95 / 100).  Else eight, with
// sixteen rows a lane four (1,024 tokens, 192 x 128 231 us, eight 240), or two where the waves are more than two a SIMD, as
// many as four leave room for (16 requests of one token and four of 256 98 us, four 165).
template <int R, int L, bool CH, int DEPTH>
__global__ __launch_bounds__(64) void delta_rule_kernel(const float* __restrict__ qk, const float* __restrict__ vv,
                                                        const float* __restrict__ gates, const float* __restrict__ decays,
                                                        int G, int H, int D, int DV,
                                                        const SeqMeta* __restrict__ seqs, float* __restrict__ state,
                                                        long state_stride, float* __restrict__ out, long ldo,
                                                        const float* __restrict__ raw, long ld, int C, int M, long conv_at) {
  typedef __attribute__((ext_vector_type(2))) unsigned int u32x2_t;
  typedef __attribute__((ext_vector_type(4))) unsigned int u32x4_t;
  constexpr int dp = L * R, COLS = 64 / L;
  constexpr int kNowhere = 0x7ffffff0;  // an offset past every buffer's end
  const int seq = blockIdx.x / H, head = blockIdx.x % H;
  const SeqMeta m = seqs[seq];
  const int n = m.q_len;
  if (n <= 0) return;
  const int lane = threadIdx.x, lc = lane / L, part = lane % L;
  const int col = blockIdx.y * COLS + lc;
  const bool col_ok = col < DV;
  const int row0 = part * R;
  const int kh = head / (H / G);
  auto buffer = [](const float* p, int bytes) LS_INLINED {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, bytes, 0x00020000);
  };
  const auto mine = buffer(state + (long)m.table_row * state_stride + (long)head * D * DV, D * DV * 4);
  int s_off[R];
  float S[R];
#pragma unroll
  for (int r = 0; r < R; ++r) s_off[r] = row0 + r < D && col_ok ? ((row0 + r) * DV + col) * 4 : kNowhere;
#pragma unroll
  for (int r = 0; r < R; ++r) S[r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(mine, s_off[r], 0, 0));
  struct Operands {
    u32x4_t q[R / 4], k[R / 4], g[CH ? R / 4 : 1];
    unsigned v;
    u32x2_t gate;  // beta, decay (CH: beta alone, see fetch)
  };
  // the first token of the block, and bytes from a token to the next
  const float* qk_at = qk + ((long)m.q_off * 2 * G + kh) * dp;
  const float* v_at = vv + (long)m.q_off * H * DV + head * DV;
  const float* g_at = gates + ((long)m.q_off * H + head) * 2;
  const float* d_at = CH ? decays + ((long)m.q_off * H + head) * dp : nullptr;
  float* o_at = out + (long)m.q_off * ldo + head * DV;
  const int qk_step = 2 * G * dp * 4, v_step = H * DV * 4, g_step = H * 8, d_step = H * dp * 4, o_step = DEPTH > 1 ? (int)ldo * 4 : 0;
  const int q_off = row0 * 4, k_off = (G * dp + row0) * 4, v_off = (col_ok ? col : 0) * 4;
  const int o_off = part == 0 && col_ok ? col * 4 : kNowhere;
  int zero = 0;
  __asm__("" : "+v"(zero));
  Operands ring[DEPTH];
  auto fetch = [&](Operands& x, auto qkb, auto vb, auto gb, auto db, int t) LS_INLINED {  // the token t tokens from the block's first
#pragma unroll
    for (int j = 0; j < R / 4; ++j) {
      x.k[j] = __builtin_amdgcn_raw_buffer_load_b128(qkb, k_off + 16 * j, t * qk_step, 0);
      x.q[j] = __builtin_amdgcn_raw_buffer_load_b128(qkb, q_off + 16 * j, t * qk_step, 0);
      if constexpr (CH) x.g[j] = __builtin_amdgcn_raw_buffer_load_b128(db, q_off + 16 * j, t * d_step, 0);
    }
    x.v = __builtin_amdgcn_raw_buffer_load_b32(vb, v_off, t * v_step, 0);
    // (a second word that nobody reads would be a register the compiler uses for something else while the load is still on
    // its way to it, behind a wait for every load in flight)
    if constexpr (CH) x.gate[0] = __builtin_amdgcn_raw_buffer_load_b32(gb, zero, t * g_step, 0);
    else x.gate = __builtin_amdgcn_raw_buffer_load_b64(gb, zero, t * g_step, 0);
  };
  float o4[4] = {};  // the lane's part of the output of the token that was worked on last
  auto token = [&](const Operands& now) LS_INLINED {
    auto of = [](const u32x4_t (&x)[R / 4], int r) LS_INLINED { return __uint_as_float(x[r >> 2][r & 3]); };
    const float beta = __uint_as_float(now.gate[0]), decay = CH ? 1.0f : __uint_as_float(now.gate[1]);
    // a lane's rows in four interleaved chains (rows r, r + 4, ... of each), added as (0 + 1) + (2 + 3)
    float ks4[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (CH) {
#pragma unroll
      for (int r = 0; r < R; ++r) S[r] = S[r] * __uint_as_float(now.g[r >> 2][r & 3]);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) ks4[r & 3] = fmaf(S[r], of(now.k, r), ks4[r & 3]);
    const float ks = lanes_sum<L>((ks4[0] + ks4[1]) + (ks4[2] + ks4[3])) * (CH ? 1.0f : decay);
    const float u = beta * (__uint_as_float(now.v) - ks);
#pragma unroll
    for (int i = 0; i < 4; ++i) o4[i] = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      S[r] = fmaf(of(now.k, r), u, CH ? S[r] : decay * S[r]);
      o4[r & 3] = fmaf(S[r], of(now.q, r), o4[r & 3]);
    }
  };
  auto put = [&](auto ob, float o, int j) LS_INLINED {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o), ob, o_off, j * o_step, 0);
  };
  // ... in a whole block every GROUP tokens at once, lane i of a column the i-th of them: a store whose lanes mostly have nothing
  // to write holds up the loads behind it (four requests of 512 tokens, 16 heads of 128 x 128, with a store a token 231 us, so 212)
  constexpr int GROUP = L < DEPTH ? L : DEPTH;
  const int group_off = part < GROUP && col_ok ? part * o_step + col * 4 : kNowhere;
  float kept = 0.f;
  auto put_grouped = [&](auto ob, float o, int j) LS_INLINED {
    kept = part == j % GROUP ? o : kept;
    if (j % GROUP == GROUP - 1)
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(kept), ob, group_off, (j - (GROUP - 1)) * o_step, 0);
  };
  {
    const auto qkb = buffer(qk_at, kNowhere), vb = buffer(v_at, kNowhere), gb = buffer(g_at, kNowhere), db = buffer(d_at, kNowhere);
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) {
      fetch(ring[j], qkb, vb, gb, db, min(j, n - 1));
      __builtin_amdgcn_sched_barrier(0);  // (in the order in which the loop waits for them)
    }
  }
  if (M > 1)
    keep_inputs<!CH>(raw, ld, C, M, m, state + (long)m.table_row * state_stride + conv_at, (head * (int)gridDim.y + (int)blockIdx.y) * 64 + lane,
                64 * H * (int)gridDim.y);
  auto next_block = [&]() LS_INLINED {
    qk_at += (long)DEPTH * 2 * G * dp;
    v_at += (long)DEPTH * H * DV;
    g_at += (long)DEPTH * H * 2;
    if constexpr (CH) d_at += (long)DEPTH * H * dp;
    o_at += (long)DEPTH * ldo;
  };
  int i0 = 0;
  for (; i0 + 2 * DEPTH <= n; i0 += DEPTH) {
    const auto qkb = buffer(qk_at, kNowhere), vb = buffer(v_at, kNowhere), gb = buffer(g_at, kNowhere), db = buffer(d_at, kNowhere);
    const auto ob = buffer(o_at, kNowhere);
    // a token's output is added up beside the next token's products: each is a chain that waits for itself
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) {
      const float before = (o4[0] + o4[1]) + (o4[2] + o4[3]);
      token(ring[j]);
      if (j > 0) put_grouped(ob, lanes_sum<L>(before), j - 1);
      __builtin_amdgcn_sched_barrier(0);
      fetch(ring[j], qkb, vb, gb, db, DEPTH + j);
      __builtin_amdgcn_sched_barrier(0);
    }
    put_grouped(ob, lanes_sum<L>((o4[0] + o4[1]) + (o4[2] + o4[3])), DEPTH - 1);
    next_block();
  }
  for (; i0 < n; i0 += DEPTH) {
    const auto qkb = buffer(qk_at, kNowhere), vb = buffer(v_at, kNowhere), gb = buffer(g_at, kNowhere), db = buffer(d_at, kNowhere);
    const auto ob = buffer(o_at, kNowhere);
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) {
      if (i0 + j >= n) break;
      token(ring[j]);
      put(ob, lanes_sum<L>((o4[0] + o4[1]) + (o4[2] + o4[3])), j);
      if (i0 + DEPTH + j < n) fetch(ring[j], qkb, vb, gb, db, DEPTH + j);
    }
    next_block();
  }
#pragma unroll
  for (int r = 0; r < R; ++r) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(S[r]), mine, s_off[r], 0, 0);
}

}  // namespace ls

using namespace ls;

extern "C" int ls_streams_max() { return kMaxStreams; }
extern "C" int ls_streams_max_width() { return 1024 * kStreamChunks; }

extern "C" int ls_streams_step(int dtype, float* X, long ldx, int n, int width, const float* P, int slices, int p_rows,
                               const float* mix, const float* gain, const float* take, const float* weight, const float* bias,
                               int centred, float eps, void* out, long ld_out, const int* rows, int n_rows, void* stream) {
  LS_REQUIRE(n_rows > 0 && n > 0 && n <= kMaxStreams && width > 0 && width <= 1024 * kStreamChunks && ldx >= (long)n * width,
             "streams_step: %d copies of %d elements (at most %d of %d)", n, width, kMaxStreams, 1024 * kStreamChunks);
  LS_REQUIRE(X && (P || out), "streams_step: nothing to do");
  LS_REQUIRE(!P || (slices > 0 && p_rows > 0 && mix && gain), "streams_step: a write needs slices, mix and gain");
  LS_REQUIRE(!out || (weight && ld_out >= width && eps > 0.f), "streams_step: a read needs a weight and eps");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const long p_stride = (long)p_rows * width;
  LS_REQUIRE(dtype == kF32 || dtype == kBF16, "streams_step: unknown dtype %d", dtype);
  const size_t lds = out ? (size_t)((width + 3) / 4) * 16 : 0;
  const bool whole = width % 4 == 0 && ldx % 4 == 0;
#define LS_STREAMS_AS(T_, N_, ONE_) \
  if (whole) LS_STREAMS_ROWS(T_, N_, ONE_, true); else LS_STREAMS_ROWS(T_, N_, ONE_, false)
#define LS_STREAMS_ROWS(T_, N_, ONE_, WHOLE_)                                                                        \
  hipLaunchKernelGGL((streams_step_kernel<T_, N_, ONE_, WHOLE_>), dim3(n_rows), dim3(256), lds, s, X, ldx, width, P, slices, \
                     p_stride, mix, gain, take, weight, bias, centred, eps, (T_*)out, ld_out, rows)
#define LS_STREAMS(N_)                                                                                               \
  case N_:                                                                                                           \
    if (dtype == kF32) {                                                                                             \
      if (width <= 1024) { LS_STREAMS_AS(float, N_, true); } else { LS_STREAMS_AS(float, N_, false); }               \
    } else {                                                                                                         \
      if (width <= 1024) { LS_STREAMS_AS(bf16_t, N_, true); } else { LS_STREAMS_AS(bf16_t, N_, false); }             \
    }                                                                                                                \
    break;
  switch (n) {
    LS_STREAMS(1) LS_STREAMS(2) LS_STREAMS(3) LS_STREAMS(4) LS_STREAMS(5) LS_STREAMS(6) LS_STREAMS(7) LS_STREAMS(8)
  }
#undef LS_STREAMS
#undef LS_STREAMS_AS
#undef LS_STREAMS_ROWS
  return check_launch("streams_step");
}

extern "C" int ls_latent_post(int dtype, const float* raw, long ld, int n_tokens, int QR, int CR, int RD, int Dp,
                              int has_kv, const float* a_weight, const float* c_weight, float eps, const float* cos_table,
                              const float* sin_table, int rot, int table_positions, int max_pos, const int* tok_seq,
                              const int* tok_pos, const void* seqs, const int* table, int table_stride, void* a_out,
                              long lda, void* k_pages, void* v_pages, int page_size, void* stream) {
  LS_REQUIRE(n_tokens > 0 && QR > 0 && raw && a_out && lda >= QR && eps > 0.f, "latent_post: bad query latent");
  LS_REQUIRE(ld >= QR + (has_kv ? CR + RD : 0), "latent_post: rows of %ld floats are too short", ld);
  if (has_kv) {
    LS_REQUIRE(CR > 0 && RD >= 0 && Dp >= CR + RD && c_weight && k_pages && v_pages && table && seqs && tok_seq && tok_pos &&
                   page_size > 0 && table_stride > 0,
               "latent_post: bad key/value latent");
    LS_REQUIRE(rot >= 0 && rot % 2 == 0 && rot <= RD, "latent_post: %d rotated dimensions of %d", rot, RD);
    LS_REQUIRE(rot == 0 || (cos_table && sin_table && max_pos < table_positions),
               "latent_post: position %d is beyond the rotation tables (%d)", max_pos, table_positions);
    LS_REQUIRE(max_pos / page_size < table_stride, "latent_post: position %d is beyond the block table", max_pos);
  }
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
#define LS_LATENT_POST(T_)                                                                                            \
  hipLaunchKernelGGL(latent_post_kernel<T_>, dim3(n_tokens), dim3(256), 0, s, raw, ld, QR, CR, RD, Dp, has_kv, a_weight, \
                     c_weight, eps, cos_table, sin_table, rot, tok_seq, tok_pos, (const SeqMeta*)seqs, table,         \
                     table_stride, (T_*)a_out, lda, (T_*)k_pages, (T_*)v_pages, page_size)
  if (dtype == kF32)
    LS_LATENT_POST(float);
  else if (dtype == kBF16)
    LS_LATENT_POST(bf16_t);
  else
    return fail("latent_post: unknown dtype %d", dtype);
#undef LS_LATENT_POST
  return check_launch("latent_post");
}

extern "C" int ls_latent_query(int dtype, const float* qf, long ld, int n_tokens, int H, int D, int RD, int CR, int Dp,
                               const float* cos_table, const float* sin_table, int rot, int table_positions, int max_pos,
                               const int* tok_pos, void* plain_out, long ldp, void* q_out, long ldq, void* stream) {
  LS_REQUIRE(n_tokens > 0 && H > 0 && D > 0 && RD >= 0 && CR > 0 && Dp >= CR + RD, "latent_query: bad sizes");
  LS_REQUIRE(qf && plain_out && q_out && tok_pos && ld >= (long)H * (D + RD) && ldp >= (long)H * D && ldq >= (long)H * Dp,
             "latent_query: bad operands");
  LS_REQUIRE(rot >= 0 && rot % 2 == 0 && rot <= RD, "latent_query: %d rotated dimensions of %d", rot, RD);
  LS_REQUIRE(rot == 0 || (cos_table && sin_table && max_pos < table_positions),
             "latent_query: position %d is beyond the rotation tables (%d)", max_pos, table_positions);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const size_t element = dtype == kF32 ? 4 : 2;
  const bool whole = D % 4 == 0 && RD % 4 == 0 && CR % 4 == 0 && Dp % 4 == 0 && ld % 4 == 0 && ldp % 4 == 0 && ldq % 4 == 0 &&
                     reinterpret_cast<uintptr_t>(qf) % 16 == 0 && reinterpret_cast<uintptr_t>(plain_out) % (4 * element) == 0 &&
                     reinterpret_cast<uintptr_t>(q_out) % (4 * element) == 0;
  const int per = 256 * (whole ? 4 : 1);
  const dim3 grid(n_tokens, (H * (D + Dp - CR) + per - 1) / per);
#define LS_LATENT_QUERY(T_, V_)                                                                                      \
  hipLaunchKernelGGL((latent_query_kernel<T_, V_>), grid, dim3(256), 0, s, qf, ld, H, D, RD, CR, Dp, cos_table,      \
                     sin_table, rot, tok_pos, (T_*)plain_out, ldp, (T_*)q_out, ldq)
  if (dtype == kF32) {
    if (whole) LS_LATENT_QUERY(float, 4); else LS_LATENT_QUERY(float, 1);
  } else if (dtype == kBF16) {
    if (whole) LS_LATENT_QUERY(bf16_t, 4); else LS_LATENT_QUERY(bf16_t, 1);
  } else {
    return fail("latent_query: unknown dtype %d", dtype);
  }
#undef LS_LATENT_QUERY
  return check_launch("latent_query");
}

extern "C" int ls_heads_product(int dtype, const void* x, long ldx, int x_stride, const void* w, int H, int N, int K,
                                int n_rows, void* out, long ldo, int o_stride, void* stream) {
  LS_REQUIRE(n_rows > 0 && H > 0 && N > 0 && K > 0 && x && w && out, "heads_product: bad sizes");
  LS_REQUIRE(x_stride >= 0 && o_stride >= 0 && ldx >= (long)(H - 1) * x_stride + K && ldo >= (long)(H - 1) * o_stride + N,
             "heads_product: the heads do not fit the rows");
  LS_REQUIRE(dtype == kF32 || dtype == kBF16, "heads_product: unknown dtype %d", dtype);
  const int vec = dtype == kF32 ? 4 : 8;
  LS_REQUIRE(reinterpret_cast<uintptr_t>(w) % 16 == 0, "heads_product: the weights must be 16-byte aligned");
  const int x_aligned = reinterpret_cast<uintptr_t>(x) % 16 == 0 && ldx % vec == 0 && x_stride % vec == 0 && K % vec == 0;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int out_vec = ldo % 4 == 0 && o_stride % 4 == 0 && reinterpret_cast<uintptr_t>(out) % (dtype == kF32 ? 16 : 8) == 0;
  const bool many = n_rows > 64;
  const int rows_a_block = many ? 64 : 16;
  const dim3 grid((n_rows + rows_a_block - 1) / rows_a_block, H, (N + 63) / 64);
  // (many rows of bfloat16 are bound by their products, and a last round of loads that is not whole is multiplied to its end: 2,048 rows, 32
  // heads of 64 x 192 18.6 / 17.7 us by the general loads, of 64 x 128 12.1 / 12.3, eight of 40 x 24 3.0 / 3.4)
  const bool padded = dtype == kBF16 && many && K > 64 && K % 128 != 0;
  const bool whole = x_aligned && !padded && 65 * std::max(ldx, (long)K) * (long)(16 / vec) <= kNoPiece;
#define LS_HEADS(T_, RT_) \
  if (whole) LS_HEADS_AS(T_, RT_, true); else LS_HEADS_AS(T_, RT_, false)
#define LS_HEADS_AS(T_, RT_, WHOLE_)                                                                                 \
  hipLaunchKernelGGL((heads_product_kernel<T_, RT_, WHOLE_>), grid, dim3(256), 0, s, (const T_*)x, ldx, x_stride, (const T_*)w, N, \
                     K, n_rows, (T_*)out, ldo, o_stride, x_aligned, out_vec)
  if (dtype == kF32) {
    if (many) LS_HEADS(float, 4); else LS_HEADS(float, 1);
  } else {
    if (many) LS_HEADS(bf16_t, 4); else LS_HEADS(bf16_t, 1);
  }
#undef LS_HEADS
#undef LS_HEADS_AS
  return check_launch("heads_product");
}

extern "C" int ls_delta_max_dim() { return 256; }

// The rows of a head's queries and keys in the scratch buffer: the head size rounded up to what the lanes of the
// recurrence hold (16, 32, 64, 128 or 256).
extern "C" int ls_delta_padded_dim(int D) {
  int dp = 16;
  while (dp < D) dp *= 2;
  return dp;
}

// Floats of scratch that ls_delta_rule needs: qk, vv and gates.
extern "C" long ls_delta_scratch_floats(int n_tokens, int G, int H, int D, int DV) {
  return (long)n_tokens * (2L * G * ls_delta_padded_dim(D) + (long)H * DV + 2L * H);
}
// ... and with a decay a key channel (chan given): the decays as well.
extern "C" long ls_delta_scratch_floats_channel(int n_tokens, int G, int H, int D, int DV) {
  return ls_delta_scratch_floats(n_tokens, G, H, D, DV) + (long)n_tokens * H * ls_delta_padded_dim(D);
}

// longest: the most tokens that one request brings, 0 if the caller does not know (it decides the time, not the result).
extern "C" int ls_delta_rule_longest(const float* raw, long ld, int n_tokens, int G, int H, int D, int DV, int M,
                                     const float* taps, const float* a_log, const float* dt_bias, float unit_eps,
                                     const int* tok_seq, const int* tok_pos, const void* seqs, int n_seqs, float* state,
                                     long state_stride, float* scratch, float* out, long ldo, const float* chan, long ldc,
                                     int longest, void* stream) {
  // chan [T][ldc] (or null): the logits of a decay a head and key channel, H * D a token; dt_bias then has H * D
  // entries, raw needs no `a` columns, and the scratch is that of ls_delta_scratch_floats_channel.
  LS_REQUIRE(!chan || ldc >= (long)H * D, "delta_rule: the channel decays' rows are too short");
  LS_REQUIRE(n_tokens > 0 && n_seqs > 0 && G > 0 && H > 0 && H % G == 0 && D > 0 && D <= 256 && DV > 0 && M >= 1,
             "delta_rule: bad sizes (%d key heads, %d heads, keys of %d, values of %d, %d taps)", G, H, D, DV, M);
  const long C = 2L * G * D + (long)H * DV;
  const long conv_at = (long)H * D * DV;
  LS_REQUIRE(ld >= C + (chan ? 1L : 2L) * H && state_stride >= conv_at + (long)(M - 1) * C && ldo >= (long)H * DV,
             "delta_rule: rows or state are too short");
  LS_REQUIRE(raw && taps && a_log && dt_bias && tok_seq && tok_pos && seqs && state && scratch && out,
             "delta_rule: null operand");
  LS_REQUIRE(reinterpret_cast<uintptr_t>(scratch) % 16 == 0, "delta_rule: the scratch must be 16-byte aligned");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int dp = ls_delta_padded_dim(D);
  float* qk = scratch;
  float* vv = qk + (long)n_tokens * 2 * G * dp;
  float* gates = vv + (long)n_tokens * H * DV;
  float* decays = chan ? gates + (long)n_tokens * H * 2 : nullptr;
  const long units = (long)n_tokens * (2 * G + H + (chan ? H : 1));
  auto prepare = M == 4 && reinterpret_cast<uintptr_t>(taps) % 16 == 0 ? delta_prep_kernel<4> : delta_prep_kernel<0>;
  hipLaunchKernelGGL(prepare, dim3((unsigned)((units + 3) / 4)), dim3(256), 0, s, raw, ld, n_tokens, G, H, D, DV,
                     dp, M, taps, a_log, dt_bias, unit_eps, tok_seq, tok_pos, (const SeqMeta*)seqs, state, state_stride,
                     conv_at, qk, vv, gates, chan, ldc, decays);
  const int most = longest > 0 ? longest : n_tokens;
  const bool mixed = n_tokens <= 2 * n_seqs;  // (and a longer request among them)
  const bool far = ldo >= (1L << 26);  // output rows that a block's 32-bit offsets do not reach: a block of one token
#define LS_DELTA_RULE(R_, L_, CH_, DEPTH_)                                                                               \
  hipLaunchKernelGGL((delta_rule_kernel<R_, L_, CH_, DEPTH_>), dim3(n_seqs * H, (DV * L_ + 63) / 64), dim3(64), 0, s, qk, vv, \
                     gates, decays, G, H, D, DV, (const SeqMeta*)seqs, state, state_stride, out, ldo, raw, ld, (int)C, M, conv_at)
#define LS_DELTA(R_, L_)                                                          \
  do {                                                                            \
    if (far) {                                                                    \
      if (chan) LS_DELTA_RULE(R_, L_, true, 1); else LS_DELTA_RULE(R_, L_, false, 1); \
    } else if (most <= 2 || (R_ > 8 && !mixed && (long)n_seqs * H * ((DV * L_ + 63) / 64) > 8L * compute_units())) { \
      if (chan) LS_DELTA_RULE(R_, L_, true, 2); else LS_DELTA_RULE(R_, L_, false, 2); \
    } else if (mixed) {                                                           \
      if (chan) LS_DELTA_RULE(R_, L_, true, 4); else LS_DELTA_RULE(R_, L_, false, 4); \
    } else {                                                                      \
      if (chan) LS_DELTA_RULE(R_, L_, true, R_ <= 8 ? 8 : 4); else LS_DELTA_RULE(R_, L_, false, R_ <= 8 ? 8 : 4); \
    }                                                                             \
  } while (0)
  switch (dp) {
    case 16: LS_DELTA(4, 4); break;
    case 32: LS_DELTA(8, 4); break;
    case 64: LS_DELTA(8, 8); break;
    case 128: LS_DELTA(8, 16); break;
    default: LS_DELTA(16, 16); break;
  }
#undef LS_DELTA
#undef LS_DELTA_RULE
  return check_launch("delta_rule");
}

extern "C" int ls_delta_rule(const float* raw, long ld, int n_tokens, int G, int H, int D, int DV, int M,
                             const float* taps, const float* a_log, const float* dt_bias, float unit_eps,
                             const int* tok_seq, const int* tok_pos, const void* seqs, int n_seqs, float* state,
                             long state_stride, float* scratch, float* out, long ldo, const float* chan, long ldc,
                             void* stream) {
  return ls_delta_rule_longest(raw, ld, n_tokens, G, H, D, DV, M, taps, a_log, dt_bias, unit_eps, tok_seq, tok_pos, seqs, n_seqs,
                               state, state_stride, scratch, out, ldo, chan, ldc, 0, stream);
}
