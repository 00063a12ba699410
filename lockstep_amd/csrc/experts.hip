// A feed-forward of many small experts of which each token uses a few (routing on the device, no
// word of it read by the host):
//
//   z[t]        = router logits of token t (float, computed by the caller's matrix product) + bias
//   chosen(t)   = the `top` experts with the largest z[t] (the lower index wins a tie), in that order
//   w[t, k]     = softmax over the chosen logits alone
//                 (scoring 1: the sigmoid of each; scoring 2: the choice is made by softmax(z) + correction, within the
//                 best groups of experts, and the weights are the chosen softmax(z) divided by their sum)
//   expert e    : y = act(W_gate[e] x, W_up[e] x),  out = W_down[e] y
//                 act(g, u) = g' sigmoid(alpha g') (u' + shift),  g' = min(g, limit),  u' = clamp(u, -limit, limit)
//                 (an infinite limit, alpha 1 and shift 0: the plain gated unit silu(g) u)
//   P[k][t]     = w[t, k] * expert chosen(t)[k] (x[t])        (float; the caller adds the slices in order)
//                 (experts from the `real`-th on have no weights: they return x[t] itself)
//
// (1) route: a wave a token picks the experts and their weights.  (2) group: the (token, choice) pairs
// are put in the order of their experts (a stable counting sort: a wave an expert counts its pairs by
// ballots, then places them; one workgroup does (1) and (2) for a step of few tokens), and every
// expert's pairs are cut into tiles of ROWS rows; the tile list has a fixed capacity that depends on the sizes only, unused
// tiles are marked.  (3) the gate and up products of every tile with the activation as epilogue; (4)
// the down products, scaled and scattered to P.  Products use the 16x16 MFMA atom with the weight
// rows as first operand (a lane ends with four consecutive output columns of one row); a row's
// contraction is one chain over ascending K from zero, so its bits do not depend on the tile it is in
// or on what else is in the step.  A weight fragment is loaded once and multiplied with all RT row
// tiles of a wave.

#include "common.h"
#include "ring_product.h"

#include <algorithm>
#include <type_traits>

namespace ls {

constexpr int kMaxTop = 16;

__device__ __forceinline__ float sigmoid_e(float x) { return 1.0f / (1.0f + expf(-x)); }

// ---------------------------------------------------------------------------
// (1) A wave a token.  Lane l holds the logits of experts l, l + 64, ...; a pick is the best of every lane's
// best (the larger value, then the lower index), found by exchanges across the wave; lane k < top keeps the
// k-th pick.  expert [T][top] int, weight [T][top] float.
// ---------------------------------------------------------------------------
constexpr int kMaxPerLane = 8;   // experts a lane holds: up to 512 experts

// scoring 0: the weights are the softmax over the chosen logits; 1: each chosen expert weighs the sigmoid of its own
// logit, and nothing is renormalised (the sigmoid grows with the logit, so the largest logits are the largest scores).
// scoring 2: scores s = softmax over all E logits; the choice goes by s + correction, among the experts of the `keep` groups
// (of `groups` equal runs of neighbours) whose largest choice score is largest; the weights are the chosen s divided by
// their sum (+ kShareEps).
constexpr float kShareEps = 1e-20f;

struct Choice {
  int scoring, groups, keep;
  const float* correction;   // [E], scoring 2
};

// A lane's (value, index) against those of the lane that a data-parallel move inside its row of sixteen names; the larger
// value stays, the lower index winning a tie (0x7fffffff: none).
__device__ __forceinline__ void keep_better(float& v, int& e, float ov, int oe) {
  const bool take = oe != 0x7fffffff && (e == 0x7fffffff || ov > v || (ov == v && oe < e));
  v = take ? ov : v;
  e = take ? oe : e;
}
template <int CTRL>
__device__ __forceinline__ void keep_better_of(float& v, int& e) {
  keep_better(v, e, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true)),
              __builtin_amdgcn_mov_dpp(e, CTRL, 0xF, 0xF, true));
}

// A lane's entries of a vector over the experts (null: zeros).
template <int PL>
__device__ __forceinline__ void lane_entries(const float* __restrict__ of, int E, int lane, float (&mine)[PL]) {
#pragma unroll
  for (int m = 0; m < PL; ++m) mine[m] = of && lane + 64 * m < E ? of[lane + 64 * m] : 0.f;
}

// PL: experts a lane holds; bias and correction: their entries
template <int PL>
__device__ __forceinline__ void pick_top(const float* __restrict__ row, const float (&bias)[PL], const float (&correction)[PL],
                                         int E, int top, int lane, int* __restrict__ picked, float* __restrict__ share,
                                         const Choice& how) {
  float mine[PL], score[PL];
#pragma unroll
  for (int m = 0; m < PL; ++m) {
    const int e = lane + 64 * m;
    mine[m] = e < E ? row[e] + bias[m] : 0.f;
    score[m] = 0.f;
  }
  // the largest of every lane's open experts, the lower index winning a tie (0x7fffffff: none is open)
  auto largest = [&](unsigned closed, float& best_v, int& best) LS_INLINED {
    best_v = 0.f;
    best = 0x7fffffff;
#pragma unroll
    for (int m = 0; m < PL; ++m) {
      const int e = lane + 64 * m;
      if (e < E && !((closed >> m) & 1u) && (best == 0x7fffffff || mine[m] > best_v)) {
        best_v = mine[m];
        best = e;
      }
    }
    // pairs, pairs of pairs, the mirror image of the half row and of the row (after each, the lanes that met agree), then
    // the rows of sixteen
    keep_better_of<0xB1>(best_v, best);
    keep_better_of<0x4E>(best_v, best);
    keep_better_of<0x141>(best_v, best);
    keep_better_of<0x140>(best_v, best);
#pragma unroll
    for (int step = 16; step < 64; step <<= 1) keep_better(best_v, best, __shfl_xor(best_v, step, kWave), __shfl_xor(best, step, kWave));
  };
  unsigned taken = 0;
  if (how.scoring == 2) {
    float top_z;
    int at;
    largest(0u, top_z, at);
    float part = 0.f;
#pragma unroll
    for (int m = 0; m < PL; ++m) {
      score[m] = lane + 64 * m < E ? expf(mine[m] - top_z) : 0.f;
      part = part + score[m];
    }
    const float inv = 1.0f / wave_sum(part);
#pragma unroll
    for (int m = 0; m < PL; ++m) {
      score[m] = score[m] * inv;
      if (lane + 64 * m < E) mine[m] = score[m] + correction[m];
    }
    if (how.keep < how.groups) {   // the groups, best first: every pick closes its group for the next one
      const int each = E / how.groups;
      unsigned open = 0;
      for (int g = 0; g < how.keep; ++g) {
        float v;
        int best;
        largest(open, v, best);
#pragma unroll
        for (int m = 0; m < PL; ++m)
          if ((lane + 64 * m) / each == best / each) open |= 1u << m;
      }
      taken = ~open;
    }
  }
  int my_pick = 0;
  float my_value = 0.f, first = 0.f;
  for (int k = 0; k < top; ++k) {
    float best_v;
    int best;
    largest(taken, best_v, best);
    if ((best & 63) == lane) taken |= 1u << (best >> 6);
    if (k == 0) first = best_v;
    if (how.scoring == 2) {   // (the weight is the score without the correction)
      float held = 0.f;
#pragma unroll
      for (int m = 0; m < PL; ++m) held = (best >> 6) == m ? score[m] : held;
      best_v = __shfl(held, best & 63, kWave);
    }
    if (lane == k) {
      my_pick = best;
      my_value = best_v;
    }
  }
  if (how.scoring == 2) {
    const float sum = wave_sum(lane < top ? my_value : 0.f);
    if (lane < top) {
      picked[lane] = my_pick;
      share[lane] = my_value / (sum + kShareEps);
    }
    return;
  }
  const float ex = lane < top ? expf(my_value - first) : 0.f;   // (the first pick is the largest)
  const float sum = wave_sum(ex);
  if (lane < top) {
    picked[lane] = my_pick;
    share[lane] = how.scoring == 1 ? sigmoid_e(my_value) : ex / sum;
  }
}

// The experts of a token come from a table instead of a router: row token_id of table [vocab][top] names them (its
// entries differ), and every one weighs 1 / top.
__global__ __launch_bounds__(256) void route_table_kernel(const int* __restrict__ token_ids, const int* __restrict__ table,
                                                          int n_tokens, int top, int* __restrict__ expert,
                                                          float* __restrict__ weight) {
  const long pair = (long)blockIdx.x * 256 + threadIdx.x;
  if (pair >= (long)n_tokens * top) return;
  expert[pair] = table[(long)token_ids[pair / top] * top + pair % top];
  weight[pair] = 1.0f / (float)top;
}

template <int PL>
__global__ __launch_bounds__(256) void route_topk_kernel(const float* __restrict__ z, long ldz,
                                                         const float* __restrict__ bias, int n_tokens, int E, int top,
                                                         int* __restrict__ expert, float* __restrict__ weight, Choice how) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= n_tokens) return;
  const int lane = threadIdx.x & 63;
  float own_bias[PL], own_correction[PL];
  lane_entries<PL>(bias, E, lane, own_bias);
  lane_entries<PL>(how.correction, E, lane, own_correction);
  pick_top<PL>(z + (long)t * ldz, own_bias, own_correction, E, top, lane, expert + (long)t * top, weight + (long)t * top, how);
}

// ---------------------------------------------------------------------------
// (2) order [P]: the pairs (token * top + choice) sorted by expert, stable.  tiles [cap][4]: expert (-1: unused),
// first place in order, rows, 0.  A wave an expert: it counts its pairs by ballots, adds up the counts of the
// experts before it, writes its tiles and places its pairs.  Many pairs: two launches of a workgroup
// an expert (count; place).  Few: one workgroup that also picks the experts, with the picks and counts in LDS.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int count_pairs(const int* expert, int p0, int p1, int e, int lane) {
  int n = 0;
  for (; p0 < p1; p0 += 512) {   // (eight loads requested together)
    int got[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) got[u] = p0 + 64 * u + lane < p1 ? expert[p0 + 64 * u + lane] : -1;
#pragma unroll
    for (int u = 0; u < 8; ++u) n += __popcll(__ballot(got[u] == e));
  }
  return n;
}

// An expert's first place in the order, and its tiles (those behind the last expert's are marked unused).
__device__ __forceinline__ int place_tiles(const int* counts, int E, int e, int lane, int rows_a_tile, int* __restrict__ tiles,
                                           int cap, bool write) {
  int base = 0, tile = 0;
  for (int j0 = 0; j0 < e; j0 += 64) {   // (sums of whole numbers: any order)
    const int c = j0 + lane < e ? counts[j0 + lane] : 0;
    base += wave_sum(c);
    tile += wave_sum((c + rows_a_tile - 1) / rows_a_tile);
  }
  if (!write) return base;
  const int n = counts[e];
  for (int i = lane; i * rows_a_tile < n; i += 64) {
    if (tile + i < cap) {
      tiles[4 * (tile + i)] = e;
      tiles[4 * (tile + i) + 1] = base + i * rows_a_tile;
      tiles[4 * (tile + i) + 2] = min(rows_a_tile, n - i * rows_a_tile);
      tiles[4 * (tile + i) + 3] = 0;
    }
  }
  if (e == E - 1) {
    const int used = tile + (n + rows_a_tile - 1) / rows_a_tile;
    for (int i = used + lane; i < cap; i += 64) {
      tiles[4 * i] = -1;
      tiles[4 * i + 1] = tiles[4 * i + 2] = tiles[4 * i + 3] = 0;
    }
  }
  return base;
}

// The pairs [p0, p1) that expert e has go to order[at], order[at + 1], ...
__device__ __forceinline__ void place_pairs(const int* expert, int p0, int p1, int e, int lane, int at, int* __restrict__ order) {
  for (; p0 < p1; p0 += 256) {
    int got[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) got[u] = p0 + 64 * u + lane < p1 ? expert[p0 + 64 * u + lane] : -1;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool mine = got[u] == e;
      const unsigned long long votes = __ballot(mine);
      if (mine) order[at + __popcll(votes & ((1ull << lane) - 1ull))] = p0 + 64 * u + lane;
      at += __popcll(votes);
    }
  }
}

// Many pairs: a workgroup an expert, whose waves take equal shares of the pairs.  What bounds both launches is the
// latency of reading the picks, so the reads are spread over up to sixteen waves; the second counts a wave's share again,
// because the place of a share follows from the shares before it.  8,192 pairs of 32 experts: 5.0 us to count and 5.1 to
// place, where one wave an expert took 12.2 and 12.7.
__device__ __forceinline__ int my_share(int P, int w, int& p1) {
  const int group = blockDim.x;  // 64 pairs a wave
  const int share = (P + group - 1) / group * 64, p0 = min(w * share, P);
  p1 = min(p0 + share, P);
  return p0;
}
// Waves an expert: one for every 256 pairs.  (Sixteen from 513 pairs on crowd the card where there are many experts: the whole
// routing of 520 pairs by 512 experts took 17.4 us, one wave an expert 14.8, so 14.7; of 1,024 pairs by 64 experts 9.7, 10.0, 9.4.)
static int route_waves(int P) { return P >= 16 * 256 ? 16 : (P + 255) / 256; }

__global__ __launch_bounds__(1024) void route_count_kernel(const int* __restrict__ expert, int P, int* __restrict__ counts) {
  __shared__ int mine_s[16];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int p1;
  const int p0 = my_share(P, w, p1);
  const int n = count_pairs(expert, p0, p1, blockIdx.x, lane);
  if (lane == 0) mine_s[w] = n;
  __syncthreads();
  if (threadIdx.x == 0) {
    int sum = 0;
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) sum += mine_s[i];
    counts[blockIdx.x] = sum;
  }
}

__global__ __launch_bounds__(1024) void route_place_kernel(const int* __restrict__ expert, const int* __restrict__ counts,
                                                           int P, int E, int rows_a_tile, int* __restrict__ order,
                                                           int* __restrict__ tiles, int cap) {
  __shared__ int mine_s[16];
  const int e = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int p1;
  const int p0 = my_share(P, w, p1);
  const int n = count_pairs(expert, p0, p1, e, lane);
  if (lane == 0) mine_s[w] = n;
  int at = place_tiles(counts, E, e, lane, rows_a_tile, tiles, cap, w == 0);
  __syncthreads();
  for (int i = 0; i < w; ++i) at += mine_s[i];
  place_pairs(expert, p0, p1, e, lane, at, order);
}

// A barrier between LDS writes and reads that waits for this wave's LDS operations only: loads from memory (and stores
// to it) stay on their way across it.
__device__ __forceinline__ void lds_barrier() { __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

constexpr int kSmallPairs = 512, kSmallExperts = 512;   // what the one-workgroup kernel keeps in LDS

constexpr int kProductTiles = 8;    // tiles of 16 experts whose logits the one-workgroup kernel forms itself

// PRODUCT: the logits come from up to 16 rows of x and the router's matrix [E][K] instead of z
template <int PL, typename T, bool PRODUCT>
__global__ __launch_bounds__(1024) void route_small_kernel(const float* __restrict__ z, long ldz,
                                                           const float* __restrict__ bias, int n_tokens, int E, int top,
                                                           int rows_a_tile, int* __restrict__ expert,
                                                           float* __restrict__ weight, int* __restrict__ order,
                                                           int* __restrict__ tiles, int cap,
                                                           const int* __restrict__ token_ids, const int* __restrict__ table,
                                                           Choice how, const T* __restrict__ x, long ldx,
                                                           const T* __restrict__ w_router, int K) {
  __shared__ int picks_s[kSmallPairs];
  __shared__ float share_s[kSmallPairs];
  __shared__ int counts_s[kSmallExperts];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int P = n_tokens * top;
  float own_bias[PL], own_correction[PL];
  lane_entries<PL>(bias, E, lane, own_bias);
  lane_entries<PL>(how.correction, E, lane, own_correction);
  if constexpr (PRODUCT) {   // the logits first: z = x W^T, the column tiles and cuts of K dealt to the sixteen waves
    __shared__ f32x4 sums_s[16][64];
    __shared__ float z_s[16][16 * kProductTiles];
    constexpr int VEC = Atom<T>::VEC, KC = Atom<T>::KCHUNK, U = 8;
    const int l16 = lane & 15, quad = lane >> 4;
    const int tiles16 = (E + 15) / 16, cuts = 16 / tiles16;
    const int ct = w % tiles16, cut = w / tiles16;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (cut < cuts) {
      const bool w_ok = 16 * ct + l16 < E, x_ok = l16 < n_tokens;
      const T* w_row = w_router + (long)(w_ok ? 16 * ct + l16 : 0) * K;
      const T* x_row = x + (long)(x_ok ? l16 : 0) * ldx;
      const int each = (K + KC * cuts - 1) / (KC * cuts) * KC;
      const int hi = min(K, (cut + 1) * each);
      for (int k0 = cut * each; k0 < hi; k0 += U * KC) {
        typename Atom<T>::vec_t a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          a[u] = load_vec<T>(w_row, 0, k0 + u * KC + VEC * quad, hi, 0, w_ok, true);
          b[u] = load_vec<T>(x_row, 0, k0 + u * KC + VEC * quad, hi, 0, x_ok, true);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) Atom<T>::mma(acc, a[u], b[u]);
      }
    }
    sums_s[w][lane] = acc;
    lds_barrier();
    if (w < tiles16) {   // (the cuts in ascending order)
      f32x4 sum = sums_s[w][lane];
      for (int o = 1; o < cuts; ++o) sum = sum + sums_s[w + o * tiles16][lane];
#pragma unroll
      for (int i = 0; i < 4; ++i) z_s[l16][16 * w + 4 * quad + i] = sum[i];
    }
    lds_barrier();
    z = &z_s[0][0];
    ldz = 16 * kProductTiles;
  }
  if (table) {   // the picks are looked up, not chosen
    for (int pair = threadIdx.x; pair < P; pair += 1024) {
      picks_s[pair] = table[(long)token_ids[pair / top] * top + pair % top];
      share_s[pair] = 1.0f / (float)top;
    }
  }
  for (int t = w; t < n_tokens && !table; t += 16)
    pick_top<PL>(z + (long)t * ldz, own_bias, own_correction, E, top, lane, picks_s + t * top, share_s + t * top, how);
  lds_barrier();
  for (int pair = threadIdx.x; pair < P; pair += 1024) {
    expert[pair] = picks_s[pair];
    weight[pair] = share_s[pair];
  }
  for (int e = w; e < E; e += 16) {
    const int n = count_pairs(picks_s, 0, P, e, lane);
    if (lane == 0) counts_s[e] = n;
  }
  lds_barrier();
  for (int e = w; e < E; e += 16)
    place_pairs(picks_s, 0, P, e, lane, place_tiles(counts_s, E, e, lane, rows_a_tile, tiles, cap, true), order);
}

// ---------------------------------------------------------------------------
// (3) act [P][ldy] (T) = act(x[token] W_gate[e]^T, x[token] W_up[e]^T) for the pairs of every tile, in the
// order of `order`.  w_gate, w_up [E][F][K].  A workgroup: one tile, four waves with 16 columns of F each.
// ---------------------------------------------------------------------------
// An expert that every token uses, worked on beside the routed ones in the launches of small steps: work items from `at`
// on are tiles of 16 tokens.  w_gate_up holds its rows interleaved in tiles of 16 (gate, up, gate, ...; the last tile padded
// with zeros), w_down [N][F]; the plain gated unit silu(g) u; act [n_tokens][ldy] scratch, out [n_tokens][N] float.
template <typename T>
struct SharedExpert {
  const T* w_gate_up;
  const T* w_down;
  int F, at;   // at: the routed experts' work items (0x7fffffff: there is no such expert)
  T* act;
  long ldy;
  float* out;
};

template <typename T, int RT, int KS>
__global__ __launch_bounds__(256) void experts_gate_up_kernel(const T* __restrict__ x, long ldx,
                                                              const T* __restrict__ w_gate, const T* __restrict__ w_up,
                                                              int F, int K, int top, const int* __restrict__ order,
                                                              const int* __restrict__ tiles, float limit, float alpha, float shift,
                                                              const float* __restrict__ in_weight, T* __restrict__ act, long ldy,
                                                              int real, int n_tokens, SharedExpert<T> sh) {
  // in_weight (or null): a pair's routing weight multiplies the expert's input, w * x, so both products are scaled
  // by it before the gated unit (the down product then adds the expert's output as it is)
  constexpr int VEC = Atom<T>::VEC, KC = Atom<T>::KCHUNK;
  const bool all = KS > 1 && (int)blockIdx.x >= sh.at;   // (the same for the whole workgroup)
  const int e = all ? 0 : tiles[4 * blockIdx.x];
  if (e < 0 || e >= real) return;   // (an expert that returns its input has nothing to multiply)
  const int first = all ? 16 * ((int)blockIdx.x - sh.at) : tiles[4 * blockIdx.x + 1];
  const int rows = all ? min(16, n_tokens - first) : tiles[4 * blockIdx.x + 2];
  if (all) F = sh.F;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int l16 = lane & 15, quad = lane >> 4;
  // KS 1: the four waves take 16 columns each.  KS 4 (few rows): they take a quarter of K each for the same 16
  // columns, so that all of a wave's operands are on their way at once, and their sums are added in wave order.
  const int col0 = KS == 1 ? (blockIdx.y * 4 + w) * 16 : blockIdx.y * 16;
  if (col0 >= F) return;
  const bool w_ok = all || col0 + l16 < F;
  const T* g_row = all ? sh.w_gate_up + (long)(2 * col0 + l16) * K : w_gate + ((long)e * F + (w_ok ? col0 + l16 : 0)) * K;
  const T* u_row = all ? g_row + 16L * K : w_up + ((long)e * F + (w_ok ? col0 + l16 : 0)) * K;
  const T* x_row[RT];
  bool x_ok[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    x_ok[r] = 16 * r + l16 < rows;
    const int token = all ? first + l16 : (x_ok[r] ? order[first + 16 * r + l16] : 0) / top;
    x_row[r] = x + (long)(x_ok[r] ? token : 0) * ldx;
  }
  f32x4 acc_g[RT], acc_u[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) acc_g[r] = acc_u[r] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool aligned = K % VEC == 0;
  // the operands of U chunks are requested together, then multiplied in ascending order
  constexpr int U = RT == 1 ? 8 : 4;
  const int k_each = KS == 1 ? K : (K + KC * KS - 1) / (KC * KS) * KC;
  const int k_lo = KS == 1 ? 0 : w * k_each, k_hi = KS == 1 ? K : min(K, k_lo + k_each);
  for (int k0 = k_lo; k0 < k_hi; k0 += U * KC) {
    typename Atom<T>::vec_t a_g[U], a_u[U], b[U][RT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * KC + VEC * quad;
      a_g[u] = load_vec<T>(g_row, 0, k, k_hi, 0, w_ok, aligned);
      a_u[u] = load_vec<T>(u_row, 0, k, k_hi, 0, w_ok, aligned);
#pragma unroll
      for (int r = 0; r < RT; ++r) b[u][r] = load_vec<T>(x_row[r], 0, k, k_hi, 0, x_ok[r], aligned);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        Atom<T>::mma(acc_g[r], a_g[u], b[u][r]);
        Atom<T>::mma(acc_u[r], a_u[u], b[u][r]);
      }
  }
  if constexpr (KS > 1) {
    __shared__ f32x4 sums_s[KS][2][RT][64];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      sums_s[w][0][r][lane] = acc_g[r];
      sums_s[w][1][r][lane] = acc_u[r];
    }
    __syncthreads();
    if (w != 0) return;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int o = 1; o < KS; ++o)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc_g[r][i] = acc_g[r][i] + sums_s[o][0][r][lane][i];
          acc_u[r][i] = acc_u[r][i] + sums_s[o][1][r][lane][i];
        }
  }
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    if (!x_ok[r]) continue;
    T* dst = all ? sh.act + (long)(first + l16) * sh.ldy : act + (long)(first + 16 * r + l16) * ldy;
    const float wt = in_weight && !all ? in_weight[order[first + 16 * r + l16]] : 1.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = col0 + 4 * quad + i;
      if (c < F) {
        if (all) {
          dst[c] = from_f32<T>((acc_g[r][i] * sigmoid_e(acc_g[r][i])) * acc_u[r][i]);
          continue;
        }
        const float g = fminf(acc_g[r][i] * wt, limit);
        const float u = fminf(fmaxf(acc_u[r][i] * wt, -limit), limit);
        dst[c] = from_f32<T>((g * sigmoid_e(alpha * g)) * (u + shift));
      }
    }
  }
}

// A tile of an expert that returns its input: P[choice][token][c] = share * x[token][c] for the columns [c0, c1), the
// routing weight multiplying the input or the output alike.  THREADS: those of the workgroup, each element one thread's.
template <typename T, int THREADS>
__device__ __forceinline__ void pass_input(const T* __restrict__ x, long ldx, const float* __restrict__ share, int first, int rows,
                                           int c0, int c1, int top, int n_tokens, int N, const int* __restrict__ order,
                                           float* __restrict__ P) {
  const int width = c1 - c0;
  for (int i = threadIdx.x; i < rows * width; i += THREADS) {
    const int pair = order[first + i / width], c = c0 + i % width;
    P[((long)(pair % top) * n_tokens + pair / top) * N + c] = share[pair] * to_f32(x[(long)(pair / top) * ldx + c]);
  }
}

// ---------------------------------------------------------------------------
// (4) P[choice][token][:] = weight[pair] * (act[place] W_down[e]^T).  w_down [E][N][F]; P [top][n_tokens][N] float.
// ---------------------------------------------------------------------------
template <typename T, int RT, int KS>
__global__ __launch_bounds__(256) void experts_down_kernel(const T* __restrict__ act, long ldy,
                                                           const T* __restrict__ w_down, int N, int F, int top,
                                                           int n_tokens, const int* __restrict__ order,
                                                           const int* __restrict__ tiles,
                                                           const float* __restrict__ weight, float* __restrict__ P,
                                                           const T* __restrict__ x, long ldx, const float* __restrict__ share,
                                                           int real, SharedExpert<T> sh) {
  constexpr int VEC = Atom<T>::VEC, KC = Atom<T>::KCHUNK;
  const bool all = KS > 1 && (int)blockIdx.x >= sh.at;
  const int e = all ? 0 : tiles[4 * blockIdx.x];
  if (e < 0) return;
  const int first = all ? 16 * ((int)blockIdx.x - sh.at) : tiles[4 * blockIdx.x + 1];
  const int rows = all ? min(16, n_tokens - first) : tiles[4 * blockIdx.x + 2];
  if (all) {
    F = sh.F;
    ldy = sh.ldy;
    act = sh.act;
    w_down = sh.w_down;
  }
  if (e >= real) {   // (the whole workgroup)
    constexpr int kCols = KS == 1 ? 64 : 16;
    pass_input<T, 256>(x, ldx, share, first, rows, blockIdx.y * kCols, min(N, (int)(blockIdx.y + 1) * kCols), top, n_tokens, N, order, P);
    return;
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int l16 = lane & 15, quad = lane >> 4;
  const int col0 = KS == 1 ? (blockIdx.y * 4 + w) * 16 : blockIdx.y * 16;
  if (col0 >= N) return;
  const bool w_ok = col0 + l16 < N;
  const T* d_row = w_down + ((long)e * N + (w_ok ? col0 + l16 : 0)) * F;
  const T* y_row[RT];
  bool y_ok[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    y_ok[r] = 16 * r + l16 < rows;
    y_row[r] = act + (long)(first + (y_ok[r] ? 16 * r + l16 : 0)) * ldy;
  }
  f32x4 acc[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool aligned = F % VEC == 0 && ldy % VEC == 0;
  constexpr int U = RT == 1 ? 8 : 4;
  const int k_each = KS == 1 ? F : (F + KC * KS - 1) / (KC * KS) * KC;
  const int k_lo = KS == 1 ? 0 : w * k_each, k_hi = KS == 1 ? F : min(F, k_lo + k_each);
  for (int k0 = k_lo; k0 < k_hi; k0 += U * KC) {
    typename Atom<T>::vec_t a[U], b[U][RT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * KC + VEC * quad;
      a[u] = load_vec<T>(d_row, 0, k, k_hi, 0, w_ok, aligned);
#pragma unroll
      for (int r = 0; r < RT; ++r) b[u][r] = load_vec<T>(y_row[r], 0, k, k_hi, 0, y_ok[r], aligned);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int r = 0; r < RT; ++r) Atom<T>::mma(acc[r], a[u], b[u][r]);
  }
  if constexpr (KS > 1) {
    __shared__ f32x4 sums_s[KS][RT][64];
#pragma unroll
    for (int r = 0; r < RT; ++r) sums_s[w][r][lane] = acc[r];
    __syncthreads();
    if (w != 0) return;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int o = 1; o < KS; ++o)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[r][i] = acc[r][i] + sums_s[o][r][lane][i];
  }
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    if (!y_ok[r]) continue;
    const int pair = all ? 0 : order[first + 16 * r + l16];
    const float factor = weight && !all ? weight[pair] : 1.0f;
    float* dst = all ? sh.out + (long)(first + l16) * N : P + ((long)(pair % top) * n_tokens + pair / top) * N;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = col0 + 4 * quad + i;
      if (c < N) dst[c] = factor * acc[r][i];
    }
  }
}

// ---------------------------------------------------------------------------
// The same two products for tiles of 16 rows where the sizes are whole chunks (`few_chunks`): decode steps, whose weights are
// read once, by workgroups of 16 columns with a quarter of K a wave.  What bounds them is the weights (a CU keeps some 64 KB on
// their way, so all of its workgroups' should be asked for at once) and, in front of those, the chain of what a workgroup has to
// look up.  So: one load of the tile's entry, then every weight of the wave's quarter (U chunks at a time) in one batch,
// without a branch, then the rows that the order names; registers for four workgroups a CU.  The kernels above, which take any
// size, have a branch in front of every operand.  Both launches, 4 of 32 experts, width 1,024, 768 a piece, weights from HBM, us by the
// kernels above / these (bytes at 5.96 TB/s): 1 token 10.9 / 8.6 (3.2), 8 tokens 31.7 / 26.9 (18.2), 40 tokens 42.3 / 34.5 (25.3);
// 8 tokens of width 2,048, 1,024 a piece 69 / 61 (49); float32 8 tokens 96 / 54 (36), of width 2,048 238 / 130 (97).
// The same sums in the same order as the kernels above give with a cut of K: the same bits.
//
// A table that names the experts, and at most 64 pairs in the step: a workgroup then stands for an expert (and sixteen of its
// rows), or for a pair where there are fewer of those, and works if that is the first of sixteen of its expert's
// (`table_groups`).  Each of its waves finds the rows by itself: lane l has pair l's expert, ballots give the expert's pairs and how many
// lie in front of them.  The launch that would put the pairs in order is saved.  The first product looks the experts up (a table's
// rows come from HBM, which takes as long as that launch did) and leaves them for the second one.  Whole requests of the design that is
// measured (28 layers, eight decode): 74.3 ms with the launch, 75.0 with an expert's blocks all on one XCD, 72.8 spread over the eight,
// 71.9 with two column tiles in the second product.
// ---------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(4))) int i32x4_t;
constexpr int kTablePairs = 64;
enum RowsFrom : int {
  kListed,  // tiles and order
  kTable,   // token ids and the table
  kPicked,  // the pairs' experts
};

// Sixteen rows of an expert: its first place among the pairs in the order of their experts, how many, and the pair of this lane's row
// (l % 16; lanes past the last row repeat it).
struct FewRows {
  int expert, first, rows, pair;
};
// at, more: tiles and order; token ids and table; the picks.  picks: where workgroup (0, 0) leaves what the table named.
template <int FROM>
__device__ __forceinline__ FewRows few_rows(const int* __restrict__ at, const int* __restrict__ more, int top, int n_tokens, int E,
                                            int (*places_s)[kTablePairs], int* __restrict__ picks) {
  const int lane = threadIdx.x & 63, l16 = lane & 15;
  if constexpr (FROM == kListed) {
    const i32x4_t tile = reinterpret_cast<const i32x4_t*>(at)[blockIdx.x];
    const int rows = tile[2];
    return {tile[0], tile[1], rows, tile[0] < 0 ? 0 : more[tile[1] + min(l16, rows - 1)]};
  } else {
    // (workgroups go round the eight XCDs: an expert's column blocks shift from one to the next, or one XCD would have all of them)
    const int at_x = ((int)blockIdx.x + (int)blockIdx.y) % (int)gridDim.x, P = n_tokens * top;
    int mine = 0x7fffffff;
    if (lane < P) mine = FROM == kTable ? more[(long)at[lane / top] * top + lane % top] : at[lane];
    if (FROM == kTable && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < P) picks[threadIdx.x] = mine;  // (its first wave)
    const bool by_pair = (long)gridDim.x < (long)E * ((n_tokens + 15) / 16);  // table_groups
    const int e = by_pair ? __builtin_amdgcn_readlane(mine, at_x) : at_x % E;
    const unsigned long long held = __ballot(mine == e);
    const int skip = by_pair ? __popcll(held & ((1ull << at_x) - 1ull)) : 16 * (at_x / E);
    const int n = __popcll(held) - skip, first = __popcll(__ballot(mine < e)) + skip;
    if (n <= 0 || skip % 16 != 0) return {-1, 0, 0, 0};  // uniform
    int* places = places_s[threadIdx.x >> 6];  // (the wave's own)
    if (mine == e) places[__popcll(held & ((1ull << lane) - 1ull))] = lane;
    // (other lanes read what this one wrote: the barrier orders instructions, the fences the memory between them)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int rows = min(16, n);
    return {e, first, rows, places[skip + min(l16, rows - 1)]};
  }
}

template <typename T, int U, int FROM>
__global__ __launch_bounds__(256, 4) void experts_few_gate_up_kernel(const int* __restrict__ at, const T* __restrict__ w_gate,
                                                                     const T* __restrict__ w_up, const int* __restrict__ more,
                                                                     const T* __restrict__ x, long ldx, int F, int K, int top,
                                                                     int real, float limit, float alpha, float shift,
                                                                     const float* __restrict__ in_weight, T* __restrict__ act,
                                                                     long ldy, int n_tokens, int E, int* __restrict__ picks) {
  typedef typename Atom<T>::vec_t vec_t;
  constexpr int VEC = Atom<T>::VEC, KC = Atom<T>::KCHUNK, KS = 4;
  __shared__ int places_s[FROM == kListed ? 1 : KS][kTablePairs];
  const FewRows mine = few_rows<FROM>(at, more, top, n_tokens, E, places_s, picks);
  const int e = mine.expert, first = mine.first, rows = mine.rows, pair = mine.pair;
  if (e < 0 || e >= real) return;  // (an expert that returns its input has nothing to multiply)
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, quad = lane >> 4;
  const int col0 = blockIdx.y * 16;
  const int k_each = K / KS;
  const long from = ((long)e * F + col0 + l16) * K + w * k_each + VEC * quad;
  const T *g = w_gate + from, *u = w_up + from;
  f32x4 acc_g = f32x4{0.f, 0.f, 0.f, 0.f}, acc_u = acc_g;
  vec_t a_g[U], a_u[U];
  auto request = [&](int k0) LS_INLINED {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < U; ++i) {
      a_g[i] = *reinterpret_cast<const vec_t*>(g + k0 + i * KC);
      a_u[i] = *reinterpret_cast<const vec_t*>(u + k0 + i * KC);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  request(0);  // before the order's entry is waited for
  const T* xr = x + (long)(pair / top) * ldx + w * k_each + VEC * quad;
  for (int k0 = 0;;) {
    vec_t b[U];
#pragma unroll
    for (int i = 0; i < U; ++i) b[i] = *reinterpret_cast<const vec_t*>(xr + k0 + i * KC);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < U; ++i) {
      Atom<T>::mma(acc_g, a_g[i], b[i]);
      Atom<T>::mma(acc_u, a_u[i], b[i]);
    }
    k0 += U * KC;
    if (k0 >= k_each) break;
    request(k0);
  }
  const float wt = in_weight ? in_weight[pair] : 1.0f;
  __shared__ f32x4 sums_s[KS - 1][2][64];
  if (w > 0) {
    sums_s[w - 1][0][lane] = acc_g;
    sums_s[w - 1][1][lane] = acc_u;
  }
  __syncthreads();
  if (w != 0 || l16 >= rows) return;
#pragma unroll
  for (int o = 0; o < KS - 1; ++o)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc_g[i] = acc_g[i] + sums_s[o][0][lane][i];
      acc_u[i] = acc_u[i] + sums_s[o][1][lane][i];
    }
  T* dst = act + (long)(first + l16) * ldy + col0 + 4 * quad;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float gv = fminf(acc_g[i] * wt, limit);
    const float uv = fminf(fmaxf(acc_u[i] * wt, -limit), limit);
    dst[i] = from_f32<T>((gv * sigmoid_e(alpha * gv)) * (uv + shift));
  }
}

// COLS: tiles of 16 columns a workgroup.  Two where its waves have to find their rows and a weight has two bytes (8 tokens, some 21 of 32
// experts, 1,024 x 768 10.9 -> 10.4 us in the decode step); with a list one is the faster (both launches 26.9 / 28.1, float32 54 / 60).
template <typename T, int U, int FROM, int COLS>
__global__ __launch_bounds__(256, 4) void experts_few_down_kernel(const int* __restrict__ at, const T* __restrict__ w_down,
                                                                  const T* __restrict__ act, long ldy,
                                                                  const int* __restrict__ more,
                                                                  const float* __restrict__ weight, float* __restrict__ P, int N,
                                                                  int F, int top, int n_tokens, int real, const T* __restrict__ x,
                                                                  long ldx, const float* __restrict__ share, int E) {
  typedef typename Atom<T>::vec_t vec_t;
  constexpr int VEC = Atom<T>::VEC, KC = Atom<T>::KCHUNK, KS = 4;
  __shared__ int places_s[FROM == kListed ? 1 : KS][kTablePairs];
  const FewRows mine = few_rows<FROM>(at, more, top, n_tokens, E, places_s, nullptr);
  const int e = mine.expert, first = mine.first, rows = mine.rows, pair = mine.pair;
  if (e < 0) return;
  const int col0 = blockIdx.y * 16 * COLS;
  if (FROM == kListed && e >= real) {  // (the whole workgroup)
    pass_input<T, 256>(x, ldx, share, first, rows, col0, col0 + 16 * COLS, top, n_tokens, N, more, P);
    return;
  }
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, quad = lane >> 4;
  const int k_each = F / KS;
  const T* d = w_down + ((long)e * N + col0 + l16) * F + w * k_each + VEC * quad;
  const T* y = act + (long)(first + min(l16, rows - 1)) * ldy + w * k_each + VEC * quad;
  f32x4 acc[COLS];
#pragma unroll
  for (int c = 0; c < COLS; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < k_each; k0 += U * KC) {
    vec_t a[COLS][U], b[U];
#pragma unroll
    for (int c = 0; c < COLS; ++c)
#pragma unroll
      for (int i = 0; i < U; ++i) a[c][i] = *reinterpret_cast<const vec_t*>(d + (long)(16 * c) * F + k0 + i * KC);
#pragma unroll
    for (int i = 0; i < U; ++i) b[i] = *reinterpret_cast<const vec_t*>(y + k0 + i * KC);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < U; ++i)
#pragma unroll
      for (int c = 0; c < COLS; ++c) Atom<T>::mma(acc[c], a[c][i], b[i]);
  }
  const float factor = FROM != kListed ? 1.0f / (float)top : weight ? weight[pair] : 1.0f;
  __shared__ f32x4 sums_s[KS - 1][COLS][64];
  if (w > 0) {
#pragma unroll
    for (int c = 0; c < COLS; ++c) sums_s[w - 1][c][lane] = acc[c];
  }
  __syncthreads();
  if (w != 0 || l16 >= rows) return;
  float* dst = P + ((long)(pair % top) * n_tokens + pair / top) * N + col0 + 4 * quad;
#pragma unroll
  for (int c = 0; c < COLS; ++c) {
#pragma unroll
    for (int o = 0; o < KS - 1; ++o)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[c][i] = acc[c][i] + sums_s[o][c][lane][i];
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[16 * c + i] = factor * acc[c][i];
  }
}

// Chunks that a wave of those kernels asks for at a time where K is a whole number of such rounds, else 0.  (Rounds of eight, six and four, for
// both products of an expert: what was built and measured, ahead at widths of 512 to 8,192.  Widths that only other rounds divide, 640, 896, 1,280 or
// 1,408 say, keep the kernels for any size in both, and the launch that orders the pairs: other rounds were not tried, nor one product by each.)
static int few_chunks(int dtype, int K) {
  const int quarter = 4 * (dtype == kF32 ? Atom<float>::KCHUNK : Atom<bf16_t>::KCHUNK);
  if (K % quarter != 0) return 0;
  for (int u : {8, 6, 4})
    if (K / quarter % u == 0) return u;
  return 0;
}

// ---------------------------------------------------------------------------
// The same two products for tiles of 64 rows (many tokens an expert), both operands through rings of three stages in LDS
// (ring_product.h).  Eight waves, NWM along the rows by NWN along the weights, take 64 rows by WEIGHTS weight rows: half of them gate rows
// and half the up rows of the same columns, which lie in LDS in tiles of 16 in turn, or columns of the down product; two workgroups share a
// CU.  A row's contraction is one chain over ascending chunks from zero: the same bits as the kernels above give without a cut of K.
// What bounds it: the loads, most of them answered by L2 once neighbouring tiles of an expert share one (below).  Measured (2,048
// tokens with 4 of 32 experts, width 1,024, 768 a piece, us, before / now): in a prompt gate and up 62 / 55 (470 TFLOP/s), down 51 / 38; both products
// alone, one call behind the other, weights from HBM, 122 / 100, of 520, 1,024 and 4,096 tokens 62 / 52, 82 / 67, 198 / 167, of 2,048 tokens of
// 4,096 and 1,536 a piece 613 / 581.  Two thirds of that are the units of tiles, a third is the loop's order.  Other shapes, gate and up / down of the
// first, alone (51 / 31 so): 64 x 256 68 / 36, five stages 70 / 38 (one workgroup a CU), 128 rows x 256 47 to 59 / 34, x 192 50; 128 rows are ahead
// for wide experts (441 for the 581).
// ---------------------------------------------------------------------------
template <typename T, int WEIGHTS, int NWM, int NWN>
struct ExpertTile {
  static constexpr int ROWS = 64, S = 3;
  static constexpr int NW = NWM * NWN, TI = WEIGHTS / (16 * NWN), TJ = ROWS / (16 * NWM);
  static constexpr int LW = WEIGHTS / (8 * NW), LX = ROWS / (8 * NW);  // a wave's loads a stage: eight rows each
  static_assert(LW * 8 * NW == WEIGHTS && LX * 8 * NW == ROWS && TI * 16 * NWN == WEIGHTS && TJ * 16 * NWM == ROWS, "tile shape");
  typedef RingProduct<T, TI, TJ, 2048, WEIGHTS, ROWS, LW, LX, S, S, 1, false> Product;
  static constexpr int kLds = Product::LDS_BYTES, kThreads = 64 * NW;
  Product product;

  static __device__ __forceinline__ int wave() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }
  // the row of this lane's outputs of row tile j, and the first of its four weight rows of weight tile i, inside the tile
  static __device__ __forceinline__ int row_of(int j) { return (wave() / NWN) * (ROWS / NWM) + j * 16 + (threadIdx.x & 15); }
  static __device__ __forceinline__ int weight_of(int i) {
    return (wave() % NWN) * (WEIGHTS / NWN) + i * 16 + ((threadIdx.x & 63) >> 4) * 4;
  }
  // the row of the tile that this lane loads in the wave's load i, of either operand
  static __device__ __forceinline__ int loaded_row(int i) { return (i * NW + wave()) * 8 + ((threadIdx.x & 63) >> 3); }

  // x_at[i]: the bytes from the start of x to row loaded_row(i) of the tile (~0: no such row); w: the buffer that this wave's
  // weights come from, w_row(i): the row in it that load i begins with
  template <typename WeightRow>
  __device__ __forceinline__ void run(u32x4_t x, const unsigned (&x_at)[LX], u32x4_t w, WeightRow w_row, int K, unsigned char* ring) {
    const int lane = threadIdx.x & 63;
    const unsigned piece = ((lane & 7) ^ (lane >> 3)) * 16;
    const unsigned w_off = (unsigned)((lane >> 3) * (long)K * sizeof(T)) + piece;
    const unsigned lds0 = (unsigned)(unsigned long)(__attribute__((address_space(3))) void*)ring + wave() * 1024;
    const int limit = K * (int)sizeof(T) - (int)piece;  // bytes of a row from this lane's piece on
    const int stages = (K + 128 / (int)sizeof(T) - 1) / (128 / (int)sizeof(T));
    auto request_w = [&](int st, int buf, int n) LS_INLINED {
      const int k = st * 128;
      buffer_to_lds16(k < limit ? w_off + k + (unsigned)((long)w_row(n) * K * sizeof(T)) : kNothing, w,
                      lds0 + buf * Product::W_BYTES + n * NW * 1024);
    };
    auto request_x = [&](int st, int buf, int n) LS_INLINED {
      const int k = st * 128;
      buffer_to_lds16(k < limit && x_at[n] != kNothing ? x_at[n] + k + piece : kNothing, x,
                      lds0 + S * Product::W_BYTES + buf * Product::X_BYTES + n * NW * 1024);
    };
    product.run(ring + (wave() % NWN) * (WEIGHTS / NWN) * 128, ring + S * Product::W_BYTES + (wave() / NWN) * (ROWS / NWM) * 128, stages,
                stages, request_w, request_x, [](int) LS_INLINED {});
  }
};

// Columns of the down product a workgroup.  float32 is bound by the matrix cores of the CUs that have a workgroup, so
// narrow tiles, of which there are more, are never slower.
template <typename T>
constexpr int kDownCols = sizeof(T) == 4 ? 64 : 128;

// Workgroups go round the eight XCDs: units of four tiles (mostly one expert's) by four columns stay on one, so that a unit's rows
// and weights are read from beyond an L2 once.  How many of the cap tiles are used nobody knows here: the units go round the XCDs in
// turn, which leaves an XCD at most one unit behind another (whole runs of tiles an XCD, 20 tiles by 11 columns: 47 us for 32; gate and up
// above with units of one, two and four tiles by all columns 70, 56, 56, of four by two, four and eight columns 55, 51, 63).  float32, bound by
// the CUs that have a workgroup, evens them out with units of two by two (2,048 tokens with 2 of 16 experts, width 256, 128 a piece, both products
// 29.7 / 22.1; 260 with 2 of 2, 7,168 and 2,048 631 / 602; others within 2 %).
// False: no such tile.
template <typename T>
constexpr int kUnit = sizeof(T) == 4 ? 2 : 4;  // tiles, and columns
template <int U>
__device__ __forceinline__ bool tile_and_column(int columns, int cap, int& tile, int& column) {
  const int at = blockIdx.x >> 3, unit = at / (U * U) * 8 + (blockIdx.x & 7), in_unit = at % (U * U);
  const int across = (columns + U - 1) / U;
  tile = unit / across * U + in_unit % U;
  column = unit % across * U + in_unit / U;
  return tile < cap && column < columns;
}
template <int U>
static long tile_grid(int columns, int cap) {
  const long units = (long)((cap + U - 1) / U) * ((columns + U - 1) / U);
  return (units + 7) / 8 * 8 * U * U;
}

template <typename T, int WEIGHTS, int NWM, int NWN>
__global__ __launch_bounds__(64 * NWM * NWN) void experts_gate_up_ring_kernel(const T* __restrict__ x, long ldx,
                                                                   const T* __restrict__ w_gate,
                                                                   const T* __restrict__ w_up, int F, int K, int top,
                                                                   const int* __restrict__ order,
                                                                   const int* __restrict__ tiles, int cap, float limit, float alpha,
                                                                   float shift, const float* __restrict__ in_weight,
                                                                   T* __restrict__ act, long ldy, int real, int n_tokens) {
  typedef ExpertTile<T, WEIGHTS, NWM, NWN> Tile;
  static_assert(Tile::TI % 2 == 0, "a wave holds the gate and the up tile of its columns");
  static_assert(Tile::NW % 4 == 0, "all loads of a wave are of gate rows, or all of up rows");
  extern __shared__ __attribute__((aligned(1024))) unsigned char ring[];
  constexpr int COLS = WEIGHTS / 2;
  int tile, column;
  if (!tile_and_column<kUnit<T>>((F + COLS - 1) / COLS, cap, tile, column)) return;
  const int e = tiles[4 * tile];
  if (e < 0 || e >= real) return;
  const int first = tiles[4 * tile + 1], rows = tiles[4 * tile + 2];
  const int col0 = column * COLS;
  const int wave = Tile::wave();
  unsigned x_at[Tile::LX];
#pragma unroll
  for (int i = 0; i < Tile::LX; ++i) {
    const int r = Tile::loaded_row(i);
    x_at[i] = r < rows ? (unsigned)((long)(order[first + r] / top) * ldx * sizeof(T)) : kNothing;
  }
  const long left = (long)(F - col0) * K * sizeof(T), from = ((long)e * F + col0) * K;
  Tile t;
  // (rows 32 p to 32 p + 15 of the weights in LDS are gate rows 16 p .., the next sixteen the same up rows)
  t.run(buffer_of(x, ((long)(n_tokens - 1) * ldx + K) * sizeof(T)), x_at, buffer_of(((wave >> 1) & 1 ? w_up : w_gate) + from, left),
        [&](int i) LS_INLINED { return ((i * Tile::NW + wave) >> 2) * 16 + (wave & 1) * 8; }, K, ring);
#pragma unroll
  for (int j = 0; j < Tile::TJ; ++j) {
    const int r = Tile::row_of(j);
    if (r >= rows) continue;
    T* dst = act + (long)(first + r) * ldy;
    const float wt = in_weight ? in_weight[order[first + r]] : 1.0f;
#pragma unroll
    for (int p = 0; p < Tile::TI; p += 2) {
      const int w0 = Tile::weight_of(p), c0 = col0 + (w0 >> 5) * 16 + (w0 & 15);
      typedef __attribute__((ext_vector_type(4))) T four_t;
      four_t y;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float g = fminf(t.product.acc[p][j][i] * wt, limit);
        const float u = fminf(fmaxf(t.product.acc[p + 1][j][i] * wt, -limit), limit);
        y[i] = from_f32<T>((g * sigmoid_e(alpha * g)) * (u + shift));
      }
      if (c0 + 3 < F) {  // (act and its rows start on 16 bytes)
        *reinterpret_cast<four_t*>(dst + c0) = y;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (c0 + i < F) dst[c0 + i] = y[i];
      }
    }
  }
}

template <typename T, int COLS, int NWM, int NWN>
__global__ __launch_bounds__(64 * NWM * NWN) void experts_down_ring_kernel(const T* __restrict__ act, long ldy,
                                                                const T* __restrict__ w_down, int N, int F, int top,
                                                                int n_tokens, const int* __restrict__ order,
                                                                const int* __restrict__ tiles, int cap,
                                                                const float* __restrict__ weight, float* __restrict__ P,
                                                                const T* __restrict__ x, long ldx,
                                                                const float* __restrict__ share, int real, int vec_out) {
  typedef ExpertTile<T, COLS, NWM, NWN> Tile;
  extern __shared__ __attribute__((aligned(1024))) unsigned char ring[];
  int tile, column;
  if (!tile_and_column<kUnit<T>>((N + COLS - 1) / COLS, cap, tile, column)) return;
  const int e = tiles[4 * tile];
  if (e < 0) return;
  const int first = tiles[4 * tile + 1], rows = tiles[4 * tile + 2];
  const int col0 = column * COLS;
  if (e >= real) {
    pass_input<T, Tile::kThreads>(x, ldx, share, first, rows, col0, min(N, col0 + COLS), top, n_tokens, N, order, P);
    return;
  }
  const int wave = Tile::wave();
  unsigned x_at[Tile::LX];
#pragma unroll
  for (int i = 0; i < Tile::LX; ++i) {
    const int r = Tile::loaded_row(i);
    x_at[i] = r < rows ? (unsigned)(r * ldy * sizeof(T)) : kNothing;
  }
  Tile t;
  t.run(buffer_of(act + (long)first * ldy, ((long)(rows - 1) * ldy + F) * sizeof(T)), x_at,
        buffer_of(w_down + ((long)e * N + col0) * F, (long)(N - col0) * F * sizeof(T)),
        [&](int i) LS_INLINED { return (i * Tile::NW + wave) * 8; }, F, ring);
#pragma unroll
  for (int j = 0; j < Tile::TJ; ++j) {
    const int r = Tile::row_of(j);
    if (r >= rows) continue;
    const int pair = order[first + r];
    const float wt = weight ? weight[pair] : 1.0f;
    float* dst = P + ((long)(pair % top) * n_tokens + pair / top) * N;
#pragma unroll
    for (int i = 0; i < Tile::TI; ++i) {
      const int c0 = col0 + Tile::weight_of(i);
      const f32x4& acc = t.product.acc[i][j];
      const f32x4 y = f32x4{wt * acc[0], wt * acc[1], wt * acc[2], wt * acc[3]};
      if (vec_out && c0 + 3 < N) {
        *reinterpret_cast<f32x4*>(dst + c0) = y;
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (c0 + q < N) dst[c0 + q] = y[q];
      }
    }
  }
}

}  // namespace ls

LS_DEFINE_ERROR_API

using namespace ls;

extern "C" int ls_experts_max_top() { return kMaxTop; }

// The two kernels of 64-row tiles.
#define LS_EXPERTS_UP(T_) experts_gate_up_ring_kernel<T_, 128, 2, 4>
#define LS_EXPERTS_DOWN(T_) experts_down_ring_kernel<T_, kDownCols<T_>, 4, 2>
template <typename T> constexpr int kUpLds = ExpertTile<T, 128, 2, 4>::kLds;
template <typename T> constexpr int kDownLds = ExpertTile<T, kDownCols<T>, 4, 2>::kLds;

// Dynamic LDS beyond 64 KB has to be granted per kernel (once).
template <typename T>
static bool ring_lds_ready() {
  auto grant = [](const void* kernel, int bytes) {
    const bool ok = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess;
    if (!ok) (void)hipGetLastError();
    return ok;
  };
  static const bool granted = grant((const void*)&LS_EXPERTS_UP(T), kUpLds<T>) && grant((const void*)&LS_EXPERTS_DOWN(T), kDownLds<T>);
  return granted;
}

// Tiles that the pairs of n_tokens tokens can need at most, with rows_a_tile rows each.
extern "C" int ls_experts_tile_capacity(int n_tokens, int E, int top, int rows_a_tile) {
  const long pairs = (long)n_tokens * top;
  return (int)(pairs / rows_a_tile + (pairs < E ? pairs : E));
}

// z [n_tokens][ldz] float router logits, bias [E] or null -> expert, weight [n_tokens][top]; order [n_tokens * top];
// tiles [cap][4]; counts: scratch of E ints.  rows_a_tile 16, 32 or 64.
extern "C" int ls_experts_route(const float* z, long ldz, const float* bias, int n_tokens, int E, int top,
                                int rows_a_tile, int* expert, float* weight, int* order, int* tiles, int cap,
                                int* counts, int scoring, const float* correction, int groups, int keep, void* stream) {
  LS_REQUIRE(scoring >= 0 && scoring <= 2, "experts_route: scoring %d (0: softmax over the chosen, 1: sigmoid, 2: softmax over all)",
             scoring);
  LS_REQUIRE(scoring != 2 || (correction && groups > 0 && keep > 0 && keep <= groups && E % groups == 0 && top <= keep * (E / groups)),
             "experts_route: %d experts in %d groups of which %d are kept, %d a token", E, groups, keep, top);
  const Choice how{scoring, groups, keep, correction};
  LS_REQUIRE(n_tokens > 0 && E > 0 && top > 0 && top <= E && top <= kMaxTop && ldz >= E,
             "experts_route: %d tokens, %d experts, %d chosen (at most %d)", n_tokens, E, top, kMaxTop);
  LS_REQUIRE(rows_a_tile == 16 || rows_a_tile == 32 || rows_a_tile == 64, "experts_route: tiles of %d rows", rows_a_tile);
  LS_REQUIRE(z && expert && weight && order && tiles && counts, "experts_route: null operand");
  LS_REQUIRE(cap >= ls_experts_tile_capacity(n_tokens, E, top, rows_a_tile), "experts_route: %d tiles are too few", cap);
  LS_REQUIRE(E <= 64 * kMaxPerLane, "experts_route: %d experts, the routing kernel takes %d", E, 64 * kMaxPerLane);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int P = n_tokens * top;
#define LS_ROUTE(PL_)                                                                                                     \
  if (P <= kSmallPairs && E <= kSmallExperts)                                                                             \
    hipLaunchKernelGGL((route_small_kernel<PL_, float, false>), dim3(1), dim3(1024), 0, s, z, ldz, bias, n_tokens, E, top, \
                       rows_a_tile, expert, weight, order, tiles, cap, (const int*)nullptr, (const int*)nullptr, how,     \
                       (const float*)nullptr, 0L, (const float*)nullptr, 0);                                              \
  else                                                                                                                    \
    hipLaunchKernelGGL(route_topk_kernel<PL_>, dim3((n_tokens + 3) / 4), dim3(256), 0, s, z, ldz, bias, n_tokens, E, top, \
                       expert, weight, how);
  if (E <= 64) { LS_ROUTE(1) }
  else if (E <= 128) { LS_ROUTE(2) }
  else { LS_ROUTE(kMaxPerLane) }
#undef LS_ROUTE
  if (!(P <= kSmallPairs && E <= kSmallExperts)) {
    hipLaunchKernelGGL(route_count_kernel, dim3(E), dim3(64 * route_waves(P)), 0, s, expert, P, counts);
    hipLaunchKernelGGL(route_place_kernel, dim3(E), dim3(64 * route_waves(P)), 0, s, expert, counts, P, E, rows_a_tile, order, tiles, cap);
  }
  return check_launch("experts_route");
}

// Whether ls_experts_route_product takes a step of n_tokens tokens.
extern "C" int ls_experts_route_product_ok(int dtype, int n_tokens, int E, int top, int K) {
  return n_tokens <= 16 && E <= 16 * kProductTiles && (long)n_tokens * top <= kSmallPairs && K % (dtype == kF32 ? 4 : 8) == 0;
}

// The same with the router's product inside: x [n_tokens][ldx] and w_router [E][K] of the compute dtype instead of logits.
extern "C" int ls_experts_route_product(int dtype, const void* x, long ldx, const void* w_router, int K, const float* bias,
                                        int n_tokens, int E, int top, int rows_a_tile, int* expert, float* weight, int* order,
                                        int* tiles, int cap, int scoring, const float* correction, int groups, int keep,
                                        void* stream) {
  LS_REQUIRE(scoring >= 0 && scoring <= 2, "experts_route_product: scoring %d", scoring);
  LS_REQUIRE(scoring != 2 || (correction && groups > 0 && keep > 0 && keep <= groups && E % groups == 0 && top <= keep * (E / groups)),
             "experts_route_product: %d experts in %d groups of which %d are kept, %d a token", E, groups, keep, top);
  LS_REQUIRE(n_tokens > 0 && E > 0 && top > 0 && top <= E && top <= kMaxTop && K > 0 && ldx >= K && ls_experts_route_product_ok(dtype, n_tokens, E, top, K),
             "experts_route_product: %d tokens, %d experts, %d chosen", n_tokens, E, top);
  LS_REQUIRE(rows_a_tile == 16 || rows_a_tile == 32 || rows_a_tile == 64, "experts_route_product: tiles of %d rows", rows_a_tile);
  LS_REQUIRE(x && w_router && expert && weight && order && tiles && cap >= ls_experts_tile_capacity(n_tokens, E, top, rows_a_tile),
             "experts_route_product: bad operands");
  LS_REQUIRE(dtype == kF32 || dtype == kBF16, "experts_route_product: unknown dtype %d", dtype);
  LS_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w_router) % 16 == 0 &&
                 ldx % (dtype == kF32 ? 4 : 8) == 0,
             "experts_route_product: operands must be 16-byte aligned");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const Choice how{scoring, groups, keep, correction};
#define LS_ROUTE_PRODUCT(PL_, T_)                                                                                         \
  hipLaunchKernelGGL((route_small_kernel<PL_, T_, true>), dim3(1), dim3(1024), 0, s, (const float*)nullptr, 0L, bias, n_tokens, E, \
                     top, rows_a_tile, expert, weight, order, tiles, cap, (const int*)nullptr, (const int*)nullptr, how,  \
                     (const T_*)x, ldx, (const T_*)w_router, K)
  if (dtype == kF32) {
    if (E <= 64) LS_ROUTE_PRODUCT(1, float); else LS_ROUTE_PRODUCT(2, float);
  } else {
    if (E <= 64) LS_ROUTE_PRODUCT(1, bf16_t); else LS_ROUTE_PRODUCT(2, bf16_t);
  }
#undef LS_ROUTE_PRODUCT
  return check_launch("experts_route_product");
}

// The same grouping for experts that a table names: token_ids [n_tokens], table [vocab][top] with entries in [0, E).
extern "C" int ls_experts_route_table(const int* token_ids, const int* table, int n_tokens, int E, int top,
                                      int rows_a_tile, int* expert, float* weight, int* order, int* tiles, int cap,
                                      int* counts, void* stream) {
  LS_REQUIRE(n_tokens > 0 && E > 0 && top > 0 && top <= E, "experts_route_table: %d tokens, %d experts, %d a token", n_tokens, E, top);
  LS_REQUIRE(rows_a_tile == 16 || rows_a_tile == 32 || rows_a_tile == 64, "experts_route_table: tiles of %d rows", rows_a_tile);
  LS_REQUIRE(token_ids && table && expert && weight && order && tiles && counts, "experts_route_table: null operand");
  LS_REQUIRE(cap >= ls_experts_tile_capacity(n_tokens, E, top, rows_a_tile), "experts_route_table: %d tiles are too few", cap);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int P = n_tokens * top;
  if (P <= kSmallPairs && E <= kSmallExperts) {
    hipLaunchKernelGGL((route_small_kernel<1, float, false>), dim3(1), dim3(1024), 0, s, (const float*)nullptr, 0L, (const float*)nullptr,
                       n_tokens, E, top, rows_a_tile, expert, weight, order, tiles, cap, token_ids, table, Choice{0, 1, 1, nullptr},
                       (const float*)nullptr, 0L, (const float*)nullptr, 0);
  } else {
    hipLaunchKernelGGL(route_table_kernel, dim3((P + 255) / 256), dim3(256), 0, s, token_ids, table, n_tokens, top, expert,
                       weight);
    hipLaunchKernelGGL(route_count_kernel, dim3(E), dim3(64 * route_waves(P)), 0, s, expert, P, counts);
    hipLaunchKernelGGL(route_place_kernel, dim3(E), dim3(64 * route_waves(P)), 0, s, expert, counts, P, E, rows_a_tile, order, tiles, cap);
  }
  return check_launch("experts_route_table");
}

// x [n_tokens][ldx]; w_gate, w_up [E][F][K]; w_down [E][N][F]; act: scratch [n_tokens * top][ldy] of the compute
// dtype; P [top][n_tokens][N] float.
extern "C" int ls_experts_apply(int dtype, const void* x, long ldx, const void* w_gate, const void* w_up,
                                const void* w_down, int n_tokens, int E, int top, int K, int F, int N,
                                int rows_a_tile, const int* order, const int* tiles, int cap, const float* weight,
                                float limit, float alpha, float shift, void* act, long ldy, float* P, int weigh_input,
                                int real, const void* sh_gate_up, const void* sh_down, int sh_F, void* sh_act, long sh_ldy,
                                float* sh_out, void* stream) {
  // sh_*: an expert that every token uses, worked on in the same launches (tiles of 16 rows only; null: none)
  const bool with_shared = sh_gate_up != nullptr;
  LS_REQUIRE(!with_shared || (rows_a_tile == 16 && sh_down && sh_act && sh_out && sh_F > 0 && sh_ldy >= sh_F &&
                              reinterpret_cast<uintptr_t>(sh_gate_up) % 16 == 0 && reinterpret_cast<uintptr_t>(sh_down) % 16 == 0 &&
                              reinterpret_cast<uintptr_t>(sh_act) % 16 == 0),
             "experts_apply: a shared expert is worked on beside tiles of 16 rows, its operands 16-byte aligned");
  // weigh_input: the routing weight multiplies the expert's input instead of its output.  real: experts from this one on
  // (of the E that the tiles may name) have no weights and return their input
  LS_REQUIRE(real > 0 && real <= E && (real == E || K == N), "experts_apply: %d of %d experts with weights", real, E);
  const float* in_weight = weigh_input ? weight : nullptr;
  const float* out_weight = weigh_input ? nullptr : weight;
  LS_REQUIRE(n_tokens > 0 && E > 0 && top > 0 && K > 0 && F > 0 && N > 0 && ldx >= K && ldy >= F, "experts_apply: bad sizes");
  LS_REQUIRE(rows_a_tile == 16 || rows_a_tile == 32 || rows_a_tile == 64, "experts_apply: tiles of %d rows", rows_a_tile);
  LS_REQUIRE(x && w_gate && w_up && w_down && order && tiles && weight && act && P && cap > 0, "experts_apply: null operand");
  LS_REQUIRE(limit > 0.f, "experts_apply: the limit must be positive");
  LS_REQUIRE(dtype == kF32 || dtype == kBF16, "experts_apply: unknown dtype %d", dtype);
  const int vec = dtype == kF32 ? 4 : 8;
  LS_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(act) % 16 == 0 &&
                 reinterpret_cast<uintptr_t>(w_gate) % 16 == 0 && reinterpret_cast<uintptr_t>(w_up) % 16 == 0 &&
                 reinterpret_cast<uintptr_t>(w_down) % 16 == 0 && (K % vec != 0 || ldx % vec == 0),
             "experts_apply: operands must be 16-byte aligned");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  // tiles of 16 rows (few tokens an expert): a workgroup takes 16 columns and cuts K over its waves
  const int cols = rows_a_tile == 16 ? 16 : 64;
  const int more = with_shared ? (n_tokens + 15) / 16 : 0, widest = with_shared && sh_F > F ? sh_F : F;
  const dim3 grid_up(cap + more, (widest + cols - 1) / cols), grid_down(cap + more, (N + cols - 1) / cols);
  auto shared_of = [&](auto* of_type) {
    typedef std::remove_pointer_t<decltype(of_type)> E_;
    return SharedExpert<E_>{(const E_*)sh_gate_up, (const E_*)sh_down, sh_F, with_shared ? cap : 0x7fffffff, (E_*)sh_act, sh_ldy, sh_out};
  };
#define LS_EXPERTS(T_, RT_, KS_)                                                                                      \
  do {                                                                                                                \
    hipLaunchKernelGGL((experts_gate_up_kernel<T_, RT_, KS_>), grid_up, dim3(256), 0, s, (const T_*)x, ldx,           \
                       (const T_*)w_gate, (const T_*)w_up, F, K, top, order, tiles, limit, alpha, shift, in_weight,   \
                       (T_*)act, ldy, real, n_tokens, shared_of((T_*)nullptr));                                       \
    hipLaunchKernelGGL((experts_down_kernel<T_, RT_, KS_>), grid_down, dim3(256), 0, s, (const T_*)act, ldy,          \
                       (const T_*)w_down, N, F, top, n_tokens, order, tiles, out_weight, P, (const T_*)x, ldx, weight, real, \
                       shared_of((T_*)nullptr));                                                                      \
  } while (0)
  // tiles of 64 rows go through LDS where every row of every operand starts on a 16-byte boundary, 32-bit offsets reach the
  // rows (all of x, whose rows are picked; 128 of the weights, 64 of act), and a grid of 512 threads a workgroup has room
  // for the tiles (2^32 threads).  Rows further apart go to the kernel that forms 64-bit addresses.
  const long across = 128 * std::max({(long)K, (long)F, ldy}), all_of_x = (n_tokens - 1) * ldx + K;
  auto grid_of = [&](int width, int columns) {
    return dtype == kF32 ? tile_grid<kUnit<float>>((width + columns - 1) / columns, cap) : tile_grid<kUnit<bf16_t>>((width + columns - 1) / columns, cap);
  };
  const long wgs_up = grid_of(F, 64), wgs_down = grid_of(N, dtype == kF32 ? kDownCols<float> : kDownCols<bf16_t>);
  const bool staged = rows_a_tile == 64 && K % vec == 0 && F % vec == 0 && ldx % vec == 0 && ldy % vec == 0 &&
                      std::max(across, all_of_x) * (16 / vec) + 128 <= (long)kNothing && std::max(wgs_up, wgs_down) < (1L << 23) &&
                      (dtype == kF32 ? ring_lds_ready<float>() : ring_lds_ready<bf16_t>());
  const int vec_out = N % 4 == 0 && reinterpret_cast<uintptr_t>(P) % 16 == 0;
#define LS_EXPERTS_STAGED(T_)                                                                                         \
  do {                                                                                                                \
    hipLaunchKernelGGL((LS_EXPERTS_UP(T_)), dim3(wgs_up), dim3(512), kUpLds<T_>, s, (const T_*)x, ldx, (const T_*)w_gate,  \
                       (const T_*)w_up, F, K, top, order, tiles, cap, limit, alpha, shift, in_weight, (T_*)act, ldy, real, n_tokens); \
    hipLaunchKernelGGL((LS_EXPERTS_DOWN(T_)), dim3(wgs_down), dim3(512), \
                       kDownLds<T_>, s, (const T_*)act, ldy, (const T_*)w_down, N, F, top, n_tokens, order, tiles, cap, out_weight, P, \
                       (const T_*)x, ldx, weight, real, vec_out);                                                     \
  } while (0)
  // tiles of 16 rows of whole chunks and columns have kernels of their own
  const int few_up = few_chunks(dtype, K), few_down = few_chunks(dtype, F);
  const bool few = rows_a_tile == 16 && !with_shared && few_up && few_down && F % 16 == 0 && N % 16 == 0 && ldx % vec == 0 &&
                   ldy % vec == 0 && reinterpret_cast<uintptr_t>(tiles) % 16 == 0 && (F + 15) / 16 < 65536 && (N + 15) / 16 < 65536;
#define LS_FEW_UP(T_, U_)                                                                                             \
  hipLaunchKernelGGL((experts_few_gate_up_kernel<T_, U_, kListed>), dim3(cap, F / 16), dim3(256), 0, s, tiles,          \
                     (const T_*)w_gate, (const T_*)w_up, order, (const T_*)x, ldx, F, K, top, real, limit, alpha, shift, \
                     in_weight, (T_*)act, ldy, n_tokens, E, (int*)nullptr)
#define LS_FEW_DOWN(T_, U_)                                                                                           \
  hipLaunchKernelGGL((experts_few_down_kernel<T_, U_, kListed, 1>), dim3(cap, N / 16), dim3(256), 0, s, tiles,        \
                     (const T_*)w_down, (const T_*)act, ldy, order, out_weight, P, N, F, top, n_tokens, real, (const T_*)x, \
                     ldx, weight, E)
#define LS_FEW(T_)                                                                                                    \
  do {                                                                                                                \
    if (few_up == 8) LS_FEW_UP(T_, 8); else if (few_up == 6) LS_FEW_UP(T_, 6); else LS_FEW_UP(T_, 4);                 \
    if (few_down == 8) LS_FEW_DOWN(T_, 8); else if (few_down == 6) LS_FEW_DOWN(T_, 6); else LS_FEW_DOWN(T_, 4);       \
  } while (0)
#define LS_EXPERTS_BY_ROWS(T_)                 \
  switch (rows_a_tile) {                       \
    case 16:                                   \
      if (few)                                 \
        LS_FEW(T_);                            \
      else                                     \
        LS_EXPERTS(T_, 1, 4);                  \
      break;                                   \
    case 32: LS_EXPERTS(T_, 2, 1); break;      \
    default:                                   \
      if (staged)                              \
        LS_EXPERTS_STAGED(T_);                 \
      else                                     \
        LS_EXPERTS(T_, 4, 1);                  \
      break;                                   \
  }
  if (dtype == kF32) {
    LS_EXPERTS_BY_ROWS(float)
  } else {
    LS_EXPERTS_BY_ROWS(bf16_t)
  }
#undef LS_EXPERTS_BY_ROWS
#undef LS_FEW
#undef LS_FEW_UP
#undef LS_FEW_DOWN
#undef LS_EXPERTS_STAGED
#undef LS_EXPERTS
  return check_launch("experts_apply");
}

// Workgroups along x that find their rows in a table: for every expert and sixteen tokens, or for every pair.  (For every expert
// alone, one token of 4 of 32, 64, 256 and 512 experts, 1,024 x 768, both launches us: 16.1, 18.5, 27.6 and 42.9; now 11.2, 11.4, 11.4 and 11.3;
// with a list, the launch that makes it included, 14.4, 17.0, 39.4 and 86.5.  Eight tokens of 32 experts are 32 either way: 27.7 for 29.5.)
static int table_groups(int n_tokens, int E, int top) {
  return (int)std::min<long>((long)n_tokens * top, (long)E * ((n_tokens + 15) / 16));
}

// Whether ls_experts_apply_table takes a step of these sizes.
extern "C" int ls_experts_apply_table_ok(int dtype, int n_tokens, int E, int top, int K, int F, int N) {
  return n_tokens > 0 && (long)n_tokens * top <= kTablePairs && few_chunks(dtype, K) && few_chunks(dtype, F) && F % 16 == 0 && N % 16 == 0 &&
         F / 16 < 65536 && N / 16 < 65536 && (long)E * ((n_tokens + 15) / 16) <= 0x7fffffffL;
}

// ... and whether it is the faster route: where it has no more workgroups than a list has room for tiles.  Each of them looks its rows up before
// it knows whether it has any (table / list, 1,024 x 768, us: 17 tokens 3 of 4, 8 workgroups for 7, 13.4 / 16.0; 3 of 64 51 for 54, 40.7 / 44.2;
// 1 of 12 17 for 13, 20.2 / 19.6; 64 tokens 1 of 16 64 for 20, 31.2 / 24.6; 2,048 x 2,048 32 tokens 1 of 4 8 for 6, 38.2 / 30.5;
// up to a ratio of 1 the table was ahead or level at every size tried, beyond it now one, now the other).
extern "C" int ls_experts_apply_table_pays(int n_tokens, int E, int top) {
  return n_tokens > 0 && table_groups(n_tokens, E, top) <= ls_experts_tile_capacity(n_tokens, E, top, 16);
}

// ls_experts_route_table and ls_experts_apply in two launches, for few pairs: token t uses the experts that row token_ids[t] of
// table [vocab][top] names (entries in [0, E), those of a row differ), each with the weight 1 / top.  picks: scratch of n_tokens * top
// ints, the pairs' experts afterwards.
extern "C" int ls_experts_apply_table(int dtype, const void* x, long ldx, const void* w_gate, const void* w_up, const void* w_down,
                                      const int* token_ids, const int* table, int n_tokens, int E, int top, int K, int F, int N,
                                      float limit, float alpha, float shift, void* act, long ldy, int* picks, float* P,
                                      void* stream) {
  LS_REQUIRE(dtype == kF32 || dtype == kBF16, "experts_apply_table: unknown dtype %d", dtype);
  LS_REQUIRE(n_tokens > 0 && E > 0 && top > 0 && top <= E && K > 0 && F > 0 && N > 0 && ldx >= K && ldy >= F &&
                 ls_experts_apply_table_ok(dtype, n_tokens, E, top, K, F, N),
             "experts_apply_table: %d tokens, %d of %d experts, sizes %d, %d, %d", n_tokens, top, E, K, F, N);
  LS_REQUIRE(x && w_gate && w_up && w_down && token_ids && table && act && picks && P, "experts_apply_table: null operand");
  LS_REQUIRE(limit > 0.f, "experts_apply_table: the limit must be positive");
  const int vec = dtype == kF32 ? 4 : 8;
  LS_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(act) % 16 == 0 &&
                 reinterpret_cast<uintptr_t>(w_gate) % 16 == 0 && reinterpret_cast<uintptr_t>(w_up) % 16 == 0 &&
                 reinterpret_cast<uintptr_t>(w_down) % 16 == 0 && ldx % vec == 0 && ldy % vec == 0,
             "experts_apply_table: operands must be 16-byte aligned");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int groups = table_groups(n_tokens, E, top);
#define LS_TABLE_UP(T_, U_)                                                                                           \
  hipLaunchKernelGGL((experts_few_gate_up_kernel<T_, U_, kTable>), dim3(groups, F / 16), dim3(256), 0, s, token_ids,    \
                     (const T_*)w_gate, (const T_*)w_up, table, (const T_*)x, ldx, F, K, top, E, limit, alpha, shift, \
                     (const float*)nullptr, (T_*)act, ldy, n_tokens, E, picks)
#define LS_TABLE_DOWN_COLS(T_, U_, COLS_)                                                                             \
  hipLaunchKernelGGL((experts_few_down_kernel<T_, U_, kPicked, COLS_>), dim3(groups, N / (16 * COLS_)), dim3(256), 0, s, picks, \
                     (const T_*)w_down, (const T_*)act, ldy, (const int*)nullptr, (const float*)nullptr, P, N, F, top, n_tokens, E, \
                     (const T_*)nullptr, 0L, (const float*)nullptr, E)
#define LS_TABLE_DOWN(T_, U_) \
  if (sizeof(T_) == 2 && N % 32 == 0) LS_TABLE_DOWN_COLS(T_, U_, 2); else LS_TABLE_DOWN_COLS(T_, U_, 1)
#define LS_TABLE(T_)                                                                                                  \
  do {                                                                                                                \
    const int up = few_chunks(dtype, K), down = few_chunks(dtype, F);                                                 \
    if (up == 8) LS_TABLE_UP(T_, 8); else if (up == 6) LS_TABLE_UP(T_, 6); else LS_TABLE_UP(T_, 4);                   \
    if (down == 8) { LS_TABLE_DOWN(T_, 8); } else if (down == 6) { LS_TABLE_DOWN(T_, 6); } else { LS_TABLE_DOWN(T_, 4); } \
  } while (0)
  if (dtype == kF32) LS_TABLE(float);
  else LS_TABLE(bf16_t);
#undef LS_TABLE
#undef LS_TABLE_UP
#undef LS_TABLE_DOWN
#undef LS_TABLE_DOWN_COLS
  return check_launch("experts_apply_table");
}
