// Grouped-query attention over the paged cache whose softmax has a sink, with a choice of what a query
// sees and of what is added to its scores:
//
//   s_h[i, j]    = (q_h[i] . k_kv(h)[j]) * scale + bias_h[min(i - j, n_dist - 1)]   (bias optional)
//   visible(i,j) = lo(i) <= j <= i,   lo(i) = max(window ? i - window + 1 : 0, chunk ? floor(i / chunk) chunk : 0),
//                  or j < keep_first (the first tokens stay visible when a window has passed them; their tiles are
//                  walked before the window's)
//   p_h[i, j]    = exp(s_h[i, j]) / (exp(sink_h) + sum over visible j' of exp(s_h[i, j']))  (without a sink: no term)
//   o_h[i]       = gate_h[i] * sum_j p_h[i, j] v_kv(h)[j],   gate = sigmoid(g_h[i]) elementwise (optional)
//
// i and j are absolute positions; the sink is a score that has no key and no value, so the weights of a
// row add up to less than one.  The bias is a table by distance, one row a head, whose last entry serves
// every larger distance.
//
// The library is compiled for one key size LS_SA_DIM and one value size LS_SA_VDIM.  A wave owns 16 RT
// rows of the 16x16 MFMA atom and walks the visible keys in tiles of 32 anchored at absolute positions.
// Keys are the first operand of the score product (S^T = K Q^T: a lane ends with four consecutive keys of
// one query row, which is how the weights enter the value product) and value columns the first operand of
// O^T += V^T P^T (the lane that holds a row's statistics also holds its accumulators).  A key or value
// fragment is loaded once and multiplied with all RT row tiles.  Two shapes of work:
//   prompt portions  a workgroup takes (request, block of 16 RT rows, key/value head); its waves are the
//                    query heads that read this key/value head, so their loads of K and V meet in the
//                    CU's cache;
//   decoded tokens   a wave takes (request, key/value head) and the MFMA rows are the query heads of the
//                    group (up to 16 a wave).
// The tiles of a row block are dealt to several work items in contiguous runs where that fills the GPU;
// each leaves (unnormalised output, max, sum) of its run for every row and a second kernel folds the
// runs in ascending order, adds the sink and applies the gate.
// Scores, weights, statistics and accumulators are float; products read the compute dtype T.  For keys
// that a request does not hold (beyond its length, pages that a window or a chunk's end has released) the first
// row of page 0 is multiplied, whatever it holds, and their scores are masked; their values are replaced by zeros before the product.

#include "common.h"
#include "ring.h"

#include <type_traits>

#ifndef LS_SA_DIM
#error "compile with -DLS_SA_DIM and -DLS_SA_VDIM"
#endif

namespace ls {

constexpr int D = LS_SA_DIM, DV = LS_SA_VDIM;
static_assert(D % 8 == 0 && D <= 640, "key size must be a multiple of 8 up to 640");
static_assert(DV >= 1 && DV <= 512, "value size must be at most 512");
constexpr int VB = (DV + 15) / 16;  // blocks of 16 value columns (the last may be partial)
constexpr int kTileKeys = 32;
constexpr int kMaxWaves = 4;        // query heads of a key/value head that share a workgroup

struct SeqMeta {
  int q_off, q_len, q_start, kv_len, table_row, reserved[3];
};

template <typename T>
__device__ __forceinline__ typename Atom<T>::vec_t load_or_zero(const T* p, bool ok) {
  typedef typename Atom<T>::vec_t vec_t;
  // (an address that is always valid, the value chosen afterwards: the loads of a tile can be in flight together)
  vec_t v = *reinterpret_cast<const vec_t*>(p);
  return ok ? v : Atom<T>::zero();
}

// A piece of a row of D elements, zeros behind them.  What a row or key that is not there gives is not chosen here: the
// compiler would put the load behind the choice, in a block of its own.
template <typename T>
__device__ __forceinline__ typename Atom<T>::vec_t load_piece(const T* p, bool in) {
  if constexpr (D % Atom<T>::KCHUNK == 0) return *reinterpret_cast<const typename Atom<T>::vec_t*>(p);
  else return load_or_zero<T>(p, in);
}

__device__ __forceinline__ float sigmoid_f(float x) { return 1.0f / (1.0f + expf(-x)); }

// First key that a query at position p sees.
__device__ __forceinline__ int first_seen(int p, int window, int chunk) {
  int lo = 0;
  if (window > 0) lo = max(lo, p - window + 1);
  if (chunk > 0) lo = max(lo, p / chunk * chunk);
  return lo;
}

// Waves a SIMD that the registers of a decoded token's wave are held to.  Two, where 256 registers hold its queries, keys, values and sums
// without a spill; left to itself the compiler takes accumulation registers besides and leaves room for one.  More than 1,024 waves want
// the second (bfloat16, keys of 192 and values of 128, eight key/value heads over 1,024 keys, us, one / two a SIMD: 160 requests 171 / 151,
// 128 requests 115 / 115; values of 192 and keys of 64, 16 requests in four runs 21.5 / 19.7).
template <typename T>
constexpr int decode_waves() { return sizeof(T) == 2 && (D + 31) / 32 + (DV + 15) / 16 <= 15 ? 2 : 1; }

// DEC: a step of single decoded tokens (the rows of a tile are the heads of a key/value group).
template <typename T, int RT, bool DEC>
__global__ __launch_bounds__(64 * (DEC ? 1 : kMaxWaves), DEC ? decode_waves<T>() : 1) void sink_attention_kernel(
    const T* __restrict__ q, long ldq, const T* __restrict__ k_pages, const T* __restrict__ v_pages, int page_size,
    const int* __restrict__ table, int table_stride, const SeqMeta* __restrict__ seqs, const int* __restrict__ items,
    int H, int G, float scale, int window, int chunk, int keep_first, const float* __restrict__ sink,
    const float* __restrict__ dist_bias, int n_dist, const float* __restrict__ gate, long ldg, T* __restrict__ out,
    long ldo, float* __restrict__ part, int part_rows) {
  constexpr int VEC = Atom<T>::VEC, KC = Atom<T>::KCHUNK;
  constexpr int KCH = (D + KC - 1) / KC;  // chunks of a key (lanes beyond D in the last one bring zeros)
  constexpr int ROWS = 16 * RT;
  // a work item: request of the step, block of ROWS of its rows, which run of the tiles, of how many runs
  const int seq = items[4 * blockIdx.x], rb = items[4 * blockIdx.x + 1];
  const int run = items[4 * blockIdx.x + 2], n_runs = max(1, items[4 * blockIdx.x + 3]);
  const SeqMeta m = seqs[seq];
  const int GS = H / G, g = blockIdx.y;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int l16 = lane & 15, quad = lane >> 4;
  const int row0 = DEC ? 0 : rb * ROWS;
  if (row0 >= m.q_len) return;
  const int nrows = DEC ? 1 : min(ROWS, m.q_len - row0);
  // the head of a lane's row: one head a wave for prompt portions, a head a row for decoded tokens
  const int in_group = DEC ? blockIdx.z * 16 + l16 : blockIdx.z * kMaxWaves + w;
  if (!DEC && in_group >= GS) return;   // (the whole wave; no barrier follows)
  const bool head_ok = in_group < GS;
  const int my_head = g * GS + (head_ok ? in_group : 0);
  const int p_first = m.q_start + row0, p_last = p_first + nrows - 1;
  const int* my_table = table + (long)m.table_row * table_stride;
  const int page_shift = __ffs(page_size) - 1, page_mask = page_size - 1;   // (pages hold a power of two of keys)

  bool row_ok[RT];
  int my_pos[RT], my_lo[RT];
  const T* q_row[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int row = DEC ? 0 : 16 * r + l16;
    row_ok[r] = DEC ? head_ok : row < nrows;
    my_pos[r] = p_first + (row_ok[r] ? row : 0);
    my_lo[r] = first_seen(my_pos[r], window, chunk);
    q_row[r] = q + (long)(m.q_off + row0 + (row_ok[r] ? row : 0)) * ldq + (long)my_head * D;
  }
  const float* my_bias = dist_bias ? dist_bias + (long)my_head * n_dist : nullptr;

  float m_run[RT], l_run[RT];
  f32x4 acc[RT][VB];
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    m_run[r] = kNegSentinel;
    l_run[r] = 0.f;
#pragma unroll
    for (int b = 0; b < VB; ++b) acc[r][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  const int lo_last = first_seen(p_last, window, chunk);   // (no row of the block begins to see later than this)
  const int lo_tile = first_seen(p_first, window, chunk) / kTileKeys;
  const int hi_tile = p_last / kTileKeys;
  const int kept_tiles = min((keep_first + kTileKeys - 1) / kTileKeys, lo_tile);   // tiles of kept first tokens below the window's
  const int n_tiles = kept_tiles + hi_tile - lo_tile + 1;
  auto tile_at = [&](int step) LS_INLINED { return step < kept_tiles ? step : lo_tile + (step - kept_tiles); };
  const int per_run = (n_tiles + n_runs - 1) / n_runs;
  const int step_end = min(n_tiles, (run + 1) * per_run);

  // A tile's keys are requested while the tile before it is worked on: its addresses (page and slot of the
  // lane's key of each half as a row of K, and of its four keys as columns of V^T), the key vectors and the values.
  typedef typename std::conditional<sizeof(T) == 2, bf16x4, f32x4>::type v4_t;   // four keys of one value column
  // (the values travel with the keys where the registers allow it: not with four row tiles of wide values)
  constexpr bool kAheadV = RT * VB <= 16;
  struct Ahead {
    long v_at[2];
    bool v_ok[2][4];
    typename Atom<T>::vec_t kv[2][KCH];
    v4_t vv[2][kAheadV ? VB : 1];
  };
  // The page ids of a tile, of each half's key as a row of K and of its four keys as columns of V^T, are requested a tile before
  // its keys, and all at once: asked for where they are used, the second half's were waited for behind the first half's keys, so that
  // a first tile was three answers of memory one after the other (eight decoded tokens, sixteen heads over a latent, keys of 192, 134 to 160
  // of them: 8.1 -> 7.4 us in a decode step).
  auto pages_of = [&](int step, int (&ids)[2][2]) LS_INLINED {
    const int key0 = tile_at(step) * kTileKeys;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      ids[half][0] = my_table[min(key0 + 16 * half + l16, p_last) >> page_shift];
      ids[half][1] = my_table[min(key0 + 16 * half + 4 * quad, p_last) >> page_shift];
    }
  };
  int ids[2][2];
  pages_of(run * per_run, ids);
  auto request = [&](int step, Ahead& t) LS_INLINED {
    const int key0 = tile_at(step) * kTileKeys;
    const T* k_row[2];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int key = key0 + 16 * half + l16, key4 = key0 + 16 * half + 4 * quad;
      __asm__ volatile("" : "+v"(ids[half][0]), "+v"(ids[half][1]));   // (loaded whatever the key: no branch around the load)
      const int page = key <= p_last ? ids[half][0] : -1, page4 = key4 <= p_last ? ids[half][1] : -1;
      // (a key that is not held has page 0 and its scores are masked)
      k_row[half] = k_pages + ((((long)max(page, 0) * G + g) << page_shift) + (page >= 0 ? key & page_mask : 0)) * D;
      t.v_at[half] = ((((long)max(page4, 0) * G + g) * DV) << page_shift) + (page4 >= 0 ? key4 & page_mask : 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) t.v_ok[half][i] = page4 >= 0 && key4 + i <= p_last;
    }
    pages_of(step + 1, ids);
    __builtin_amdgcn_sched_barrier(0);   // (the next tile's page ids in front of this one's keys)
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int c = 0; c < KCH; ++c) {
        const bool in = c * KC + VEC * quad + VEC <= D;
        t.kv[half][c] = load_piece<T>(k_row[half] + (in ? c * KC + VEC * quad : 0), in);
      }
      if constexpr (kAheadV) {   // (the values too: they are on their way while the scores are formed)
#pragma unroll
        for (int b = 0; b < VB; ++b) {
          const long column = (long)(16 * b + l16 < DV ? 16 * b + l16 : 0) << page_shift;
          t.vv[half][b] = *reinterpret_cast<const v4_t*>(v_pages + t.v_at[half] + column);
        }
      }
    }
  };

  // The queries do not change from tile to tile: they stay in registers where that takes at most 64 of them.
  constexpr bool kKeepQ = RT * KCH * (int)(sizeof(typename Atom<T>::vec_t) / 4) <= 64;
  typename Atom<T>::vec_t qv[kKeepQ ? RT : 1][kKeepQ ? KCH : 1];
  if constexpr (kKeepQ) {
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < KCH; ++c) {
        const bool in = c * KC + VEC * quad + VEC <= D;
        qv[r][c] = load_piece<T>(q_row[r] + (in ? c * KC + VEC * quad : 0), in);
      }
  }

  Ahead now;
  if (run * per_run < step_end) request(run * per_run, now);
  for (int step = run * per_run; step < step_end; ++step) {
    const int key0 = tile_at(step) * kTileKeys;
    bool v_ok[2][4];
    long v_at[2];
    v4_t vv[2][kAheadV ? VB : 1];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      v_at[half] = now.v_at[half];
#pragma unroll
      for (int i = 0; i < 4; ++i) v_ok[half][i] = now.v_ok[half][i];
      if constexpr (kAheadV) {
#pragma unroll
        for (int b = 0; b < VB; ++b) vv[half][b] = now.vv[half][b];
      }
    }
    // -- 1. transposed scores ----------------------------------------------------------------------
    f32x4 s[RT][2];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        s[r][half] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < KCH; ++c) {
          if constexpr (kKeepQ) {
            Atom<T>::mma(s[r][half], now.kv[half][c], qv[r][c]);
          } else {
            // (with a choice, or the compiler would keep all of these in registers it does not have)
            const bool in = c * KC + VEC * quad + VEC <= D;
            Atom<T>::mma(s[r][half], now.kv[half][c],
                         load_or_zero<T>(q_row[r] + (in ? c * KC + VEC * quad : 0), row_ok[r] && in));
          }
        }
      }
    if (step + 1 < step_end) request(step + 1, now);  // (the products above have taken this tile's keys)
    // -- 2. scale, bias, mask, online softmax ------------------------------------------------------------
    // A tile that every row of the block sees whole (most tiles of a long prompt) needs no mask: the same for the
    // whole wave, so the choice costs a scalar branch.
    float shrink[RT];
    bool moved = false;
    auto softmax_tile = [&](auto whole, auto biased) LS_INLINED {
      constexpr bool kWhole = decltype(whole)::value, kBiased = decltype(biased)::value;
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        bool see[2][4];
        float top = kNegSentinel;
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int key = key0 + 16 * half + 4 * quad + i;
            see[half][i] = kWhole || (row_ok[r] && key <= my_pos[r] && (key >= my_lo[r] || key < keep_first));
            float v = s[r][half][i] * scale;
            if constexpr (kBiased) v = v + my_bias[min(max(my_pos[r] - key, 0), n_dist - 1)];
            s[r][half][i] = v;
            top = fmaxf(top, see[half][i] ? v : kNegSentinel);
          }
        top = quad16_max(top);
        const float m_new = fmaxf(m_run[r], top);
        shrink[r] = softmax_exp<T>(m_run[r] - m_new);
        float sum = 0.f;
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            s[r][half][i] = see[half][i] ? softmax_exp<T>(s[r][half][i] - m_new) : 0.f;
            sum = sum + s[r][half][i];
          }
        sum = quad16_sum(sum);
        l_run[r] = l_run[r] * shrink[r] + sum;
        m_run[r] = m_new;
        moved = moved || shrink[r] != 1.0f;
      }
    };
    // (the mask and the bias are instances of the code, chosen by scalar branches once a tile)
    const bool whole_tile = key0 + kTileKeys - 1 <= p_first && (key0 >= lo_last || key0 + kTileKeys <= keep_first);
    if (my_bias) {
      if (whole_tile) softmax_tile(std::true_type{}, std::true_type{});
      else softmax_tile(std::false_type{}, std::true_type{});
    } else {
      if (whole_tile) softmax_tile(std::true_type{}, std::false_type{});
      else softmax_tile(std::false_type{}, std::false_type{});
    }
    // -- 3. values: column 16 b + l16 of V^T, keys 4 quad .. 4 quad + 3 of each half ----------------
    bool held = true;
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int i = 0; i < 4; ++i) held = held && v_ok[half][i];
    const bool all_held = __all(held) != 0 && DV % 16 == 0;
    if (__all(!moved) == 0) {
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int b = 0; b < VB; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[r][b][i] = acc[r][b][i] * shrink[r];
    }
    typename Atom<T>::vec_t pb[RT][sizeof(T) == 2 ? 1 : 2];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      if constexpr (sizeof(T) == 2) {
        typedef __attribute__((ext_vector_type(8))) float f32x8;
        const f32x8 both = __builtin_shufflevector(s[r][0], s[r][1], 0, 1, 2, 3, 4, 5, 6, 7);
        pb[r][0] = __builtin_convertvector(both, bf16x8);
      } else {
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int i = 0; i < 4; ++i) pb[r][half][i] = s[r][half][i];
      }
    }
#pragma unroll
    for (int b = 0; b < VB; ++b) {
      const bool col_ok = 16 * b + l16 < DV;
      const long column = (long)(col_ok ? 16 * b + l16 : 0) << page_shift;
      auto value4 = [&](int half) LS_INLINED {
        if constexpr (kAheadV) {
          return vv[half][b];
        } else {
          return *reinterpret_cast<const v4_t*>(v_pages + v_at[half] + column);
        }
      };
      if constexpr (sizeof(T) == 2) {
        const bf16x4 v0 = value4(0), v1 = value4(1);
        bf16x8 a;
        if (all_held) {
          a = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            a[i] = (v_ok[0][i] && col_ok) ? v0[i] : (bf16_t)0.f;
            a[4 + i] = (v_ok[1][i] && col_ok) ? v1[i] : (bf16_t)0.f;
          }
        }
#pragma unroll
        for (int r = 0; r < RT; ++r) Atom<T>::mma(acc[r][b], a, pb[r][0]);
      } else {
        f32x4 a[2];
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          const f32x4 v = value4(half);
          if (all_held) {
            a[half] = v;
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) a[half][i] = (v_ok[half][i] && col_ok) ? v[i] : 0.f;
          }
        }
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int half = 0; half < 2; ++half) Atom<T>::mma(acc[r][b], a[half], pb[r][half]);
      }
    }
  }

#pragma unroll
  for (int r = 0; r < RT; ++r) {
    if (!row_ok[r]) continue;
    const int row = DEC ? 0 : 16 * r + l16;
    if (n_runs > 1) {
      // [item][row][head][DV + 2]: the unnormalised output, then max and sum
      float* dst = part + (((long)blockIdx.x * part_rows + row) * H + my_head) * (DV + 2);
#pragma unroll
      for (int b = 0; b < VB; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (16 * b + 4 * quad + i < DV) dst[16 * b + 4 * quad + i] = acc[r][b][i];
      if (quad == 0) {
        dst[DV] = m_run[r];
        dst[DV + 1] = l_run[r];
      }
      continue;
    }
    // the sink joins the sum as one more score; the row's weights then add up to less than one
    float top = m_run[r], total = l_run[r], keep = 1.0f;
    if (sink) {
      const float sv = sink[my_head];
      top = fmaxf(m_run[r], sv);
      keep = softmax_exp<T>(m_run[r] - top);
      total = l_run[r] * keep + softmax_exp<T>(sv - top);
    }
    const float inv = keep / total;
    T* dst = out + (long)(m.q_off + row0 + row) * ldo + (long)my_head * DV;
    const float* g_row = gate ? gate + (long)(m.q_off + row0 + row) * ldg + (long)my_head * DV : nullptr;
#pragma unroll
    for (int b = 0; b < VB; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = 16 * b + 4 * quad + i;
        if (c < DV) {
          float v = acc[r][b][i] * inv;
          if (g_row) v = v * sigmoid_f(g_row[c]);
          dst[c] = from_f32<T>(v);
        }
      }
  }
}

// ---------------------------------------------------------------------------
// Prompt portions, key and value tiles staged in LDS.  The kernel above spends some 25 vector instructions on
// every MFMA: addresses and selects for each fragment it takes from global memory, and the row statistics of a
// tile of only 32 keys.  Here a workgroup of four waves has a tile of kKeys keys (128 bytes of keys a
// value column: 64 in bfloat16, 32 in float) loaded straight into LDS, and every wave
// reads its fragments from there.  A wave owns 32 rows of one head; the waves of a workgroup
// are min(GS, 4) query heads of the key/value head times 4 / min(GS, 4) groups of 32 rows, so a work item names a
// block of 32, 64 or 128 rows.  A tile's values are asked for among its score products, the next tile's keys among
// the exponentials.  The arithmetic of a row (scores, statistics, sums) is that of the kernel above with larger tiles.
//
// Layout: the 16-byte piece `piece` of key row r lies in slot slot_of_piece(r, piece) of the row; the values lie as [VEC
// keys][column][16 bytes].  In bfloat16 the rows of a pair of 16-key score blocks are dealt (key_of_row) so that the eight
// probabilities a lane ends with belong to eight consecutive keys, which is one read of the values.
//
// ONE_PAGE (rows of a multiple of 128 bytes, 64, 128, ... value columns, pages of 8 keys at least): the 64 pieces of a
// wave's load lie in one page, whose address is a scalar; else every lane looks its piece's page up.
//
// What bounds it: the vector unit (scales, maxima, exponentials: 1,200 of a wave's cycles a tile of 64 keys) in turn with the
// matrix cores (1,280 at keys of 192 and values of 128 elements), two workgroups a CU where the registers allow it.  Measured with its
// fold, us, tiles through registers with one workgroup a CU / now, 16 heads: 2,048 tokens, keys of 192 and values of 128, one key/value
// head 134 / 62, keys of 128 and eight of them 120 / 53; 700 from 1,500 on in a window of 600 45 / 34; 2,048 from 6,000 on 433 / 150.
// ---------------------------------------------------------------------------
template <typename T> struct Staged {
  static constexpr int kKeys = 128 / (int)sizeof(T);                 // keys of a tile
  static constexpr int kKeyPieces = D * (int)sizeof(T) / 16;         // 16-byte pieces of a key
  static constexpr int kKeyBytes = kKeys * kKeyPieces * 16;          // of the tile's keys
  static constexpr int kValueBytes = (8 * DV + 63) / 64 * 1024;      // and of its values (whole loads of a wave)
  static constexpr int kTilePages = 16;                              // page ids of a tile, at most
  static constexpr int kWindow =                                     // tiles whose page ids a workgroup holds
      kKeyBytes + kValueBytes + 32 * kTilePages * 4 <= 64 * 1024 ? 32 : 8;
  static constexpr int kBytes = kKeyBytes + kValueBytes + kWindow * kTilePages * 4;
  static constexpr bool kFits = kBytes <= 64 * 1024 && D % Atom<T>::VEC == 0;
  static constexpr bool kOnePage = kKeyPieces % 8 == 0 && DV % 64 == 0;
  // A lane's query and its sums are eight registers for each of these; with all else 256 hold them, and two workgroups share a CU, up
  // to a limit, beyond which registers would spill, and the wait for one is a wait for every load in flight.  Loads that
  // look pages up take a few more.  bfloat16, us, two / one a CU, 2,048 tokens from 6,000 on and 700 from 1,500 on in a window of 600:
  // keys of 192 and values of 128 elements (14 of these) 169 / 262 and 34 / 36; 128 and 192 (16) 245 / 299 and 46 / 41; 192 and
  // 192 (18) 289 / 325 and 53 / 42; 128 and 256 (20) 484 / 384 and 64 / 47; 112 and 112 (11, pages looked up) 158 / 255 and 32 / 34;
  // 144 and 144 (14, looked up) 262 / 306 and 50 / 40.  float32 128 and 192 (20) 946 / 1120 and 92 / 91; 256 and 128 (24)
  // 1336 / 1195 and 126 / 99; 144 and 144 (18, looked up) 884 / 1043 and 91 / 87; 160 and 160 (20, looked up) 1106 / 1132 and 111 / 94.
  static constexpr int kRowRegisters = (D + Atom<T>::KCHUNK - 1) / Atom<T>::KCHUNK + (DV + 15) / 16;
  static constexpr bool two_a_cu(bool one_page) { return kRowRegisters <= (sizeof(T) == 2 ? 14 : 20) - (one_page ? 0 : 2); }
};

// Which key of a tile row r (0..15) of the score block kb stands for.
template <typename T>
__device__ __forceinline__ constexpr int key_of_row(int kb, int r) {
  return sizeof(T) == 2 ? 32 * (kb >> 1) + 8 * (r >> 2) + 4 * (kb & 1) + (r & 3) : 16 * kb + r;
}
// The slot of a piece in its key's row (and the piece in a slot: each of these is its own inverse).  `l` is the row's place among
// the sixteen that a read takes together; of those LDS serves 0-3 and 12-15 at one piece with 4-11 at the piece beside it.
template <typename T>
__device__ __forceinline__ constexpr int slot_at(int l, int piece) {
  constexpr int P = Staged<T>::kKeyPieces;
  if (P % 16 == 0) return (piece & ~15) + ((piece & 15) ^ l);
  if (P % 8 == 0) return (piece & ~7) + ((piece & 7) ^ (l >> 1));
  if (P % 4 == 0) return (piece & ~3) + ((piece & 3) ^ (((l >> 1) & 2) ^ ((l >> 3) * 3)));
  return piece;
}
template <typename T>
__device__ __forceinline__ constexpr int slot_of_piece(int key, int piece) {
  return slot_at<T>(sizeof(T) == 2 ? (key & 3) + 4 * ((key >> 3) & 3) : key & 15, piece);
}

template <typename T, bool ONE_PAGE>
__global__ __launch_bounds__(256, Staged<T>::two_a_cu(ONE_PAGE) ? 2 : 1) void sink_attention_staged_kernel(
    const T* __restrict__ q, long ldq, const T* __restrict__ k_pages, const T* __restrict__ v_pages, int page_size,
    const int* __restrict__ table, int table_stride, const SeqMeta* __restrict__ seqs, const int* __restrict__ items,
    int H, int G, float scale, int window, int chunk, int keep_first, const float* __restrict__ sink,
    const float* __restrict__ dist_bias, int n_dist, const float* __restrict__ gate, long ldg, T* __restrict__ out,
    long ldo, float* __restrict__ part, int part_rows) {
  typedef Atom<T> A;
  typedef typename A::vec_t vec_t;
  typedef Staged<T> S;
  typedef __attribute__((address_space(3))) void* lptr_t;
  constexpr int SZ = sizeof(T), VEC = A::VEC, KC = A::KCHUNK;
  constexpr int KCH = D / KC + (D % KC ? 1 : 0);
  constexpr int TK = S::kKeys, NG = TK / 16;                       // keys of a tile, and groups of 16 of them
  constexpr int KP = S::kKeyPieces > 0 ? S::kKeyPieces : 1;
  constexpr int K_TOTAL = TK * KP, V_TOTAL = 8 * DV;               // pieces of a tile
  constexpr int KPER = (K_TOTAL + 255) / 256, VPER = (V_TOTAL + 255) / 256;
  constexpr int NC = sizeof(T) == 2 ? NG / 2 : NG;                 // chunks of keys of the value product
  static_assert(!ONE_PAGE || (K_TOTAL % 256 == 0 && V_TOTAL % 256 == 0 && KPER <= 32 && VPER <= 32), "whole loads");
  __shared__ __attribute__((aligned(16))) unsigned char lds[S::kFits ? S::kBytes : 16];
  unsigned char* const k_lds = lds;
  unsigned char* const v_lds = lds + S::kKeyBytes;
  int* const tile_pages = reinterpret_cast<int*>(lds + S::kKeyBytes + S::kValueBytes);  // [kWindow][kTilePages]

  const int seq = items[4 * blockIdx.x], rb = items[4 * blockIdx.x + 1];
  const int run = items[4 * blockIdx.x + 2], n_runs = max(1, items[4 * blockIdx.x + 3]);
  const SeqMeta m = seqs[seq];
  const int GS = H / G, g = blockIdx.y;
  const int HW = GS < 4 ? GS : 4, RG = 4 / HW;                     // heads and groups of 32 rows a workgroup
  const int block_rows = 32 * RG;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, quad = lane >> 4;
  const int row0 = rb * block_rows;
  if (row0 >= m.q_len) return;                                      // (the whole workgroup)
  const int nrows = min(block_rows, m.q_len - row0);
  const int p_first = m.q_start + row0, p_last = p_first + nrows - 1;
  const int* my_table = table + (long)m.table_row * table_stride;
  const int page_shift = __ffs(page_size) - 1, page_mask = page_size - 1;

  // this wave's head and rows
  const int in_group = blockIdx.z * HW + w % HW, rg = w / HW;
  const int wave_row0 = 32 * rg;
  const bool active = in_group < GS && rg < RG && wave_row0 < nrows;
  const int my_head = g * GS + (in_group < GS ? in_group : 0);
  const int wave_first = p_first + min(wave_row0, nrows - 1), wave_last = p_first + min(wave_row0 + 31, nrows - 1);
  bool row_ok[2];
  int my_pos[2], my_lo[2], seen_to[2];
  vec_t qv[2][KCH];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int row = wave_row0 + 16 * r + l16;
    row_ok[r] = active && row < nrows;
    my_pos[r] = p_first + (row_ok[r] ? row : 0);
    my_lo[r] = first_seen(my_pos[r], window, chunk);
    seen_to[r] = row_ok[r] ? my_pos[r] : -1;
    const T* q_row = q + (long)(m.q_off + row0 + (row_ok[r] ? row : 0)) * ldq + (long)my_head * D;
#pragma unroll
    for (int c = 0; c < KCH; ++c) {
      const bool in = c * KC + VEC * quad + VEC <= D;
      qv[r][c] = load_or_zero<T>(q_row + (in ? c * KC + VEC * quad : 0), row_ok[r] && in);
    }
  }
  const int wave_lo_last = first_seen(wave_last, window, chunk);
  const float* my_bias = dist_bias ? dist_bias + (long)my_head * n_dist : nullptr;

  float m_run[2], l_run[2];
  f32x4 acc[2][VB];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    m_run[r] = kNegSentinel;
    l_run[r] = 0.f;
#pragma unroll
    for (int b = 0; b < VB; ++b) acc[r][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  const int block_lo = first_seen(p_first, window, chunk);           // no row of the block sees a key in front of it (but kept ones)
  const int lo_tile = block_lo / TK;
  const int hi_tile = p_last / TK;
  const int kept_tiles = min((keep_first + TK - 1) / TK, lo_tile);   // tiles of kept first tokens below the window's
  const int n_tiles = kept_tiles + hi_tile - lo_tile + 1;
  auto tile_at = [&](int step) LS_INLINED { return step < kept_tiles ? step : lo_tile + (step - kept_tiles); };
  const int per_run = (n_tiles + n_runs - 1) / n_runs;
  const int step_begin = run * per_run, step_end = min(n_tiles, (run + 1) * per_run);

  // The page ids of kWindow tiles at a time, by ordinary loads while no tile's load is in flight.  Keys behind the block's last row have the
  // page of that row, pages that were given back page 0: what is loaded from there is masked, or cleared in LDS.
  auto fill_pages = [&](int first_step) LS_INLINED {
    for (int idx = threadIdx.x; idx < S::kWindow * S::kTilePages; idx += 256) {
      const int step = first_step + idx / S::kTilePages;
      if (step < step_end) {
        const int key = min(((tile_at(step) * TK >> page_shift) + idx % S::kTilePages) << page_shift, p_last);
        tile_pages[idx] = max(my_table[key >> page_shift], 0);
      }
    }
  };
  auto opens = [&](int step) LS_INLINED { return (step - step_begin) % S::kWindow == 0; };

  // Loads.  Piece p of the keys is slot p % KP of key p / KP; piece p of the values is VEC keys (p / DV) of column p % DV.
  // ONE_PAGE: lane i of `from` holds where the wave's key load i starts, lane 32 + i where its value load i does, and a
  // lane's offset from there is the same for every tile.
  constexpr int KO = ONE_PAGE ? KPER : 1;
  unsigned k_off[KO];
  const unsigned v_off = ONE_PAGE ? (unsigned)((lane << page_shift) * SZ) : 0u;   // (64 columns from the load's first)
  auto group_of = [&](int load) LS_INLINED { return (load * 256 + w * 64) / (8 * KP) * 8; };   // first of the eight keys a load lies in
#pragma unroll
  for (int i = 0; i < KO; ++i) {
    const int p = i * 256 + (int)threadIdx.x, key = p / KP;
    k_off[i] = (unsigned)(((key - group_of(i)) * D + slot_of_piece<T>(key, p % KP) * VEC) * SZ);
  }
  const bool values_lane = lane >= 32;
  const int my_load = lane & 31;
  const int my_piece = values_lane && my_load < VPER ? my_load * 256 + w * 64 : 0, my_col = my_piece % DV;   // (the waves' first columns differ where DV does not divide 256)
  const int my_key = values_lane ? my_piece / DV * VEC : (my_load < KPER ? group_of(my_load) : 0);
  auto loads_of = [&](int step) LS_INLINED -> unsigned long long {
    const int key = tile_at(step) * TK + my_key;
    const int id = tile_pages[(step - step_begin) % S::kWindow * S::kTilePages + (key >> page_shift) - (tile_at(step) * TK >> page_shift)];
    const long page = (long)id * G + g;
    return values_lane ? (unsigned long long)(v_pages + ((page * DV + my_col) << page_shift) + (key & page_mask))
                       : (unsigned long long)(k_pages + ((page << page_shift) + (key & page_mask)) * D);
  };
  auto load_at = [&](unsigned long long from, int index) LS_INLINED -> unsigned long long {
    return (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(unsigned)from, index) |
           (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(unsigned)(from >> 32), index) << 32;
  };
  const unsigned lds_base = __builtin_amdgcn_readfirstlane((unsigned)(unsigned long)(lptr_t)lds) + w * 1024;
  auto load_k = [&](unsigned long long from, int i) LS_INLINED {
    load_to_lds16_from(load_at(from, i), k_off[i % KO], lds_base + i * 4096);
  };
  auto load_v = [&](unsigned long long from, int i) LS_INLINED {
    load_to_lds16_from(load_at(from, 32 + i), v_off, lds_base + S::kKeyBytes + i * 4096);
  };
  auto request = [&](int step, auto values) LS_INLINED {              // all of a tile's keys, or values
    constexpr bool V = decltype(values)::value;
    if constexpr (ONE_PAGE) {
      const unsigned long long from = loads_of(step);
#pragma unroll
      for (int i = 0; i < (V ? VPER : KPER); ++i) {
        if (V) load_v(from, i);
        else load_k(from, i);
      }
    } else {
      const int key0 = tile_at(step) * TK;
      const int* pages = tile_pages + (step - step_begin) % S::kWindow * S::kTilePages;
#pragma unroll
      for (int i = 0; i < (V ? VPER : KPER); ++i) {
        if (i * 256 + w * 64 >= (V ? V_TOTAL : K_TOTAL)) break;       // uniform for the wave
        const int p = min(i * 256 + (int)threadIdx.x, (V ? V_TOTAL : K_TOTAL) - 1);
        const int key = V ? p / DV * VEC : p / KP;
        const long page = (long)pages[((key0 + key) >> page_shift) - (key0 >> page_shift)] * G + g;
        const int slot = (key0 + key) & page_mask;
        const T* src = V ? v_pages + ((page * DV + p % DV) << page_shift) + slot
                         : k_pages + ((page << page_shift) + slot) * D + slot_of_piece<T>(key, p % KP) * VEC;
        load_to_lds16(src, (lptr_t)((V ? v_lds : k_lds) + (i * 256 + w * 64) * 16));
      }
    }
  };
  constexpr std::false_type keys{};
  constexpr std::true_type values{};
  // where a lane's fragment of chunk c lies, but for a constant: the swizzle repeats every PERIOD chunks
  constexpr int PERIOD = KP % 16 == 0 ? 4 : KP % 8 == 0 ? 2 : 1;
  const unsigned char* k_at[PERIOD];
#pragma unroll
  for (int c = 0; c < PERIOD; ++c) k_at[c] = k_lds + (key_of_row<T>(0, l16) * KP + slot_at<T>(l16, 4 * c + quad)) * 16;

  const unsigned char* const v_at = v_lds + (quad * DV + l16) * 16;   // (a value operand: this and constants)

#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < KCH; ++c) __asm__ volatile("" ::"v"(qv[r][c]));  // the query rows are awaited here, not inside the loop
  for (int step = step_begin; step < step_end; ++step) {
    const int key0 = tile_at(step) * TK;
    const bool fresh = opens(step);          // the tile's page ids were not there when the tile before ran
    if (fresh) {
      ring_barrier();
      fill_pages(step);
      __syncthreads();
      request(step, keys);
      request(step, values);
    }
    wait_loads<0>();
    ring_barrier();                          // the keys are there, and every wave has read the values before
    const bool mine = active && key0 <= wave_last;
    if (!fresh && !(ONE_PAGE && mine)) request(step, values);
    // -- 1. transposed scores of the tile's groups of 16 keys; two groups in turn, the values' loads between ------
    f32x4 s[2][NG];
    auto score_products = [&](auto with_loads) LS_INLINED {
      constexpr int N = NG * KCH, RING = N < 4 ? N : 4;
      constexpr int PLACES = N < VPER ? 1 : N / VPER;                 // products a load
      constexpr int AT_ONCE = N < VPER ? (VPER + N - 1) / N : 1;      // loads at such a place
      auto group = [](int idx) constexpr { return 2 * (idx / (2 * KCH)) + idx % 2; };
      auto chunk_of = [](int idx) constexpr { return idx / 2 % KCH; };
      auto k_read = [&](int idx) LS_INLINED -> vec_t {
        const int c = chunk_of(idx);
        const unsigned char* src = k_at[c % PERIOD] + (key_of_row<T>(group(idx), 0) * KP + (c - c % PERIOD) * 4) * 16;
        const bool in = KP % 4 == 0 || c * 4 + quad < KP;
        vec_t kf = *reinterpret_cast<const vec_t*>(in ? src : k_lds);
        return in ? kf : A::zero();
      };
      unsigned long long from = 0;
      if constexpr (decltype(with_loads)::value) from = loads_of(step);
      vec_t ring[RING];
#pragma unroll
      for (int i = 0; i < RING; ++i) ring[i] = k_read(i);
      __builtin_amdgcn_sched_barrier(0);     // (left to itself the compiler reads an operand when it is needed)
#pragma unroll
      for (int idx = 0; idx < N; ++idx) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          if (chunk_of(idx) == 0) s[r][group(idx)] = f32x4{0.f, 0.f, 0.f, 0.f};
          A::mma(s[r][group(idx)], ring[idx % RING], qv[r][chunk_of(idx)]);
        }
        if (idx + RING < N) ring[idx % RING] = k_read(idx + RING);
        if constexpr (decltype(with_loads)::value) {
          if (idx % PLACES == 0) {
#pragma unroll
            for (int n = idx / PLACES * AT_ONCE; n < (idx / PLACES + 1) * AT_ONCE && n < VPER; ++n) load_v(from, n);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    __builtin_amdgcn_s_setprio(1);
    if (mine) {
      if (ONE_PAGE && !fresh) score_products(std::bool_constant<ONE_PAGE>{});
      else score_products(std::false_type{});
    }
    __builtin_amdgcn_s_setprio(0);
    ring_barrier();                          // every wave has read these keys
    const bool ahead = step + 1 < step_end && !opens(step + 1);
    if (ahead && !(ONE_PAGE && mine)) request(step + 1, keys);
    vec_t pb[2][NC];
    float shrink[2] = {1.f, 1.f};            // of the sums so far; they are multiplied where the products add to them
    if (mine) {
      // -- 2. scale, bias, mask, online softmax; the next keys' loads among it --------------------------------
      unsigned long long from = 0;
      if (ONE_PAGE && ahead) from = loads_of(step + 1);
      auto softmax_tile = [&](auto whole, auto biased, auto with_loads) LS_INLINED {
        constexpr bool kWhole = decltype(whole)::value, kBiased = decltype(biased)::value;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          float top = kNegSentinel;
#pragma unroll
          for (int ng = 0; ng < NG; ++ng)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int key = key0 + key_of_row<T>(ng, 4 * quad + i);
              const bool see = kWhole || ((key <= seen_to[r]) & ((key >= my_lo[r]) | (key < keep_first)));
              float v = s[r][ng][i] * scale;
              if constexpr (kBiased) v = v + my_bias[min(max(my_pos[r] - key, 0), n_dist - 1)];
              v = see ? v : -__builtin_huge_valf();                   // (its weight is then exp(-inf) = 0)
              s[r][ng][i] = v;
              top = fmaxf(top, v);
              // four biases at a time where the registers of all would not be there; else their loads stand together (700 tokens
              // from 1,500 on in a window of 600, keys and values of 40 elements, 32.9 -> 27.9 us, of 64 32.3 -> 28.6)
              if constexpr (kBiased && S::kRowRegisters > 8) {
                if (i == 3) __builtin_amdgcn_sched_barrier(0);
              }
            }
          top = quad16_max(top);
          const float m_new = fmaxf(m_run[r], top);
          shrink[r] = softmax_exp<T>(m_run[r] - m_new);
          float sum = 0.f;
#pragma unroll
          for (int ng = 0; ng < NG; ++ng) {
            float p[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              p[i] = softmax_exp<T>(s[r][ng][i] - m_new);
              pb[r][ng * NC / NG][(sizeof(T) == 2 ? ng % 2 * 4 : 0) + i] = from_f32<T>(p[i]);
            }
            sum = sum + ((p[0] + p[1]) + (p[2] + p[3]));
            if constexpr (decltype(with_loads)::value) {
              constexpr int PLACES = 2 * NG;
#pragma unroll
              for (int n = (r * NG + ng) * KPER / PLACES; n < (r * NG + ng + 1) * KPER / PLACES; ++n) load_k(from, n);
            }
          }
          sum = quad16_sum(sum);
          l_run[r] = l_run[r] * shrink[r] + sum;
          m_run[r] = m_new;
        }
      };
      const bool whole_tile = key0 + TK - 1 <= wave_first && (key0 >= wave_lo_last || key0 + TK <= keep_first) && wave_row0 + 31 < nrows;
      auto softmax_of = [&](auto biased, auto with_loads) LS_INLINED {
        if (whole_tile) softmax_tile(std::true_type{}, biased, with_loads);
        else softmax_tile(std::false_type{}, biased, with_loads);
      };
      if (my_bias) {                         // (its loads are ordinary ones, whose waits would be for the keys' too)
        if (ONE_PAGE && ahead) request(step + 1, keys);
        softmax_of(std::true_type{}, std::false_type{});
      } else {
        if (ONE_PAGE && ahead) softmax_of(std::false_type{}, std::bool_constant<ONE_PAGE>{});
        else softmax_of(std::false_type{}, std::false_type{});
      }
    }
    // the values have landed; the next keys, asked for after them, are still on their way
    if (ONE_PAGE && ahead) wait_loads<ONE_PAGE ? KPER : 0>();
    else wait_loads<0>();
    ring_barrier();
    if (key0 + TK - 1 > p_last || (key0 < block_lo && key0 + TK > keep_first)) {   // uniform: clear the values of keys that are not held
#pragma unroll
      for (int i = 0; i < VPER; ++i) {
        const int p = i * 256 + (int)threadIdx.x;
        if (p >= V_TOTAL) break;
        vec_t* at = reinterpret_cast<vec_t*>(v_lds + p * 16);
        vec_t v = *at;
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          const int key = key0 + p / DV * VEC + e;
          if (!(key <= p_last && (key >= block_lo || key < keep_first))) v[e] = (T)0.f;
        }
        *at = v;
      }
      ring_barrier();
    }
    if (mine) {
      // -- 3. values ---------------------------------------------------------------------------
      constexpr int N = VB * NC, RING = N < 4 ? N : 4;
      auto v_read = [&](int idx) LS_INLINED -> vec_t {
        const bool in = DV % 16 == 0 || 16 * (idx / NC) + l16 < DV;
        vec_t a = *reinterpret_cast<const vec_t*>((in ? v_at : v_lds) + (4 * (idx % NC) * DV + (in ? 16 * (idx / NC) : 0)) * 16);
        return in ? a : A::zero();
      };
      __builtin_amdgcn_s_setprio(1);
      vec_t ring[RING];
#pragma unroll
      for (int i = 0; i < RING; ++i) ring[i] = v_read(i);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int idx = 0; idx < N; ++idx) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          if (idx % NC == 0)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[r][idx / NC][i] = acc[r][idx / NC][i] * shrink[r];
          A::mma(acc[r][idx / NC], ring[idx % RING], pb[r][idx % NC]);
        }
        if (idx + RING < N) ring[idx % RING] = v_read(idx + RING);
        __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_s_setprio(0);
    }
  }

  if (!active) return;
  const bool vec_ok = DV % 16 == 0 && ldo % 4 == 0 && reinterpret_cast<uintptr_t>(out) % (4 * SZ) == 0;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    if (!row_ok[r]) continue;
    const int row = wave_row0 + 16 * r + l16;
    if (n_runs > 1) {
      typedef __attribute__((ext_vector_type(2))) float f32x2;
      float* dst = part + (((long)blockIdx.x * part_rows + row) * H + my_head) * (DV + 2);
#pragma unroll
      for (int b = 0; b < VB; ++b) {
        if constexpr (DV % 16 == 0) {        // (rows of an even number of floats)
          *reinterpret_cast<f32x2*>(dst + 16 * b + 4 * quad) = f32x2{acc[r][b][0], acc[r][b][1]};
          *reinterpret_cast<f32x2*>(dst + 16 * b + 4 * quad + 2) = f32x2{acc[r][b][2], acc[r][b][3]};
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (16 * b + 4 * quad + i < DV) dst[16 * b + 4 * quad + i] = acc[r][b][i];
        }
      }
      if (quad == 0) {
        dst[DV] = m_run[r];
        dst[DV + 1] = l_run[r];
      }
      continue;
    }
    float top = m_run[r], total = l_run[r], keep = 1.0f;
    if (sink) {
      const float sv = sink[my_head];
      top = fmaxf(m_run[r], sv);
      keep = softmax_exp<T>(m_run[r] - top);
      total = l_run[r] * keep + softmax_exp<T>(sv - top);
    }
    const float inv = keep / total;
    T* dst = out + (long)(m.q_off + row0 + row) * ldo + (long)my_head * DV;
    const float* g_row = gate ? gate + (long)(m.q_off + row0 + row) * ldg + (long)my_head * DV : nullptr;
#pragma unroll
    for (int b = 0; b < VB; ++b) {
      typedef typename std::conditional<sizeof(T) == 2, bf16x4, f32x4>::type v4_t;
      v4_t o;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = 16 * b + 4 * quad + i;
        float v = acc[r][b][i] * inv;
        if (g_row && c < DV) v = v * sigmoid_f(g_row[c]);
        o[i] = from_f32<T>(v);
        if (!vec_ok && c < DV) dst[c] = o[i];
      }
      if (vec_ok) *reinterpret_cast<v4_t*>(dst + 16 * b + 4 * quad) = o;
    }
  }
}

// Fold the runs of row blocks: a fold item (first work item, runs, first packed row, rows) names the work items
// first .. first + runs - 1 of one row block, whose partial results are folded in ascending order for each of its
// rows; the sink joins the sum and the gate multiplies the result.  One workgroup a (fold item, head, row).
template <typename T>
__global__ __launch_bounds__(64) void sink_combine_kernel(const float* __restrict__ part, int part_rows, int H,
                                                          const int* __restrict__ folds, const float* __restrict__ sink,
                                                          const float* __restrict__ gate, long ldg, T* __restrict__ out,
                                                          long ldo) {
  const int first = folds[4 * blockIdx.x], n_runs = folds[4 * blockIdx.x + 1];
  const int row0 = folds[4 * blockIdx.x + 2], rows = folds[4 * blockIdx.x + 3];
  const int h = blockIdx.y;
  const long stride = (long)part_rows * H * (DV + 2);  // from a run to the next
  __shared__ float factor_s[64];
  for (int r = blockIdx.z; r < rows; r += gridDim.z) {
    const float* mine = part + (((long)first * part_rows + r) * H + h) * (DV + 2);
    // lane k holds run k's statistics (runs <= 64): all of them are requested at once
    const int k_mine = threadIdx.x;
    const float m_k = k_mine < n_runs ? mine[k_mine * stride + DV] : kNegSentinel;
    const float l_k = k_mine < n_runs ? mine[k_mine * stride + DV + 1] : 0.f;
    const float sink_h = sink ? sink[h] : kNegSentinel;
    const float top = fmaxf(sink_h, wave_max(m_k));
    const float f_k = k_mine < n_runs ? softmax_exp<T>(m_k - top) : 0.f;
    __syncthreads();
    factor_s[k_mine] = f_k;
    float total = 0.f;
    for (int k = 0; k < n_runs; ++k)   // ascending
      total = total + __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, l_k), k)) *
                          __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f_k), k));
    if (sink) total = total + softmax_exp<T>(sink_h - top);
    const float inv = 1.0f / total;
    __syncthreads();
    for (int c = threadIdx.x; c < DV; c += 64) {
      float sum = 0.f;
      int k = 0;
      for (; k + 4 <= n_runs; k += 4) {
        const float p0 = mine[k * stride + c], p1 = mine[(k + 1) * stride + c], p2 = mine[(k + 2) * stride + c],
                    p3 = mine[(k + 3) * stride + c];
        sum = (((sum + p0 * factor_s[k]) + p1 * factor_s[k + 1]) + p2 * factor_s[k + 2]) + p3 * factor_s[k + 3];
      }
      for (; k < n_runs; ++k) sum = sum + mine[k * stride + c] * factor_s[k];
      float v = sum * inv;
      if (gate) v = v * sigmoid_f(gate[(long)(row0 + r) * ldg + (long)h * DV + c]);
      out[(long)(row0 + r) * ldo + h * DV + c] = from_f32<T>(v);
    }
  }
}

}  // namespace ls

LS_DEFINE_ERROR_API

using namespace ls;

extern "C" int ls_sink_dim() { return D; }
extern "C" int ls_sink_vdim() { return DV; }
extern "C" int ls_sink_max_row_tiles() { return 4; }
// The staged kernel for prompt portions: keys of a tile (0: this library's sizes do not fit it) and rows of a work
// item's block for H query heads over G key/value heads.
extern "C" int ls_sink_staged_keys(int dtype) {
  if (dtype == kF32) return Staged<float>::kFits ? Staged<float>::kKeys : 0;
  return Staged<bf16_t>::kFits ? Staged<bf16_t>::kKeys : 0;
}
extern "C" int ls_sink_staged_rows(int H, int G) {
  const int GS = H / (G > 0 ? G : 1);
  return 32 * (4 / (GS < 4 ? (GS > 0 ? GS : 1) : 4));
}

// q [T][ldq] (H heads of D); key pages [pages][G][page_size][D], value pages [pages][G][DV][page_size]; table
// [slots][table_stride]; seqs: the step's requests; items: n_items work items of four ints (request of the step,
// block of 16 row_tiles of its rows, run, runs); row_tiles 1, 2 or 4, or 0 for a step of single decoded tokens.
// sink [H] float or null; dist_bias [H][n_dist] float or null; gate: float [T][ldg] (H heads of DV) or null;
// out [T][ldo].  Work items with runs > 1 leave their results in part (n_items * part_rows * H * (DV + 2) floats;
// part_rows 16 row_tiles, or 1 for decoded tokens) and the n_folds fold items of four ints (first work item, runs,
// first packed row, rows) say which to fold into which rows of out in a second launch.
extern "C" int ls_sink_attention(int dtype, const void* q, long ldq, const void* k_pages, const void* v_pages,
                                 int page_size, const int* table, int table_stride, const void* seqs,
                                 const int* items, int n_items, int row_tiles, int H, int G, float scale, int window,
                                 int chunk, int keep_first, const float* sink, const float* dist_bias, int n_dist, const float* gate,
                                 long ldg, void* out, long ldo, const int* folds, int n_folds, float* part,
                                 int part_rows, void* stream) {
  LS_REQUIRE(row_tiles == 0 || row_tiles == 1 || row_tiles == 2 || row_tiles == 4 || row_tiles == 8,
             "sink_attention: %d row tiles", row_tiles);
  LS_REQUIRE(H > 0 && G > 0 && H % G == 0, "sink_attention: %d query heads over %d key/value heads", H, G);
  LS_REQUIRE(part_rows == (row_tiles == 8 ? ls_sink_staged_rows(H, G) : row_tiles ? 16 * row_tiles : 1),
             "sink_attention: partial results of %d rows", part_rows);
  LS_REQUIRE(row_tiles != 8 || (ls_sink_staged_keys(dtype) > 0 && page_size % (dtype == kF32 ? 4 : 8) == 0),
             "sink_attention: the staged kernel does not take these sizes (page size %d)", page_size);
  LS_REQUIRE(n_folds >= 0 && (n_folds == 0 || (part && folds)), "sink_attention: %d fold items need partial results", n_folds);
  LS_REQUIRE(n_items > 0 && q && k_pages && v_pages && table && seqs && items && out, "sink_attention: null operand");
  LS_REQUIRE(ldq >= (long)H * D && ldo >= (long)H * DV && (!gate || ldg >= (long)H * DV), "sink_attention: rows are too short");
  LS_REQUIRE(page_size >= 4 && (page_size & (page_size - 1)) == 0 && table_stride > 0,
             "sink_attention: page size %d is not a power of two", page_size);
  LS_REQUIRE(window >= 0 && chunk >= 0 && (!dist_bias || n_dist > 0), "sink_attention: window %d, chunk %d, %d distances",
             window, chunk, n_dist);
  LS_REQUIRE(keep_first >= 0 && (keep_first == 0 || (window > 0 && chunk == 0)),
             "sink_attention: %d kept first tokens need a window (and no chunks)", keep_first);
  LS_REQUIRE(reinterpret_cast<uintptr_t>(q) % 16 == 0 && reinterpret_cast<uintptr_t>(k_pages) % 16 == 0 &&
                 reinterpret_cast<uintptr_t>(v_pages) % 16 == 0,
             "sink_attention: operands must be 16-byte aligned");
  LS_REQUIRE(dtype == kF32 || dtype == kBF16, "sink_attention: unknown dtype %d", dtype);
  LS_REQUIRE(ldq % (dtype == kF32 ? 4 : 8) == 0, "sink_attention: query rows must be 16-byte aligned");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int GS = H / G;
#define LS_SINK_LAUNCH(T_, RT_, DEC_)                                                                                  \
  hipLaunchKernelGGL((sink_attention_kernel<T_, RT_, DEC_>),                                                           \
                     dim3(n_items, G, DEC_ ? (GS + 15) / 16 : (GS + kMaxWaves - 1) / kMaxWaves),                       \
                     dim3(DEC_ ? 64 : 64 * (GS < kMaxWaves ? GS : kMaxWaves)), 0, s, (const T_*)q, ldq,                \
                     (const T_*)k_pages, (const T_*)v_pages, page_size, table, table_stride, (const SeqMeta*)seqs,     \
                     items, H, G, scale, window, chunk, keep_first, sink, dist_bias, n_dist, gate, ldg, (T_*)out, ldo, \
                     part, part_rows)
#define LS_SINK_STAGED_AS(T_, ONE_PAGE_)                                                                               \
  hipLaunchKernelGGL((sink_attention_staged_kernel<T_, ONE_PAGE_>), dim3(n_items, G, (GS + 3) / 4), dim3(256), 0, s,   \
                     (const T_*)q, ldq, (const T_*)k_pages, (const T_*)v_pages, page_size, table, table_stride,        \
                     (const SeqMeta*)seqs, items, H, G, scale, window, chunk, keep_first, sink, dist_bias, n_dist,     \
                     gate, ldg, (T_*)out, ldo, part, part_rows)
#define LS_SINK_STAGED(T_)                                                                                             \
  if (Staged<T_>::kOnePage && page_size >= 8) LS_SINK_STAGED_AS(T_, Staged<T_>::kOnePage);                             \
  else LS_SINK_STAGED_AS(T_, false)
#define LS_SINK_BY_ROWS(T_)                       \
  switch (row_tiles) {                            \
    case 0: LS_SINK_LAUNCH(T_, 1, true); break;   \
    case 1: LS_SINK_LAUNCH(T_, 1, false); break;  \
    case 2: LS_SINK_LAUNCH(T_, 2, false); break;  \
    case 4: LS_SINK_LAUNCH(T_, 4, false); break;  \
    default: LS_SINK_STAGED(T_); break;           \
  }
  if (dtype == kF32) {
    LS_SINK_BY_ROWS(float)
    if (n_folds > 0)
      hipLaunchKernelGGL(sink_combine_kernel<float>, dim3(n_folds, H, part_rows), dim3(64), 0, s, part, part_rows, H,
                         folds, sink, gate, ldg, (float*)out, ldo);
  } else {
    LS_SINK_BY_ROWS(bf16_t)
    if (n_folds > 0)
      hipLaunchKernelGGL(sink_combine_kernel<bf16_t>, dim3(n_folds, H, part_rows), dim3(64), 0, s, part, part_rows, H,
                         folds, sink, gate, ldg, (bf16_t*)out, ldo);
  }
#undef LS_SINK_BY_ROWS
#undef LS_SINK_STAGED
#undef LS_SINK_STAGED_AS
#undef LS_SINK_LAUNCH
  return check_launch("sink_attention");
}
