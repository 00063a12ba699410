// The loop of every product whose operands come through rings in LDS (gemm_ring.h, experts.hip): a workgroup's tile of
// weight rows times rows of X, stage by stage, loads, waits, fragments and multiplications in the order written here.
//
// A stage is SUB parts of 128 bytes of K of all the tile's rows (two chunks of 64 bytes a part), W's rows and X's rows in rings of their
// own (the ring of W may be longer: its lines come from HBM, X's mostly from the XCD's L2).  Within a part the 16-byte piece q of
// row r lies in slot q ^ (r & 7) of the row's 128 bytes, so that the sixteen rows a fragment read takes together lie in different
// banks; a lane of a load picks its piece accordingly, inside the same 128-byte line.
//
// How the steps interlock (WS and XS stages of W and X in LDS, one barrier a stage):
//   first half of stage st:  multiply its first SUB chunks, read the fragments of the others;
//                            request W's stage st + WS - 1 into the buffer that stage st - 1 left;
//   wait until the own loads of stage st + 1 are there, then the barrier: now stage st + 1 is whole, and
//   everyone's reads of stage st are done (lgkmcnt(0) in front of the barrier);
//   second half:             request X's stage st + XS into the buffer of stage st;
//                            multiply the other chunks, read the first fragments of stage st + 1.
// Loads complete in the order of their issue, so a wait counts the younger ones.  The last WS - 1 stages request nothing and wait for
// all that is in flight (an instance of the loop's body of its own, so that no stage has a branch; requesting stages beyond the end,
// which answer zeros, in order to keep the counts cost 10 % where K is 1,024 and less; only the largest tile, which would spill with four
// instances, does that).  All loads have landed when the loop returns, so no workgroup
// ends with LDS still being written.
//
// What bounds it, and why the order is written out: a CU takes a load into LDS every 16 cycles at best, and a wave that issues
// several in a row stands behind the other waves' and multiplies nothing meanwhile; a fragment comes 100 cycles and more after it was
// asked for; and the compiler, left to itself, moves the reads of a half stage to its end, behind all the products, and the fold of
// a K slice to where the slice ends, as a block of additions in front of which the matrix cores run dry.  So a scheduling barrier ends
// every few products, with one load or read among them, and the sums of a finished slice are added to the totals one tile at a
// time, each in front of the product that starts that tile's next slice from zero.  2,048 rows, weights from HBM, us (before / this
// order; bfloat16): SwiGLU 24,576 x 4,096 353 / 326 (256 x 192 outputs a workgroup; without any load in the loop 283), 6,144 x 4,096
// 96 / 83, 4,096 x 12,288 191 / 177, 1,024 x 2,048 17.6 / 15.6; 8 rows SwiGLU 24,576 x 4,096 43.7 / 39.0 (64 x 64).
//
// Fragments are kept twice, a half stage's read during the half before it, or (IN_PLACE, from eight products a chunk on, where
// twice would spill) once: the weight tiles in two groups, a group's columns one after the other, every fragment replaced as soon
// as its last product is issued, at least TJ * TI / 2 products before its next use.  With the barrier between the second half's two
// groups nothing is read from a stage that is not whole, and the reads that the barrier waits for are a group old.
//
// Stages of two parts (SUB 2) have a barrier and an LDS latency every 128 elements of K: worth it where few products stand between
// two barriers and one workgroup has the CU (97 x 1,024 x 2,048 in tiles of 64 x 64: 10.2 / 9.4 us), not where a second one fills the gaps.
//
// float32 multiplies four times as long a byte: with four tiles a wave the compiler's own order has products enough between a read and
// its use, and the order above only holds products back (us, above / compiler's: 128 x 6,144 x 5,120 102.0 / 99.0, 256 x 3,072 x 12,288
// 238 / 229, SwiGLU 256 x 4,096 x 4,096 85.6 / 79.5, slice sums 40 x 10,240 x 8,192 102.1 / 94.0; 2,000 x 6,144 x 1,024 level).  With one
// or two tiles it stays ahead (32 x 32, 128 x 4,096 x 12,288 136 / 153).
#pragma once

#include <type_traits>

#include "common.h"
#include "ring.h"

namespace ls {

// TI weight tiles and TJ row tiles of 16 a wave, its weight tiles W_TILE bytes of LDS apart; W_ROWS and X_ROWS rows of the workgroup;
// LW and LX loads a wave and stage.  FOLD: K slices are folded in ascending order into total (else acc is one chain over all of K).
template <typename T, int TI, int TJ, int W_TILE, int W_ROWS, int X_ROWS, int LW, int LX, int WS, int XS, int SUB, bool FOLD>
struct RingProduct {
  typedef Atom<T> A;
  typedef typename A::vec_t vec_t;
  static constexpr int W_BYTES = SUB * W_ROWS * 128, X_BYTES = SUB * X_ROWS * 128;
  static constexpr int LDS_BYTES = WS * W_BYTES + XS * X_BYTES;
  static constexpr bool IN_PLACE = SUB == 1 && TI % 2 == 0 && TI * TJ >= 8;
  static constexpr bool TAIL = TI * TJ < 24;
  static constexpr bool ORDERED = sizeof(T) == 2 || TI * TJ < 4;
  static_assert(WS >= XS && XS >= 2 && WS >= 3, "rings");
  static_assert(!TAIL || WS <= XS + 1, "X's last stage is requested before the tail begins");
  static_assert(LDS_BYTES <= 160 * 1024, "the rings fit the LDS of a CU");

  f32x4 total[TI][TJ], acc[TI][TJ];  // [weight tile][row tile]

  static __device__ __forceinline__ void in_order() {
    if constexpr (ORDERED) __builtin_amdgcn_sched_barrier(0);
  }

  template <bool FIRST>  // FIRST: the tile's first product of a slice
  __device__ __forceinline__ void product(int i, int j, const vec_t& a, const vec_t& b) {
    if constexpr (FIRST) {
      if constexpr (FOLD) {
#pragma unroll
        for (int r = 0; r < 4; ++r) total[i][j][r] = total[i][j][r] + acc[i][j][r];
        __asm__ volatile("" : "+v"(total[i][j]));  // here, and not where the slice ends: until then both would be alive
      }
      acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    A::mma(acc[i][j], a, b);
  }

  // w_at, x_at: this wave's first weight and row tile in the first stage.  request_w(st, buf, n), request_x(st, buf, n): load n of
  // stage st into buffer buf.  slice_done(st): called in front of stage st, where a slice of per_slice stages has ended.
  // (Behind the loop the fragments of a stage that is not there have been read: nobody uses them.)
  template <typename RequestW, typename RequestX, typename SliceDone>
  __device__ __forceinline__ void run(const unsigned char* w_at, const unsigned char* x_at, int stages, int per_slice,
                                      RequestW request_w, RequestX request_x, SliceDone slice_done) {
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    const int lane = threadIdx.x & 63;
    const unsigned at = (lane & 15) * 128 + (((lane >> 4) ^ (lane & 7)) << 4);
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j) total[i][j] = acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // a lane's 16 bytes of chunk c of a tile; the odd chunk of a part lies four slots (64 bytes) across
    auto w_frag = [&](int buf, int i, int c) LS_INLINED {
      return *reinterpret_cast<const vec_t*>(w_at + buf * W_BYTES + (c >> 1) * W_ROWS * 128 + (at ^ ((c & 1) * 64)) + i * W_TILE);
    };
    auto x_frag = [&](int buf, int j, int c) LS_INLINED {
      return *reinterpret_cast<const vec_t*>(x_at + buf * X_BYTES + (c >> 1) * X_ROWS * 128 + (at ^ ((c & 1) * 64)) + j * 2048);
    };

#pragma unroll
    for (int s = 0; s < WS; ++s) {
      if (s < XS && (!TAIL || s < stages))
#pragma unroll
        for (int n = 0; n < LX; ++n) request_x(s, s, n);
      if (s < WS - 1 && (!TAIL || s < stages))
#pragma unroll
        for (int n = 0; n < LW; ++n) request_w(s, s, n);
    }
    if (!TAIL || stages >= WS) wait_loads<(XS - 1) * LX + (WS - 2) * LW>(); else wait_loads<0>();
    ring_barrier();
    // in flight behind what stage st + 1 needs, when stage st waits for it: W's last stage and XS - 2 whole stages (XS == WS: no
    // newer W than X's)
    constexpr int YOUNGER = (XS - 2) * (LX + LW) + (XS < WS ? LW : 0);
    int wb = 0, xb = 0;
    auto before = [](int buf, int n) LS_INLINED { return buf == 0 ? n - 1 : buf - 1; };
    auto after = [](int buf, int n) LS_INLINED { return buf + 1 == n ? 0 : buf + 1; };

    // stage(first, load, st) for every stage; those that load run to the one that requests W's last stage (and X's, or where
    // XS == WS one behind it: zeros)
    auto all_stages = [&](auto stage) LS_INLINED {
      int st = 0, left = 0;  // stages of this slice to come
      auto up_to = [&](auto load, int end) LS_INLINED {
        while (st < end) {
          if (left == 0) {
            if (st) slice_done(st);
            stage(yes, load, st);
            ++st;
            left = per_slice - 1;
          }
          const int stop = min(end, st + left);
          left -= stop - st;
          for (; st < stop; ++st) stage(no, load, st);
        }
      };
      if constexpr (TAIL) up_to(yes, stages - WS + 1);
      up_to(std::bool_constant<!TAIL>(), stages);
    };
    if constexpr (!IN_PLACE) {
      vec_t a[2][SUB][TI], b[2][SUB][TJ];
      auto read = [&](int set, int wbuf, int xbuf, int half) LS_INLINED {
#pragma unroll
        for (int u = 0; u < SUB; ++u) {
#pragma unroll
          for (int j = 0; j < TJ; ++j) b[set][u][j] = x_frag(xbuf, j, half * SUB + u);
#pragma unroll
          for (int i = 0; i < TI; ++i) a[set][u][i] = w_frag(wbuf, i, half * SUB + u);
        }
        in_order();
      };
      auto multiply = [&](auto first, int set, auto load, auto loads) LS_INLINED {
        constexpr int ROWS = SUB * TI, L = decltype(loads)::value;
#pragma unroll
        for (int u = 0; u < SUB; ++u)
#pragma unroll
          for (int i = 0; i < TI; ++i) {
#pragma unroll
            for (int n = 0; n < L; ++n)
              if (n * ROWS / L == u * TI + i) load(n);
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
              if (u == 0) product<decltype(first)::value>(i, j, a[set][u][i], b[set][u][j]);
              else product<false>(i, j, a[set][u][i], b[set][u][j]);
            }
            in_order();
          }
      };
      read(0, 0, 0, 0);
      all_stages([&](auto first, auto load, int st) LS_INLINED {
        constexpr bool LOAD = decltype(load)::value;
        const int w_left = before(wb, WS), x_left = xb;
        read(1, wb, xb, 1);
        multiply(first, 0, [&](int n) LS_INLINED { request_w(st + WS - 1, w_left, n); },
                 std::integral_constant<int, LOAD ? LW : 0>());
        wait_loads<LOAD ? YOUNGER : 0>();
        ring_barrier();
        wb = after(wb, WS);
        xb = after(xb, XS);
        read(0, wb, xb, 0);
        multiply(no, 1, [&](int n) LS_INLINED { request_x(st + XS, x_left, n); }, std::integral_constant<int, LOAD ? LX : 0>());
      });
    } else {
      constexpr int G = TI / 2;
      vec_t a[TI], b[TJ];
#pragma unroll
      for (int j = 0; j < TJ; ++j) b[j] = x_frag(0, j, 0);
#pragma unroll
      for (int i = 0; i < TI; ++i) a[i] = w_frag(0, i, 0);
      // the products of half of the weight tiles, column by column; then(j) behind each
      auto columns = [&](auto first, auto group, auto then) LS_INLINED {
        constexpr int I0 = decltype(group)::value * G;
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
#pragma unroll
          for (int i = I0; i < I0 + G; ++i) product<decltype(first)::value>(i, j, a[i], b[j]);
          then(j);
          in_order();
        }
      };
      auto read_a = [&](int group, int c) LS_INLINED {
#pragma unroll
        for (int i = 0; i < G; ++i) a[group * G + i] = w_frag(wb, group * G + i, c);
      };
      constexpr std::integral_constant<int, 0> low{};
      constexpr std::integral_constant<int, 1> high{};
      all_stages([&](auto first, auto load, int st) LS_INLINED {
        constexpr bool LOAD = decltype(load)::value;
        const int w_left = before(wb, WS), x_left = xb;
        auto load_w = [&](int column) LS_INLINED {  // spread over the first half's columns
#pragma unroll
          for (int n = 0; n < LW; ++n)
            if (LOAD && n * 2 * TJ / LW == column) request_w(st + WS - 1, w_left, n);
        };
        columns(first, low, [&](int j) LS_INLINED {
          load_w(j);
          if (j == TJ - 1) read_a(0, 1);
        });
        columns(first, high, [&](int j) LS_INLINED {
          load_w(TJ + j);
          b[j] = x_frag(xb, j, 1);
          if (j == TJ - 1) read_a(1, 1);
        });
        columns(no, low, [](int) LS_INLINED {});
        wait_loads<LOAD ? YOUNGER : 0>();
        ring_barrier();
        wb = after(wb, WS);
        xb = after(xb, XS);
        read_a(0, 0);
        in_order();
        columns(no, high, [&](int j) LS_INLINED {
#pragma unroll
          for (int n = 0; n < LX; ++n)
            if (LOAD && n * TJ / LX == j) request_x(st + XS, x_left, n);
          b[j] = x_frag(xb, j, 0);
          if (j == TJ - 1) read_a(1, 0);
        });
      });
    }
    wait_loads<0>();  // (stages beyond the end)
    if constexpr (FOLD) {
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) total[i][j][r] = total[i][j][r] + acc[i][j][r];
    }
  }
};

}  // namespace ls
