// Segments of a strided scan axis in one launch: the scan axis is cut into segments of NW * U positions, a
// workgroup takes one segment of 64 * VEC adjacent rows (wave w the run [w*U, w*U + U) of every row), and the
// segments of a row are chained by decoupled look-back, row by row, through descriptors in global memory.
//   1. every lane loads its run, folds it into an affine map value_out = a * value_in + b, the maps go to LDS;
//   2. waves 0 .. VEC-1 (wave e: row e of every lane) compose the NW maps of a row, publish them, walk back over
//      the segments before until one has published the value that leaves it, and publish what leaves their own;
//   3. every wave composes the maps of the waves before it onto that value, walks its run again and stores.
// The data stays in registers (packed in 16-bit storage) between 1 and 3, so every tensor is read and written
// once: 12 / 20 bytes per element where the three launches (reduce, carry, apply: column_kernel.hpp) move 20 / 28.
//
// What bounds it: memory, and for a launch of a few microseconds the chain load -> publish -> look back -> store.
// Workgroups are numbered segment by segment, all blocks of rows of one segment next to each other: the launch
// sweeps the tensors in the order of their addresses (a matrix with its scan axis strided is stored segment after
// segment), and the segment a workgroup looks back to was started one whole round of blocks earlier.
//
// A lane's rows need not be aligned to more than an element: what a wave reads of a position that does not start on a
// 128-byte line takes one line more than it holds, whatever the phase (memory-only, 16-bit matrices of 2050 and 2052
// columns, 8 bytes to a lane: 93 and 89 us where 2048 take 64), so the wider the access the less of that, and rows off
// 16 bytes get the same widths as the others.  The line at the border of two blocks is wanted by both: such launches load
// through the caches, and eight segments are dealt out at a time so that the blocks of a segment run on one XCD and
// find the border lines in its L2 (memory-only, 16640 x 4022, 8 bytes to a lane: 101.7 us as before, 93 with cached loads,
// 85 with both; where positions start on lines cached loads cost 4 %).  On whole lines
// that order serves some fp32 backwards only (32768 x 1024 123 us instead of 130, 16384 x 4096 233 instead of 247; lookback_lanes.hpp),
// not forwards (16 x 2048 x 512 43.6 instead of 39.5).
//
// Measured (medians of launches replayed from a graph over several buffer sets, forward / backward): bf16 1 x 4096 x 2048
// (batch x time x channels) 15.1 / 22.0 us, 3.3 / 3.8 TB/s, where the three launches take 28.1 / 37.4; 8 x 4096 x 1024
// 42.1 / 64.9 us, 4.8 / 5.2 TB/s, where the column drift kernels take 54.5 / 78.4; fp32 16 x 2048 x 512 39.5 / 66.8 us,
// 5.1 / 5.0 TB/s, where column blocks / drift take 45.5 / 70.9.  Off the lines, with narrow aligned accesses in the order
// of the segments before / now: fp32 2 x 125567 x 222 189 / 329 before, 158 / 265 now, bf16 131 / 233 and 97 / 167, 8 x 4096 x 175
// 20.0 / 35.3 and 13.0 / 24.3, fp32 30 x 1024 x 1500 137 / 203 and 126 / 206.  What is left to the rate of a plain stream is
// the width of the accesses (bf16 8 x 4096 x 1024 with two rows to a lane instead of four 48.4 / 75.6 us, with one in eight
// waves 52.9 / 82.8) and the one workgroup per CU, whose loads and stores do not overlap: a memory-only launch of this
// shape takes 79 us for fp32 32768 x 1024 forward where small workgroups take 63, but smaller segments pay more for the
// exchange than that brings (two workgroups of half the segment 84.6 us, four of a quarter 89 against 82.9).  Runs as
// long as the registers hold: descriptors per byte halve.
//
// A segment's map multiplies 128 or 256 coefficients, and the look-back composes several: the product can overflow where
// the recurrence does not (nothing put in yet, or small values that grow and shrink again).  Where what leaves a segment
// comes out non-finite, its row takes the value that leaves the segment before and goes through the waves' maps of U
// positions one after the other.  From the position on at which a row itself is infinite or NaN every segment of its block
// does, so the segments follow each other about 0.9 us apart: bf16 65536 x 512 with an infinity after an eighth of the
// positions takes 305 / 311 us (47 / 68 without; 69 / 95 in three launches either way), 588412 x 64 4.0 / 4.1 ms (90 / 117 us; 121 / 169),
// 4096 x 2048 29 / 36 us (14 / 21).
//
// A segment only waits for segments with smaller numbers, which are started first; every wait is bounded, and a
// lane whose wait runs out computes what enters its row from the row's own data.
//
// The reference has no strided kernel (linrec/impl/cuda/linrec_pipe.cu:35) and never splits a row.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "coldrift_kernel.hpp"  // ColDriftArgs, Held
#include "lookback_lanes.hpp"

namespace linrec {

constexpr int PHASE_LOOKBACK = 3;         // the kernel table's codes beside PHASE_REDUCE and PHASE_APPLY:
constexpr int PHASE_LOOKBACK_SHARED = 4;  // ... where a batch's rows are not a multiple of the rows of a lane

// VEC adjacent rows of one position by one access that need not be aligned to more than an element.
template <typename T, int VEC>
struct AnyPack {
  typedef T type __attribute__((ext_vector_type(VEC), aligned(sizeof(T))));
};
template <int VEC, bool STREAM, typename T>
__device__ __forceinline__ Held<T, VEC> ld_any(const T* p) {
  Held<T, VEC> h;
  if constexpr (VEC == 1) {
    const T q = STREAM ? stream_load(p) : *p;
    if constexpr (std::is_same_v<T, float>) h.q.v[0] = q;
    else h.q[0] = q;
  } else {
    using V = typename Pack<T, VEC>::type;
    using A = typename AnyPack<T, VEC>::type;
    const A* pa = reinterpret_cast<const A*>(p);
    const V q = STREAM && LINREC_NT_LOAD ? V(__builtin_nontemporal_load(pa)) : V(*pa);
    if constexpr (std::is_same_v<T, float>) {
#pragma unroll
      for (int e = 0; e < VEC; ++e) h.q.v[e] = q[e];
    } else {
      h.q = q;
    }
  }
  return h;
}
template <int VEC, typename T>
__device__ __forceinline__ void st_any(T* p, const Lanes<VEC>& r) {
  if constexpr (VEC == 1) {
    stream_store(T(r.v[0]), p);
  } else {
    using A = typename AnyPack<T, VEC>::type;
    A q;
#pragma unroll
    for (int e = 0; e < VEC; ++e) q[e] = T(r.v[e]);
#if LINREC_NT_STORE
    __builtin_nontemporal_store(q, reinterpret_cast<A*>(p));
#else
    *reinterpret_cast<A*>(p) = q;
#endif
  }
}

// The same for rows `first` (at least 1, the same for all lanes) and up only.
template <int VEC, typename T>
__device__ __forceinline__ void st_from(T* p, const Lanes<VEC>& r, unsigned first) {
  static_assert(VEC == 2 || VEC == 4, "rows left out: one, or one to three");
  if constexpr (VEC == 2) {
    st_any<1>(p + 1, Lanes<1>{{r.v[1]}});
  } else {
    if (first & 1u) st_any<1>(p + first, Lanes<1>{{first == 1u ? r.v[1] : r.v[3]}});
    if (first < 3u) st_any<2>(p + 2, Lanes<2>{{r.v[2], r.v[3]}});
  }
}

// SHARED: a batch's last lane shares rows with the lane before it and leaves them to that one (lookback_lanes.hpp).  A kernel
// of its own: with both kinds of stores in one, fp32 16 x 2048 x 512 backward, which has no such lane, took 64.6 us
// instead of 62.5.  Which rows a lane leaves out is the same for all lanes that do, so the branches are scalar (a mask per
// row and lane: fp32 23 x 25862 x 77 forward 160 us, where this takes 148; bf16 2 x 125567 x 222 107 / 184 and 98 / 165).
// (of args.chain: tasks = blocks of lanes, num_tiles = workgroups; of args.col: lanes_per_segment = lanes of a segment)
template <typename T, int VEC, int U, int NW, int MODE, bool DESC, bool SHARED = false>
__global__ __launch_bounds__(64 * NW) void collook_kernel(ColDriftArgs args) {
  static_assert(VEC <= NW, "a wave per row of a lane looks back");
  static_assert(!SHARED || VEC > 1, "a lane of one row shares none");
  const ColumnArgs& p = args.col;
  const TileArgs& ch = args.chain;
  constexpr int RPB = 64 * VEC;  // rows of a block
  constexpr int STEP = NW * U;   // positions of a segment
  constexpr bool NEED_Y = MODE == 1;
  // segments asked for in one round trip: one where the run itself takes most of the 128 registers there are
  constexpr int LOOK = U * VEC * int(sizeof(T)) / 4 * (NEED_Y ? 3 : 2) <= 48 ? 4 : 1;
  __shared__ float sh_a[NW][RPB];
  __shared__ float sh_b[NW][RPB];
  __shared__ float sh_in[RPB];  // the value entering the segment

  const T* in0 = static_cast<const T*>(p.in0);
  const T* coef = static_cast<const T*>(p.coef);
  const T* aux = static_cast<const T*>(p.aux);
  T* out0 = static_cast<T*>(p.out0);
  T* out1 = static_cast<T*>(p.out1);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int blocks = ch.tasks;
  // Segment and block of lanes.  Workgroups are dealt to the eight XCDs in turn, so with eight segments dealt out at a time
  // (ch.row_groups; 1 otherwise) one XCD runs the blocks of a segment.  A segment's workgroup still has a larger number
  // than the same block's of the segments before.
  int k, block;
  {
    const unsigned id = blockIdx.x, nb = unsigned(blocks), at_once = unsigned(ch.row_groups);
    const unsigned group = at_once * nb, g = id / group, r = id - g * group;
    if (at_once > 1u && (g + 1u) * group <= gridDim.x) {
      block = int(r / at_once);
      k = int(g * at_once + (r - unsigned(block) * at_once));
    } else {  // (also the last segments, less than eight of them)
      k = int(id / nb);
      block = int(id - unsigned(k) * nb);
    }
  }
  unsigned lane_no = unsigned(block) * 64u + unsigned(lane);  // (the planner keeps lanes and rows of a segment below 2^31)
  const bool active = lane_no < unsigned(p.lanes_per_segment);
  if (!active) lane_no = unsigned(p.lanes_per_segment) - 1u;  // lanes beyond the last row read the last rows again and store nothing
  const unsigned rows = unsigned(p.rows_per_batch < p.numseq ? p.rows_per_batch : p.numseq);
  const LaneRows held = lookback_lane_rows(lane_no, rows, unsigned(VEC), p.rows_per_batch < p.numseq);
  const unsigned own_from = lookback_own_from(rows, unsigned(VEC));  // (a scalar)
  // A wave's accesses are a scalar address plus 32 bits per lane (the planner sees to it that a block's rows span
  // less than 2^31 bytes): 64-bit addresses per lane took 30 to 40 registers, and with them a workgroup per CU.
  const long long base = (long long)held.batch * p.batch_stride + (long long)held.row * p.row_stride;
  const long long wbase = (long long)(uint32_t)__builtin_amdgcn_readfirstlane(int(base)) |
                          ((long long)__builtin_amdgcn_readfirstlane(int(base >> 32)) << 32);
  const uint32_t lane_bytes = uint32_t(base - wbase) * uint32_t(sizeof(T));
  const int L = p.seqlen;
  auto at = [&](auto* tensor, int l) __attribute__((always_inline)) {
    using P = decltype(tensor);
    using C = std::conditional_t<std::is_const_v<std::remove_pointer_t<P>>, const char*, char*>;
    return reinterpret_cast<P>(reinterpret_cast<C>(tensor + (wbase + (long long)l * p.elem_stride)) + lane_bytes);
  };
  const int ksteps = (L + STEP - 1) / STEP;
  const uint32_t seq = load_seq_through_caches(ch.ws);
  const uint32_t want = (seq << 2) | STATUS_AGGREGATE, done = (seq << 2) | STATUS_INCLUSIVE;
  // descriptors of segment s of this block: the first words of all rows, then the second words (a wave stores whole
  // lines of them), row e of lane i in place e * 64 + i
  auto desc_of = [&](int s) __attribute__((always_inline)) { return ch.desc + 2 * ((long long)s * blocks + block) * RPB; };

  struct Batch {
    Held<T, VEC> x[U], c[U], yn[NEED_Y ? U : 1];
  };
  const int n0 = k * STEP + wave * U;
  // positions a whole number of 128-byte lines apart: no line is wanted twice if the base starts on one too (what torch allocates
  // does; a view that does not reads its border lines twice, as it would without this)
  const bool on_lines = p.elem_stride * (long long)sizeof(T) % 128 == 0;
  // FULL: all positions of the segment exist and, for the backward, so does the last one's successor.  OWN: some of the
  // block's lanes store part of their rows only.
  auto segment = [&](auto full_tag, auto stream_tag, auto own_tag) __attribute__((always_inline)) {
    constexpr bool FULL = decltype(full_tag)::value, STREAM = decltype(stream_tag)::value, OWN = decltype(own_tag)::value;
    auto store = [&](T* to, const Lanes<VEC>& r) __attribute__((always_inline)) {
      if constexpr (OWN) {
        if (held.own != 0) st_from<VEC>(to, r, own_from);
        else st_any<VEC>(to, r);
      } else {
        st_any<VEC>(to, r);
      }
    };
    Batch bt;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int n = n0 + u;  // position in scan order
      const int l = DESC ? L - 1 - n : n;
      if (FULL || n < L) {
        bt.x[u] = ld_any<VEC, STREAM>(at(in0, l));
        bt.c[u] = ld_any<VEC, STREAM>(at(coef, l));
        if constexpr (NEED_Y) {
          const int ln = DESC ? l - 1 : l + 1;  // saved output one step further along this scan
          if (FULL || (ln >= 0 && ln < L)) {
            bt.yn[u] = ld_any<VEC, STREAM>(at(aux, ln));
          } else {
            bt.yn[u] = held_zero<T, VEC>();
          }
        }
      }
    }
    Lanes<VEC> ma, mb;
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      ma.v[e] = 1.0f;
      mb.v[e] = 0.0f;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int n = n0 + u;
      if (FULL || n < L) {
        const Lanes<VEC> x = widen(bt.x[u]), c = widen(bt.c[u]);
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          if constexpr (MODE == 0) {
            // the coefficient of the first position takes no part (linrec_ref.cuh:63)
            mb.v[e] = n == 0 ? x.v[e] : fmaf(mb.v[e], c.v[e], x.v[e]);
            ma.v[e] = n == 0 ? 0.0f : ma.v[e] * c.v[e];
          } else {
            mb.v[e] = (mb.v[e] + x.v[e]) * c.v[e];
            ma.v[e] *= c.v[e];
          }
        }
      }
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      sh_a[wave][e * 64 + lane] = ma.v[e];
      sh_b[wave][e * 64 + lane] = mb.v[e];
    }
    __syncthreads();
    if (wave < VEC) {
      const int i = wave * 64 + lane;
      float ta = sh_a[0][i], tb = sh_b[0][i];
#pragma unroll 4
      for (int w = 1; w < NW; ++w) {
        tb = fmaf(tb, sh_a[w][i], sh_b[w][i]);
        ta *= sh_a[w][i];
      }
      uint64_t* mine = desc_of(k) + i;
      float entering = 0.0f;
      if (k == 0) {
        if (ksteps > 1) st_desc(mine + RPB, pack_desc(done, tb));
      } else {
        if (k + 1 < ksteps) {
          st_desc(mine, pack_desc(want, ta));
          st_desc(mine + RPB, pack_desc(want, tb));
        }
        // (acc_a, acc_b): the segments j+1 .. k-1 composed.  The wave walks back as one, so the words' addresses
        // are scalar; a lane that has found its value ignores what else is read.
        float acc_a = 1.0f, acc_b = 0.0f;
        int j = k - 1, polls = 0;
        bool found = false;
        for (;;) {
          uint64_t w0[LOOK], w1[LOOK];
#pragma unroll
          for (int q = 0; q < LOOK; ++q) {
            const uint64_t* d = desc_of(j >= q ? j - q : 0);  // (beyond segment 0: asked for again, not used)
            w0[q] = ld_desc(d + i);
            w1[q] = ld_desc(d + RPB + i);
          }
          int moved = 0;
#pragma unroll
          for (int q = 0; q < LOOK; ++q) {
            const uint32_t f1 = uint32_t(w1[q] >> 32);
            const bool there = f1 == done || (f1 == want && uint32_t(w0[q] >> 32) == want);
            if (moved == q && __ballot(!found && !there) == 0) {
              const float b = __builtin_bit_cast(float, uint32_t(w1[q]));
              if (!found) {
                if (f1 == done) {  // (segment 0 always publishes what leaves it, so the walk never goes past it)
                  entering = fmaf(b, acc_a, acc_b);
                  found = true;
                } else {
                  acc_b = fmaf(b, acc_a, acc_b);
                  acc_a *= __builtin_bit_cast(float, uint32_t(w0[q]));
                }
              }
              ++moved;
            }
          }
          if (__ballot(!found) == 0) break;
          j -= moved;
          if (moved > 0) {
            polls = 0;
          } else {
            if (++polls >= ch.spin_limit) break;
            __builtin_amdgcn_s_sleep(1);
          }
        }
        float leaving = fmaf(entering, ta, tb);
        // (one test in the chain from segment to segment: what leaves cannot be finite if what enters is not)
        const bool astray = found && !__builtin_isfinite(leaving);
        if (__builtin_expect(__ballot(!found || astray) != 0, 0)) {
          bool have = found && !astray, waits = astray;
          const uint64_t* d = desc_of(k - 1) + RPB + i;
          for (polls = 0; __ballot(waits) != 0 && polls < ch.spin_limit; ++polls) {
            if (polls > 0) __builtin_amdgcn_s_sleep(1);
            const uint64_t w = ld_desc(d);
            if (waits && uint32_t(w >> 32) == done) {
              entering = __builtin_bit_cast(float, uint32_t(w));
              have = true;
              waits = false;
            }
          }
          if (__ballot(!have)) {
            if (lane == 0) __hip_atomic_fetch_add(&ch.ws->gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (!have) {
              // what enters the segment from the row's own data: the plain sequential walk
              const long long rb = base + (VEC > 1 ? wave : 0) * p.row_stride;
              float val = 0.0f;
              for (int n = 0; n < k * STEP; ++n) {
                const int l = DESC ? L - 1 - n : n;
                const long long off = rb + (long long)l * p.elem_stride;
                const float x = float(in0[off]), c = float(coef[off]);
                if constexpr (MODE == 0) val = n == 0 ? x : fmaf(val, c, x);
                else val = (val + x) * c;
              }
              entering = val;
            }
          }
          float val = entering;
#pragma unroll 1
          for (int w = 0; w < NW; ++w) val = fmaf(val, sh_a[w][i], sh_b[w][i]);
          if (!found || astray) leaving = val;
        }
        if (k + 1 < ksteps) st_desc(mine + RPB, pack_desc(done, leaving));
      }
      sh_in[i] = entering;
    }
    __syncthreads();
    Lanes<VEC> val;
#pragma unroll
    for (int e = 0; e < VEC; ++e) val.v[e] = sh_in[e * 64 + lane];
    for (int w = 0; w < wave; ++w) {
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        const float a = sh_a[w][e * 64 + lane], b = sh_b[w][e * 64 + lane];
        // before the first map of a row there is nothing: its b is taken as it is, so that 0 * inf can never arise
        val.v[e] = (k == 0 && w == 0) ? b : fmaf(val.v[e], a, b);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int n = n0 + u;
      const int l = DESC ? L - 1 - n : n;
      if (FULL || n < L) {
        const Lanes<VEC> x = widen(held_again(bt.x[u])), c = widen(held_again(bt.c[u]));
        if constexpr (MODE == 0) {
#pragma unroll
          for (int e = 0; e < VEC; ++e) val.v[e] = n == 0 ? x.v[e] : fmaf(val.v[e], c.v[e], x.v[e]);
          if (active) store(at(out0, l), val);
        } else {
          const Lanes<VEC> yn = widen(held_again(bt.yn[u]));
          Lanes<VEC> dx, dc;
#pragma unroll
          for (int e = 0; e < VEC; ++e) {
            dx.v[e] = val.v[e] + x.v[e];
            dc.v[e] = dx.v[e] * yn.v[e];
            val.v[e] = dx.v[e] * c.v[e];
          }
          if (active) {
            store(at(out0, l), dx);
            store(at(out1, l), dc);
          }
        }
      }
    }
  };
  const bool full = (k + 1) * (long long)STEP <= (NEED_Y ? L - 1 : L);
  if constexpr (SHARED) {
    // (the waves of a workgroup hold the same lanes, so they all take the same form)
    const bool own = __ballot(active && held.own != 0) != 0;
    if (full && !own) segment(std::true_type{}, std::false_type{}, std::false_type{});
    else if (full) segment(std::true_type{}, std::false_type{}, std::true_type{});
    else segment(std::false_type{}, std::false_type{}, std::true_type{});
  } else {
    if (full && on_lines) segment(std::true_type{}, std::true_type{}, std::false_type{});
    else if (full) segment(std::true_type{}, std::false_type{}, std::false_type{});
    else segment(std::false_type{}, std::false_type{}, std::false_type{});
  }

  // (the look-back waves are past the last barrier: no descriptor of this launch is touched by this workgroup again)
  if (threadIdx.x == 0) {
    const uint32_t leaf_count = signal_tile_done_begin(ch, blockIdx.x);
    signal_tile_done_end(ch, blockIdx.x, seq, leaf_count);
  }
}

}  // namespace linrec
