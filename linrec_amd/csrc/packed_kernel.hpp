// Packed tiles: dense rows (no gaps between them) of a slot and more, several whole rows to a workgroup.  One row to a workgroup leaves the lanes between the row's end and the tile's idle (a row of 333 floats
// takes 84 or 85 slots of 128), and rows that are not whole slots make every wave look at every slot.  Here a workgroup
// takes `tasks` consecutive rows as one array: slots are whole except the first and the last of the workgroup, all
// lanes but those of the last row's remainder have work, and the scan is cut at the row starts.
//
// A lane knows by arithmetic how many slots back its row started, so the cut needs no flag that travels with the maps (as
// the flat kernels have, whose rows may be shorter than a slot): a step of the wave's scan is skipped where it would reach
// beyond the row start.  Nothing of a row, non-finite values included, reaches the next one.  Rows never cross a
// workgroup, so there is no look-behind and no wait.
//
// Requirements (the planner's): unit element stride, row stride == row length, row length >= VEC (a slot holds at most
// one row start), the workgroup's rows and the phase of the first one within NW * S * 64 slots.
//
// What bounds it: memory.  fp32, 2^25 elements, forward / backward in us, in rows of 333: 65.4 / 118 (6.2 / 5.7 TB/s), where
// one row to a workgroup takes 77.5 / 124.5; 257: 65.0 / 116 against 86.9 / 149; 150: 65.0 / 115 against the flat kernels' 78.9 /
// 121; bf16 333: 34.9 / 63.7 against 46.4 / 81; 511: 35.1 / 64.2 against 53.8 / 86; 150: 34.7 / 62.9 against 45.2 / 72.8.  The first and
// last wave of a workgroup load whole slots and mask them once everything has arrived (slot by slot, each waiting for its
// loads: bf16 333 39.8 / 64.6).
//
// The reference has no counterpart: its kernels give a block to every row (linrec/impl/cuda/linrec_tile.cuh:11-95).
#pragma once
#include <hip/hip_runtime.h>

#include "tile_kernel.hpp"

namespace linrec {

// One step of the scan over the lanes of a row of slots.  back: slots from a lane's own to the one its row starts in;
// `reach`: slots the lane read from lies back, more than any row's where there is none.
template <int CTRL, int ROW_MASK, int S>
__device__ __forceinline__ void packed_scan_step(float (&a)[S], float (&b)[S], const int (&back)[S], int reach) {
#pragma unroll
  for (int j = 0; j < S; ++j) {
    const float pa = dpp_move<CTRL, ROW_MASK>(1.0f, a[j]);
    const float pb = dpp_move<CTRL, ROW_MASK>(0.0f, b[j]);
    b[j] = back[j] >= reach ? fmaf(pb, a[j], b[j]) : b[j];
    a[j] = pa * a[j];  // (where a row starts in between, nobody looks at it again)
  }
}

template <typename T, int NW, int S, int VEC, int MODE, bool DESC>
__global__ __launch_bounds__(64 * NW) void packed_kernel(TileArgs p) {
  constexpr int WAVE_SLOTS = S * 64;
  constexpr int LOG_VEC = VEC == 4 ? 2 : 3;
  static_assert(VEC == 1 << LOG_VEC, "whole slots");
  __shared__ float sh_a[NW], sh_b[NW];
  __shared__ int sh_cut[NW];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int L = p.seqlen;
  const long long row = (long long)blockIdx.x * p.tasks;
  const int rows = p.numseq - row < p.tasks ? int(p.numseq - row) : p.tasks;
  const long long row_off = row * L;
  // (the workgroup's rows as one row; positions below are counted in scan order)
  const RowView rv = make_row_view<VEC>(p.base_mis, row_off, rows * L);
  const RowPtrs<T> q = make_row_ptrs<T, MODE>(p.in0, p.coef, p.aux, p.out0, p.out1, row_off, rv.lo);
  const int u_wave = wave * WAVE_SLOTS;
  const bool interior = slots_interior<VEC, DESC>(u_wave, WAVE_SLOTS, rv);

  TileData<S, VEC, MODE> d;
  if (interior) tile_load<S, VEC, MODE, DESC, true>(d, q, rv, u_wave, lane, false);
  else tile_load_edge<S, VEC, MODE, DESC>(d, q, rv, u_wave, lane);

  // Row position of a slot's first element, taken modulo L; elements before the first row and after the last count on.
  int cut_at[S];   // the slot's element a row starts with (VEC and more: none)
  int back[S];     // slots back to the one the row of the slot's last element starts in
  int ex_back[S];  // the same for the slot before, from there
  {
    const int before = DESC ? rv.nslots * VEC - rv.hi : rv.lo;  // elements of the first slot that lie before the first row
    int r = int(unsigned((u_wave + lane) * VEC - before + L) % unsigned(L));
    const int step = int(unsigned(64 * VEC) % unsigned(L));
#pragma unroll
    for (int j = 0; j < S; ++j) {
      cut_at[j] = r == 0 ? 0 : L - r;
      const int last = r + VEC - 1;
      back[j] = (last >= L ? last - L : last) >> LOG_VEC;
      ex_back[j] = (r == 0 ? L - 1 : r - 1) >> LOG_VEC;
      r += step;
      if (r >= L) r -= L;
    }
  }

  if (!interior) tile_mask<S, VEC, MODE, DESC>(d, rv, u_wave, lane);

  // lane level (the two forms of tile_scan): a slot's map, of which only b counts once a row starts in the slot
  float agg_a[S], agg_b[S];
#pragma unroll
  for (int j = 0; j < S; ++j) {
    float a = MODE == MODE_FWD ? d.cs[j][0] : 1.0f, b = d.xs[j][0];
#pragma unroll
    for (int i = 1; i < VEC; ++i) {
      const float c = MODE == MODE_FWD ? d.cs[j][i] : d.cs[j][i - 1];
      a *= c;
      b = cut_at[j] == i ? d.xs[j][i] : fmaf(b, c, d.xs[j][i]);
    }
    agg_a[j] = MODE == MODE_FWD ? a : a * d.cs[j][VEC - 1];
    agg_b[j] = MODE == MODE_FWD ? b : b * d.cs[j][VEC - 1];
  }

  // wave level: the lanes of every row of slots, then the rows of slots in scan order
  const int in_row = lane & 15;
  packed_scan_step<DPP_ROW_SHR1, 0xf, S>(agg_a, agg_b, back, in_row >= 1 ? 1 : 1 << 30);
  packed_scan_step<DPP_ROW_SHR2, 0xf, S>(agg_a, agg_b, back, in_row >= 2 ? 2 : 1 << 30);
  packed_scan_step<DPP_ROW_SHR4, 0xf, S>(agg_a, agg_b, back, in_row >= 4 ? 4 : 1 << 30);
  packed_scan_step<DPP_ROW_SHR8, 0xf, S>(agg_a, agg_b, back, in_row >= 8 ? 8 : 1 << 30);
  packed_scan_step<DPP_ROW_BCAST15, 0xa, S>(agg_a, agg_b, back, lane & 16 ? in_row + 1 : 1 << 30);
  packed_scan_step<DPP_ROW_BCAST31, 0xc, S>(agg_a, agg_b, back, lane & 32 ? lane - 31 : 1 << 30);
  float ex_a[S], ex_b[S];  // what enters the slot: ex_a * E + ex_b, E what enters the wave; ex_b where a row starts in between
  bool reached[S];         // ... no row starts in between
  float run_a = 1.0f, run_b = 0.0f;
  bool run_cut = false;
#pragma unroll
  for (int j = 0; j < S; ++j) {
    const float lane_a = shift_up_one_lane(agg_a[j], 1.0f), lane_b = shift_up_one_lane(agg_b[j], 0.0f);
    const bool cut = lane > 0 && ex_back[j] <= lane - 1;
    const float total_a = read_lane(agg_a[j], 63), total_b = read_lane(agg_b[j], 63);
    const bool total_cut = __builtin_amdgcn_readlane(back[j], 63) <= 63;
    if (j == 0) {
      ex_a[j] = lane_a;
      ex_b[j] = lane_b;
      run_a = total_a;
      run_b = total_b;
    } else {
      ex_a[j] = run_a * lane_a;
      ex_b[j] = cut ? lane_b : fmaf(run_b, lane_a, lane_b);
      run_a *= total_a;
      run_b = total_cut ? total_b : fmaf(run_b, total_a, total_b);
    }
    reached[j] = !cut && !run_cut;
    run_cut = run_cut || total_cut;
  }

  // the waves: every wave folds the maps in front of it, from the last row start on
  if (lane == 0) {
    sh_a[wave] = run_a;
    sh_b[wave] = run_b;
    sh_cut[wave] = run_cut;
  }
  __syncthreads();
  float entry = 0.0f;
  {
    const int w = lane < NW ? lane : NW - 1;
    const float wa = sh_a[w], wb = sh_b[w];
    const int wc = sh_cut[w];
#pragma unroll
    for (int i = 0; i + 1 < NW; ++i) {
      if (i >= wave) break;
      const float b = read_lane(wb, i);
      // (wave 0 starts with a row)
      entry = i == 0 || __builtin_amdgcn_readlane(wc, i) ? b : fmaf(entry, read_lane(wa, i), b);
    }
  }

  float r0[S][VEC], r1[MODE == MODE_BWD ? S : 1][VEC];
#pragma unroll
  for (int j = 0; j < S; ++j) {
    const float enter = reached[j] && wave > 0 ? fmaf(entry, ex_a[j], ex_b[j]) : ex_b[j];
    // the recurrence over the slot's elements from what enters it (fewer operations than the elements' maps, which
    // would each have to be cut as well)
    r0[j][0] = cut_at[j] == 0 ? d.xs[j][0] : MODE == MODE_FWD ? fmaf(enter, d.cs[j][0], d.xs[j][0]) : enter + d.xs[j][0];
#pragma unroll
    for (int i = 1; i < VEC; ++i) {
      const float c = MODE == MODE_FWD ? d.cs[j][i] : d.cs[j][i - 1];
      r0[j][i] = cut_at[j] == i ? d.xs[j][i] : fmaf(r0[j][i - 1], c, d.xs[j][i]);
    }
    if constexpr (MODE == MODE_BWD) {
      // the saved output one step further along the scan (see tile_apply_store), zero where the row ends
      const float for_lane63 = (j + 1 < S) ? read_lane(d.ys[(j + 1) % S][0], 0) : d.y_edge;
      const float y_next_slot = shift_down_one_lane(d.ys[j][0], for_lane63);
      // (a row starts with the next slot: VEC elements on from this one's first, or, where one starts here, L)
      const bool next_starts = cut_at[j] == VEC || (cut_at[j] < VEC && cut_at[j] + L == VEC);
#pragma unroll
      for (int i = 0; i < VEC; ++i) {
        const bool ends = i + 1 < VEC ? cut_at[j] == i + 1 : next_starts;
        r1[j][i] = r0[j][i] * (ends ? 0.0f : i + 1 < VEC ? d.ys[j][(i + 1) % VEC] : y_next_slot);
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  if (interior) {
    const long long s_low = DESC ? (long long)rv.nslots - u_wave - WAVE_SLOTS : (long long)u_wave;
    const unsigned lane_idx = DESC ? 63u - unsigned(lane) : unsigned(lane);
#pragma unroll
    for (int j = 0; j < S; ++j) {
      store_slot_full<VEC, DESC>(q.out0 + s_low * VEC, (DESC ? unsigned(S - 1 - j) : unsigned(j)) * 64u + lane_idx, r0[j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (MODE == MODE_BWD) {
#pragma unroll
      for (int j = 0; j < S; ++j) {
        store_slot_full<VEC, DESC>(q.out1 + s_low * VEC, (DESC ? unsigned(S - 1 - j) : unsigned(j)) * 64u + lane_idx, r1[j]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < S; ++j) {
      store_slot<VEC, DESC>(q.out0, u_wave + j * 64 + lane, rv, r0[j]);
      if constexpr (MODE == MODE_BWD) store_slot<VEC, DESC>(q.out1, u_wave + j * 64 + lane, rv, r1[j]);
    }
  }
}

}  // namespace linrec
