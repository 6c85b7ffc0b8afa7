// Which rows a lane of the look-back segments (collook_kernel.hpp) reads and which of them it stores, and how many segments
// are dealt out at a time: plain C++, shared by the kernels, the planner and whoever wants to check it on a host.
#pragma once

namespace linrec {

// Lanes are numbered batch by batch, `vec` adjacent rows each (`rows` of a batch, no fewer than `vec`).  Where those are not
// a multiple of `vec` a batch's last lane starts early: it reads, and computes, rows of the lane before it as well, but
// every row is stored by one lane only.  The two need not see the same descriptors, nor run in the same workgroup, so
// what they compute can differ in the last bit, and two stores would leave to chance which of them stays.
struct LaneRows {
  unsigned batch;  // of the lane
  unsigned row;    // its first row there
  unsigned own;    // the first of its rows that it stores, counted from `row`
};
// LaneRows::own of every lane that shares rows.
constexpr unsigned lookback_own_from(unsigned rows, unsigned vec) { return vec - rows % vec; }
constexpr LaneRows lookback_lane_rows(unsigned lane_no, unsigned rows, unsigned vec, bool batched) {
  const unsigned lanes = (rows + vec - 1u) / vec;
  const unsigned batch = batched ? lane_no / lanes : 0u;
  const unsigned row = (lane_no - batch * lanes) * vec;
  const unsigned last = rows - vec;
  return row > last ? LaneRows{batch, last, row - last} : LaneRows{batch, row, 0u};
}

// Segments dealt out at a time (collook_kernel.hpp): eight where that is as good or better, whole groups of which there are
// at least two.  Forward / backward in us, eight against one: off the 128-byte lines fp32 8326 x 4022 (time x channels) 91.6 /
// 140.7 against 98.0 / 150.2, 2 x 125567 x 222 165.9 / 244 against 172.4 / 251, bf16 8 x 4096 x 700 40.6 / 69.0 against 42.9 /
// 73.2, but 3 x 1813 x 1464 (eight segments) 33.7 against 28.0; on them fp32 32768 x 1024 79.9 / 122.8 against 82.9 / 129.7,
// 16 x 2048 x 512 43.6 / 66.8 against 39.5 / 69.5, bf16 32768 x 1024 47.6 / 67.6 against 44.4 / 68.8, of two blocks fp32
// 16384 x 512 24.2 / 33.9 against 22.3 / 32.6; the 16-bit backward of sixteen blocks and more 1.09 in the geometric mean up to one
// and a half rounds of workgroups and 1.02 beyond (fp16 2 x 3859 x 4160 71.1 against 62.0).
constexpr long long lookback_segments_at_once(bool on_lines, bool is_bwd, bool half, long long blocks, long long segments) {
  const bool eight = on_lines ? is_bwd && blocks >= 4 && !(half && blocks >= 16) : blocks >= 2;
  return segments >= 16 && eight ? 8 : 1;
}

}  // namespace linrec
