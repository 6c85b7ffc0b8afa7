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

// Segments dealt out at a time (collook_kernel.hpp): eight where that is as good or better, whole groups of which there is
// at least one.  Forward / backward in us, eight against one: off the 128-byte lines fp32 8326 x 4022 (time x channels) 91.6 /
// 140.7 against 98.0 / 150.2, 2 x 125567 x 222 165.9 / 244 against 172.4 / 251, bf16 8 x 4096 x 700 40.6 / 69.0 against 42.9 /
// 73.2, in the geometric means of 1100 shapes 0.92 / 0.97 in fp32 and 0.94 / 0.93 in 16-bit storage; with eight to fifteen segments
// the backward too (30 x 1024 x 1500 205 against 216, 0.97 and 0.90 in the means), not all forwards (3 x 1813 x 1464 33.7 against
// 28.0).  On lines only the fp32 backward of a multiple of four blocks gains, whose segments then end with a group of eight workgroups
// or in its middle: after a forward, on new inputs each time, 8 x 4096 x 512 64.4 against 68.8, 8 x 2048 x 1024 65.0 against 67.0, 16 x
// 2048 x 512 68.7 against 68.5, in the means of 180 shapes 0.98 of multiples of eight, 1.00 of the other multiples of four, 1.01 to
// 1.03 of other numbers (4 x 3859 x 1088 66.3 against 64.0).  The others lose the look-back's own locality, a block's segments being
// on one or two XCDs otherwise: 16-bit backwards 8 x 4096 x 1024 70.9 against 66.0, 2 x 3859 x 4160 69.7 against 61.5, up to one and a
// half rounds of workgroups 1.03 in the mean; forwards 1.02.
constexpr long long lookback_segments_at_once(bool on_lines, bool is_bwd, bool half, long long blocks, long long segments) {
  const bool eight = on_lines ? is_bwd && !half && blocks % 4 == 0 && segments >= 16 : blocks >= 2 && segments >= (is_bwd ? 8 : 16);
  return eight ? 8 : 1;
}

}  // namespace linrec
