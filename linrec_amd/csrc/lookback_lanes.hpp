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
// 73.2, in the geometric means of 1100 shapes 0.92 / 0.97 in fp32 and 0.94 / 0.93 in 16-bit storage, but 3 x 1813 x 1464 (eight
// segments) 33.7 against 28.0.  On lines only the fp32 backward of many segments in a few blocks gains (32768 x 1024 122.8 against
// 129.7, 0.99 in the mean of such shapes); the others lose the look-back's own locality, a block's segments being on one XCD when
// its number alone decides that: 16 x 2048 x 512 backward 73.7 against 70.2, fp16 2 x 3859 x 4160 71.1 against 62.0, up to one and
// a half rounds of workgroups 1.05 to 1.12 in the means; forward 1.02.
constexpr long long lookback_segments_at_once(bool on_lines, bool is_bwd, bool half, long long blocks, long long segments) {
  const bool eight = on_lines ? is_bwd && !half && blocks >= 4 && segments >= 100 : blocks >= 2 && segments >= 16;
  return eight ? 8 : 1;
}

}  // namespace linrec
