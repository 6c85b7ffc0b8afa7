// Which rows a lane of the look-back segments (collook_kernel.hpp) reads and which of them it stores: plain C++, shared by
// the kernels and whoever wants to check it on a host.
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

}  // namespace linrec
