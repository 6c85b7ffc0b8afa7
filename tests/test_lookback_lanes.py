"""Which rows the lanes of the look-back segments store: every row of every batch has exactly one lane that does, also
where a batch's rows are not a multiple of the rows of a lane.  The kernel's own header, compiled for the host."""
import ctypes
import os
import subprocess

import pytest
import torch

from linrec_amd import _native as nat

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "linrec_amd", "csrc")
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "lookback_lanes.hpp"
int main(int argc, char** argv) {
  const unsigned batches = std::atoi(argv[1]), rows = std::atoi(argv[2]), vec = std::atoi(argv[3]);
  const unsigned lanes = (rows + vec - 1) / vec;
  std::vector<int> stored(batches * rows, 0), read(batches * rows, 0);
  for (unsigned i = 0; i < batches * lanes; ++i) {
    const linrec::LaneRows r = linrec::lookback_lane_rows(i, rows, vec, batches > 1);
    if (r.batch >= batches || r.row + vec > rows || r.own >= vec) return 1;
    if (r.own != 0 && r.own != linrec::lookback_own_from(rows, vec)) return 1;
    for (unsigned e = 0; e < vec; ++e) {
      ++read[r.batch * rows + r.row + e];
      if (e >= r.own) ++stored[r.batch * rows + r.row + e];
    }
  }
  for (unsigned i = 0; i < batches * rows; ++i)
    if (stored[i] != 1 || read[i] < 1) { std::printf("row %u: stored by %d lanes, read by %d\n", i, stored[i], read[i]); return 2; }
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    where = tmp_path_factory.mktemp("lanes")
    (where / "lanes.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(where / "lanes.cpp"), "-o", str(where / "lanes")], check=True)
    return str(where / "lanes")


@pytest.mark.parametrize("vec", [1, 2, 4])
def test_every_row_is_stored_by_one_lane(program, vec):
    for batches in (1, 2, 3, 7):
        for rows in sorted({vec, vec + 1, 2 * vec - 1, 2 * vec, 63, 64, 66, 129, 203, 257, 64 * vec, 64 * vec + 1, 64 * vec + vec - 1}):
            if rows >= vec:
                got = subprocess.run([program, str(batches), str(rows), str(vec)], stdout=subprocess.PIPE, text=True)
                assert got.returncode == 0, (batches, rows, vec, got.returncode, got.stdout)


AT_ONCE = r"""
#include "lookback_lanes.hpp"
using linrec::lookback_segments_at_once;
constexpr bool LINES = true, BWD = true, HALF = true;
static_assert(lookback_segments_at_once(LINES, BWD, HALF, 33, 16) == 1 && lookback_segments_at_once(LINES, BWD, HALF, 4, 1000) == 1,
              "16-bit backwards on lines take one segment after the other");
static_assert(lookback_segments_at_once(LINES, BWD, !HALF, 17, 100) == 1 && lookback_segments_at_once(LINES, BWD, !HALF, 32, 15) == 1,
              "fp32 backwards on lines too, but of a multiple of four blocks");
static_assert(lookback_segments_at_once(LINES, BWD, !HALF, 4, 16) == 8 && lookback_segments_at_once(LINES, BWD, !HALF, 2, 100) == 1);
static_assert(lookback_segments_at_once(LINES, !BWD, !HALF, 33, 256) == 1 && lookback_segments_at_once(LINES, !BWD, HALF, 33, 256) == 1);
static_assert(lookback_segments_at_once(!LINES, BWD, HALF, 33, 16) == 8 && lookback_segments_at_once(!LINES, !BWD, HALF, 2, 16) == 8);
static_assert(lookback_segments_at_once(!LINES, BWD, !HALF, 176, 8) == 8 && lookback_segments_at_once(!LINES, BWD, HALF, 20, 7) == 1);
static_assert(lookback_segments_at_once(!LINES, !BWD, HALF, 33, 15) == 1 && lookback_segments_at_once(!LINES, BWD, HALF, 1, 100) == 1);
"""


def test_segments_dealt_out_at_a_time(tmp_path):
    (tmp_path / "at_once.cpp").write_text(AT_ONCE)
    subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-I", CSRC, str(tmp_path / "at_once.cpp")], check=True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_lanes_that_share_rows_take_the_kernels_that_know(dtype):
    old = nat.set_compute_units(256)
    try:
        seen = set()
        for batch, time, channels in [(8, 4096, 1024), (8, 4096, 1025), (8, 4096, 1026), (8, 4096, 1027), (23, 5000, 77), (4, 4096, 700),
                                      (1, 11944, 2809), (1, 8326, 4022), (2, 40000, 222), (8, 4096, 175), (5, 777, 1001),
                                      (7, 2048, 192)]:
            for is_bwd in (0, 1):
                p = nat.Plan()
                if batch > 1:
                    rc = nat.lib().linrec_plan_batched(nat.DTYPES[dtype], None, batch, channels, time, time * channels, 1, channels, 0,
                                                       is_bwd, None, ctypes.byref(p))
                else:
                    rc = nat.lib().linrec_plan(nat.DTYPES[dtype], None, channels, time, 1, channels, 0, is_bwd, None, ctypes.byref(p))
                name = nat.kernel_table()[p.kernel_id]
                if rc == 0 and "segment_lookback" in name:
                    assert ("shared" in name) == (channels % p.vec != 0), (batch, time, channels, is_bwd, name)
                    seen.add((p.vec, "shared" in name))
        assert {(2, True), (2, False), (4, True), (4, False)} <= seen, seen
    finally:
        nat.set_compute_units(old)
