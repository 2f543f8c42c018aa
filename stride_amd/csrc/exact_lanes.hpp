// Which batch lanes a matrix tile of the exact path reads (plain C++: the tests build
// it for the host).
#pragma once

namespace stride_tc {

// First of the L batch lanes that a thread of the tile at `lane` loads: its own, or the
// last whole L of the live lane groups where the tile reaches past them. Their end bounds
// it, not the row stride: x may be a run of lanes inside a wider buffer, whose last
// column ends with the last live lane.
constexpr int exact_tile_lane(int lane, int lane_groups, int L) {
  return lane < 4 * lane_groups - L ? lane : 4 * lane_groups - L;
}

}  // namespace stride_tc
