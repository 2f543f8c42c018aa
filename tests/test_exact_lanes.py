"""The batch lanes that a matrix tile of the exact path reads (CPU: the rule of
stride_amd/csrc/exact_lanes.hpp built for the host). x may be a run of lane groups
inside a wider dim-major buffer; a tile that reaches past its last live lane group
must not read past it, which in the buffer's last column would leave the buffer."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stride_amd", "csrc")

PROBE = r"""
#include <cstdio>
#include "exact_lanes.hpp"
int by_stride(int lane, int, int L) { return lane < 96 - L ? lane : 96 - L; }  // a run of a 96-lane buffer
template <class F>
int outside(F first) {
  int bad = 0;
  for (int lane_groups = 1; lane_groups <= 20; ++lane_groups)
    for (int L = 1; L <= 4; L *= 2)
      for (int tile = 0; tile * 16 * L < 4 * lane_groups; ++tile)
        for (int i = 0; i < 16; ++i) {
          const int lane = tile * 16 * L + L * i, at = first(lane, lane_groups, L);
          const bool live = lane + L <= 4 * lane_groups;
          bad += at < 0 || at % L != 0 || at + L > 4 * lane_groups || (live && at != lane);
        }
  return bad;
}
int main() { printf("%d %d\n", outside(stride_tc::exact_tile_lane), outside(by_stride)); }
"""


def test_tile_lanes_stay_inside_the_live_groups(tmp_path):
    src, exe = tmp_path / "probe.cpp", tmp_path / "probe"
    src.write_text(PROBE)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    bad, by_stride = map(int, subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split())
    assert by_stride > 0  # bounded by the row stride, tiles read dead lanes
    assert bad == 0


def test_the_matrix_kernel_uses_the_rule():
    text = open(os.path.join(CSRC, "exact.hip")).read()
    body = text[text.index("void k_exact_gemm_m("):text.index("Batch B[2];")]
    assert "exact_tile_lane(lg0 * 4 + L * i, p.l.lane_groups, L)" in body and "stride - L" not in body
