"""The LDS layout of the filter kernel, checked on the host for every group size and
number of rays: the kernel reads and writes a wave's values, staged triangles and exp terms
as float4, so each wave's part and each area read that way starts at a multiple of 16 bytes,
the areas do not overlap, and a block fits the 64 KB that a launch may ask for."""
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "renderer2_amd" / "csrc"

PROGRAM = r"""
#include <cstdio>
#include "r2_filter_lds.hpp"
using namespace r2::filter_lds;
int main() {
  for (int n = 1; n <= 1000; ++n) {
    const int cap = ts_cap(n);
    if (cap < n || cap % 4) return std::printf("cap %d of %d rays\n", cap, n), 1;
    for (int g = 1; g <= max_group(cap); ++g) {
      const int wave = wave_floats(g, cap);
      const int terms = g * cap;  // the exp terms of the density pass share the values' space
      if (wave % 4) return std::printf("%d rays, %d voxels: a wave's part is %d floats\n", n, g, wave), 1;
      if ((kVals * kRow) % 4 || kRow % 4) return std::printf("rows\n"), 1;
      if (terms > kVals * kRow) return std::printf("%d rays, %d voxels: %d exp terms\n", n, g, terms), 1;
      if (wave < kVals * kRow + g * cap + g * kSumRow) return std::printf("%d rays, %d voxels: overlap\n", n, g), 1;
      if (4 * kWaves * wave > 65536) return std::printf("%d rays, %d voxels: %d bytes\n", n, g, 4 * kWaves * wave), 1;
    }
  }
  return 0;
}
"""


def test_filter_lds_layout(tmp_path):
    src = tmp_path / "lds.cpp"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", str(CSRC), str(src), "-o", str(tmp_path / "lds")], check=True)
    r = subprocess.run([str(tmp_path / "lds")], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
