"""Byte offsets of the stage kernel's geometry planes on the largest grid that
wtg_grid_create takes (level 12, six planes of areas): base and 32-bit offset
together are the plane's place, and base plus cell stays below 4 GiB.  Runs on
the CPU: the header has no device code.
"""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, os.pardir, "wavetrisk_hydrostatic_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "grid.h"
#include "planes.h"
int main() {
  for (int level = 4; level <= 12; ++level) {
    const int64_t S = (1 << level) + 2 * wtg::HALO, nc = wtg::NLOZ * S * S;
    for (int p = 0; p < 6; ++p) {
      const wtg::PlaneAt at = wtg::plane_at(p, nc);
      const unsigned long long last = (unsigned long long)at.byte + 8ull * (nc - 1) + 8;
      if (at.first * 8 + (int64_t)at.byte != p * nc * 8 || last > 0xffffffffull) {
        std::printf("level %d plane %d\n", level, p);
        return 1;
      }
    }
  }
  return 0;
}
"""


def test_planes_of_the_largest_grid(tmp_path):
    src, exe = tmp_path / "planes.cpp", tmp_path / "planes"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
