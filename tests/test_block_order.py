"""The order of a compute list's blocks over the XCDs (csrc/xcd.h): every block
is taken once, whatever the launch's size, and lists of one field keep their
order up to J7, where the rows per XCD cost time.  Compiled for the CPU with
the launch's indices as plain variables.
"""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, os.pardir, "wavetrisk_hydrostatic_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <vector>
#define __device__
#define __forceinline__ inline
struct { unsigned x; } blockIdx, gridDim;
#include "xcd.h"
int taken_once(unsigned n, unsigned (*at)(unsigned), unsigned per) {
  std::vector<int> seen(n, 0);
  gridDim.x = n;
  for (blockIdx.x = 0; blockIdx.x < n; ++blockIdx.x) {
    const unsigned b = at(per);
    if (b >= n || seen[b]++) return 0;
  }
  return 1;
}
int main() {
  for (unsigned n = 1; n < 5000; n = n < 70 ? n + 1 : n + 61)
    for (int planes : {1, 2, 5, 60})
      if (!taken_once(n, list_block, xcd_rows(n, planes)) || !taken_once(n, [](unsigned) { return xcd_block(); }, 0)) {
        std::printf("%u blocks, %d planes\n", n, planes);
        return 1;
      }
  // blocks of 256 entries of the lists of J6, J7, J8
  const unsigned j6 = 165, j7 = 660, j8 = 2600;
  return xcd_rows(j6, 64) == 0 && xcd_rows(j7, 1) == 0 && xcd_rows(j7, 3) == 82 && xcd_rows(j8, 1) == 325 ? 0 : 2;
}
"""


def test_every_block_once(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text("")
    src, exe = tmp_path / "order.cpp", tmp_path / "order"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", str(tmp_path), "-I", CSRC, "-o", str(exe), str(src)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, (run.returncode, run.stdout)
