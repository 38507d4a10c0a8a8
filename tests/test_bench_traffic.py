"""The benchmark's HBM traffic is that of the kernel it times: the counter
summary of another kernel is not taken, and the committed ones are of kernels
in the library.  Runs on the CPU.
"""
import os

import bench

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_traffic_of_the_timed_kernels():
    lib = open(os.path.join(ROOT, "wavetrisk_hydrostatic_amd", "csrc", "trisk.hip")).read()
    for summary, kernel in (("trisk_stage", "trisk_stage_tile_kernel"), ("trisk_stage_mixed", "trisk_stage_mixed_kernel")):
        assert f"{kernel}(" in lib
        assert bench.measured_traffic(8, 30, summary, kernel) > 0
        assert bench.measured_traffic(8, 30, summary, "another_kernel") is None
        assert bench.measured_traffic(3, 30, summary, kernel) is None
