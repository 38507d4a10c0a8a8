"""Registers of the stage kernels in the built library: the FP32-bulk forms run
at three waves a SIMD (one-layer form: five) and the FP64 forms at two, so a few
more registers or spilled values show as time.  Read from the kernels' metadata
in the library's code objects; runs on the CPU.
"""
import os
import re
import struct
import subprocess

import pytest

from wavetrisk_hydrostatic_amd import build

READOBJ = "/opt/rocm/llvm/bin/llvm-readobj"


def _code_objects(path):
    """gfx950 code objects of the library's offload bundles"""
    blob = open(path, "rb").read()
    pos = blob.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while pos >= 0:
        at = pos + 32
        for _ in range(min(struct.unpack_from("<Q", blob, pos + 24)[0], 16)):
            off, size, n = struct.unpack_from("<QQQ", blob, at)
            name = blob[at + 24:at + 24 + n]
            at += 24 + n
            if name.endswith(b"gfx950") and size:
                yield blob[pos + off:pos + off + size]
        pos = blob.find(b"__CLANG_OFFLOAD_BUNDLE__", pos + 24)


@pytest.fixture(scope="module")
def registers(tmp_path_factory):
    if not (os.path.exists(build.LIB) and os.path.exists(READOBJ)):
        pytest.skip("needs the built library and llvm-readobj")
    out, path = {}, tmp_path_factory.mktemp("co") / "co.o"
    for co in _code_objects(build.LIB):
        path.write_bytes(co)
        notes = subprocess.run([READOBJ, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for m in re.finditer(r"\.name: +_Z\S*?\d((?:trisk|vd|remap|fs)_\w+_kernel)(I\w*E)?\S*\n.*?\.vgpr_count: +(\d+)"
                             r"\s+\.vgpr_spill_count: (\d+)", notes, re.S):
            args = re.findall(r"Lb([01])|L[ij](\d+)|([df])(?=L|E)", m[2] or "")
            out[m[1], tuple("".join(a) for a in args)] = int(m[3]), int(m[4])
    return out


# the counts of the code whose times are noted beside the kernels:
# (HasD, output, edge tasks) of the layer-pair forms, (HasD, output) of the one-layer form
@pytest.mark.parametrize("kernel,args,vgprs,spills", [
    ("trisk_stage_mixed_kernel", ("0", "f", "0"), 115, 0), ("trisk_stage_mixed_kernel", ("1", "f", "0"), 124, 0),
    ("trisk_stage_mixed_kernel", ("1", "d", "0"), 143, 0), ("trisk_stage_mixed_kernel", ("0", "f", "1"), 126, 0),
    ("trisk_stage_mixed_kernel", ("1", "f", "1"), 133, 0), ("trisk_stage_mixed_kernel", ("1", "d", "1"), 155, 0),
    ("trisk_stage_mixed1_kernel", ("0", "f"), 96, 0), ("trisk_stage_mixed1_kernel", ("1", "f"), 96, 12),
    ("trisk_stage_mixed1_kernel", ("1", "d"), 96, 43),
    # (KEEP, SPLIT, DIFF)
    ("trisk_stage_tile_kernel", ("0", "0", "0"), 256, 0), ("trisk_stage_tile_kernel", ("0", "1", "0"), 256, 0),
    ("trisk_stage_tile_kernel", ("1", "0", "0"), 256, 0)])
def test_stage_kernels(registers, kernel, args, vgprs, spills):
    assert (kernel, args) in registers, sorted(registers)
    got = registers[kernel, args]
    assert got[0] <= vgprs and got[1] <= spills, got
