"""Registers that the pair kernels' grids and the kernels beside them count on, read
from the device code the build produces (AMD assembly of this repository's own
source, no GPU), and the kernel that a batch's grid is made for.

A SIMD holds 512 VGPRs per lane, given out in eights; a pair kernel's block has one
wavefront on each of a CU's four SIMDs.
"""
import os
import re
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "nexusmd_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is absent")


def _vgprs(name, tmp):
    out = os.path.join(str(tmp), name + ".s")
    cmd = [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", "-I" + os.path.join(REPO, "include"), "-I" + CSRC, "--cuda-device-only", "-S", "-o", out,
           os.path.join(CSRC, name + ".hip")]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    got = {}
    for block in open(out).read().split("  - .agpr_count:")[1:]:
        assert int(re.search(r"\.vgpr_spill_count:\s+(\d+)", block).group(1)) == 0
        got[re.search(r"\.name:\s+(\S+)", block).group(1)] = (int(re.search(r"\.vgpr_count:\s+(\d+)", block).group(1)) + 7) // 8 * 8
    return lambda *parts: next(v for k, v in got.items() if all(p in k for p in parts))


def test_fp64_pair_grid_is_resident(tmp_path):
    """The kernel without library functions leaves room for three blocks a CU (batches
    up to 50,000 atoms) and, at two, for two 96-register wavefronts beside them (the
    gather, the plane passes); the one with them holds two."""
    v = _vgprs("nonbonded", tmp_path)
    series, chooses = v("pair_kernel_fp64", "ILb0ELb1E"), v("pair_kernel_fp64", "ILb0ELb0E")
    print("FP64 pair kernel %d VGPRs, with library functions %d" % (series, chooses))
    assert 3 * series <= 512 and 2 * series + 2 * 96 <= 512
    assert 512 // chooses == 2


def test_pme_kernels_fit_beside_the_pair_kernel(tmp_path):
    """Mixed: three wavefronts of a plane pass beside three of the pair kernel; FP64:
    two, and two of the gather, beside two."""
    v = _vgprs("pme", tmp_path)
    budget = int(re.search(r"pair_max_vgpr = (\d+)", open(os.path.join(CSRC, "nx_device.h")).read()).group(1))
    for name in ("fft_plane_fwdINS_9PrecMixedELb1E", "fft_plane_invINS_9PrecMixedE"):
        assert 3 * v(name) <= 512 - 3 * budget, name
    for name in ("fft_plane_fwdINS_8PrecFP64ELb1E", "fft_plane_invINS_8PrecFP64E", "pme_gather_kernelINS_8PrecFP64E"):
        assert v(name) <= 96, name


def test_the_grid_asks_for_the_kernel_that_is_launched():
    """A batch with a system outside the series' range launches the kernel with library
    functions: its occupancy, not the other one's, makes the grid."""
    src = open(os.path.join(CSRC, "nonbonded.hip")).read()
    asked = re.search(r"hipOccupancyMaxActiveBlocksPerMultiprocessor\(&n, pair_kernel_of<P, false>\((\w+)\)", src).group(1)
    assert asked not in ("true", "false")
    launched = set(re.findall(r"pair_kernel_of<P, (?:true|false)>\((B\.\w+)\)<<<", src))
    engine = open(os.path.join(CSRC, "engine.hip")).read()
    assert launched == {"B.all_series"} and "pair_blocks_occupancy<P>(B.all_series)" in engine
    assert re.search(r"pair_grid_blocks<P>\([^;]*B\.all_series", engine)
