"""The mesh build's scratch arena (csrc/vsdmo_internal.h, BuildArena) on the
CPU, over a stand-in device allocator whose allocations lie side by side: no
piece may reach over the border of two allocations (tests/cpp/build_arena.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "volumesurfacediscretemeshoptimization_amd", "csrc")


def test_pieces_stay_in_one_allocation(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "build_arena")
    r = subprocess.run([gxx, "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I", CSRC, "-I",
                        os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "cpp", "build_arena.cpp"), "-o", exe],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.stdout, r.stderr)
