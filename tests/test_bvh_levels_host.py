"""The packed box tree's shape on the CPU (tests/bvh_levels_check.hip)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_levels_launches_stack_and_curve(tmp_path):
    exe = str(tmp_path / "bvh_levels_check")
    try:
        subprocess.run(["/opt/rocm/bin/hipcc", "-std=c++17", "-O2", "--offload-arch=gfx950",
                        "-I", os.path.join(ROOT, "distance3d_amd", "csrc"),
                        os.path.join(ROOT, "tests", "bvh_levels_check.hip"), "-o", exe],
                       check=True, capture_output=True, timeout=300)
    except FileNotFoundError:
        pytest.skip("hipcc not available")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
