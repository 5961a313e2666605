"""The pair queue on the CPU.  The hand-over of LDS rows inside a group of lanes,
read from the sources: a group's first lane writes the rows of its pair and all
its lanes read them, and without a fence between the two the compiler may keep
the old row on the other lanes.  No run can show it missing while the compiler
happens not to, so the step functions of the queue's modes are read instead.
And the queue's claims of pairs and the rule for its launch shape, run on the
host."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "distance3d_amd", "csrc")


def _bodies(path, name):
    """The bodies of the functions called ``name``, without comments."""
    src = re.sub(r"//[^\n]*", "", open(path).read())
    for m in re.finditer(r"\b%s\([^;{}]*\)\s*{" % name, src):
        depth, i = 1, m.end()
        while depth:
            depth += {"{": 1, "}": -1}.get(src[i], 0)
            i += 1
        yield src[m.end():i]


@pytest.mark.parametrize("source, name, count", [("d3d_gjk_queue.hip", "gjk_distance_step", 1),
                                                 ("d3d_gjk_queue.hip", "step", 2),
                                                 ("d3d_mpr.hip", "step", 1)])
def test_steps_fence_before_they_read_rows(source, name, count):
    bodies = list(_bodies(os.path.join(CSRC, source), name))
    assert len(bodies) == count
    for body in bodies:
        read = re.search(r"\bpq\.[PQ]\(|\bload_y\(|\bmpr_row\(", body)
        if read is not None:
            fence = re.search(r"\brow_fence\(\)", body)
            assert fence is not None and fence.start() < read.start()


def test_claims_and_launch_shape(tmp_path):
    exe = str(tmp_path / "queue_host_check")
    try:
        subprocess.run(["/opt/rocm/bin/hipcc", "-std=c++17", "-O1", "--offload-arch=gfx950", "-I", CSRC,
                        "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "queue_host_check.hip"),
                        "-o", exe], check=True, capture_output=True, timeout=300)
    except FileNotFoundError:
        pytest.skip("hipcc not available")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
