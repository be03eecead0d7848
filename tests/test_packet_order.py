"""A packet takes a node's children in the order of its first lane's distances,
which may lie past everything, be infinite or no number where only other lanes
enter the child.  Such a child still has to come before those that no lane
enters (the sort's key for these is kNotEntered).  Compiled for the host."""
import os
import subprocess

import pytest

from raycer_amd import build

PROGRAM = """
#include <cmath>
#include <cstdio>
#include "rc_device.hpp"
int main() {
    const float t[] = {0.0f, 0.5f, 0.99999994f, 1.0f, 1.5f, 2.0f, 5.0f, 1e30f, INFINITY, NAN};
    for (float x : t) {
        const float k = rcd::packet_entry(x);
        if (!(k >= 0.0f && k < rcd::kNotEntered) || (x < 1.0f && k != x)) {
            std::printf("%g sorts at %g\\n", x, k);
            return 1;
        }
    }
}
"""


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="hipcc not installed")
def test_entered_children_sort_before_the_others(tmp_path):
    src = tmp_path / "order.hip"
    src.write_text(PROGRAM)
    exe = tmp_path / "order"
    cmd = [build.HIPCC, "--offload-arch=gfx950", "-std=c++17", "-O0", f"-I{build.ROOT / 'include'}", f"-I{build.CSRC}",
           str(src), "-o", str(exe)]
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert p.returncode == 0, p.stdout
    p = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True)
    assert p.returncode == 0, p.stdout
