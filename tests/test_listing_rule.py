"""When the deep-stack kernel may be left out (rc_may_list), in every build: a
traversal that spills finds room for as many walks as there are slots, one that
does not spill lists each ray whose stack outgrows its rows.  The rule is
compiled for the host and asked (no GPU)."""
import os
import subprocess

import pytest

from raycer_amd import build

PROGRAM = """
#include <cstdio>
#include "rc_internal.hpp"
int main() {
    rc_scene s;
    for (unsigned need : {18u, 20u, 60u})
        for (size_t walks : {size_t(1), size_t(2048), size_t(2049)}) {
            s.stack_need = need;
            std::printf("%d", int(rc_may_list(&s, 19, walks, kMinSpillSlots)));
        }
    std::printf("\\n");
}
"""


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="hipcc not installed")
@pytest.mark.parametrize("defines,expected", [
    ([], "000001001"),
    (["RC_QNODE=0"], "000001001"),
    (["RC_PACKET_CAMERA=1"], "000111111"),
    (["RC_QNODE=0", "RC_TRAV_IFIF=0"], "000111111"),
])
def test_builds_that_do_not_spill_list(tmp_path, defines, expected):
    src = tmp_path / "rule.hip"
    src.write_text(PROGRAM)
    exe = tmp_path / "rule"
    cmd = [build.HIPCC, "--offload-arch=gfx950", "-std=c++17", "-O0", f"-I{build.ROOT / 'include'}", f"-I{build.CSRC}",
           *(f"-D{d}" for d in defines), str(src), "-o", str(exe)]
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert p.returncode == 0, p.stdout
    assert subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, check=True).stdout.strip() == expected
